"""The tree's bottom-up passes at the edges of their phases: one chunk of 1024 leaves, the first
leaf of a second one, one workgroup of 32 chunks and the first leaf past it, and a cloud of nearly
chain-like subtrees whose chunks leave more nodes than a workgroup of the later phases holds at a
time.  The walk groups (selected by one workgroup up to 32768 particles), every node's moments, box and smoothing-length bound equal the twin's bit for bit (the
quadrupoles to rounding, as in the twin's other comparisons); so do the bounds after the h-rho pass
(the pass over the smoothing lengths alone)."""
import numpy as np
import pytest

import oracle as O
from gandalf_amd import ic as ICS

pytestmark = pytest.mark.gpu


def chains(N):
    """Coordinates of sparse binary digits: 5 % of the bits set, so most nodes split off little."""
    bits = np.random.default_rng(1).random((N, 3, 21)) < 0.05
    r = (bits * 2.0 ** -np.arange(1, 22)).sum(-1)
    r[0], r[1] = 0.0, 1.0 - 2.0 ** -21
    return r


def left_by_chunks(t, N):
    """Largest number of maximal chunk nodes in a run of 32 chunks."""
    f = np.concatenate([t["first"][:N - 1], np.arange(N)])
    l = np.concatenate([t["last"][:N - 1], np.arange(N)])
    parent = np.full(2 * N - 1, -1)
    for side in ("left", "right"):
        parent[t[side][:N - 1]] = np.arange(N - 1)
    inside = f // 1024 == l // 1024
    top = inside & ~np.where(parent >= 0, inside[parent], False)
    return int(np.bincount(f[top] // 32768).max())


@pytest.mark.parametrize("kind,N", [("sphere", n) for n in (2, 63, 1024, 1025, 32768, 32769, 70001)] +
                         [("chains", 70000)])
def test_moments_match_twin_at_phase_edges(kind, N):
    from gandalf_amd.gpu import GpuSim
    g = ICS.cold_sphere(N=N, seed=3)
    r = chains(N) if kind == "chains" else g["r"]
    rng = np.random.default_rng(2)
    h = 0.01 + 0.05 * rng.random(N)
    s = GpuSim(g["params"], precision="fp64")
    s.set_particles(r, g["v"], g["m"], g["u"], h=h)
    s.build_tree()
    p = O.params_from_dict(g["params"])
    t = O.TreeTwin(p, r, g["m"], h).arrays()
    if kind == "chains":
        assert left_by_chunks(t, N) > 768
    a = s.tree_arrays()
    for k in ("perm", "first", "last", "mass", "com", "quad", "bbmin", "bbmax", "hmax",
              "group_first", "group_count", "group_node"):
        if k == "quad":
            assert np.max(np.abs(a[k] - t[k])) <= 1e-14 * max(np.max(np.abs(t[k])), 1e-300), k
        else:
            assert np.array_equal(a[k], t[k]), k
    if kind == "sphere" and N >= 1024:
        s.density()
        t = O.TreeTwin(p, r, g["m"], s.get("h")).arrays()
        assert np.array_equal(s.tree_arrays()["hmax"], t["hmax"])
