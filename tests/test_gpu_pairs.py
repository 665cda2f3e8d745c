"""The h-rho and hydro passes at the sizes where their work division changes: one walk group, one
partly filled batch of candidates, two batches and a remainder, and one, two and four wavefronts
sharing a group's candidates (more than 2048 groups, 257 to 2048, at most 256 - reached here with
small groups).  Open clouds with self-gravity and periodic boxes, some with ranges that reach past
half the box from a group, the three kernels, both precisions.

Against the oracle's brute-force passes.  FP64: h, rho and the grad-h sums add up to a few hundred
terms of one sign in another order, 1e-14 each, amplified by less than ten in h and rho: 1e-12 of
the field's maximum; the forces cancel by up to a hundred more: 1e-11.  Mixed: pair terms in FP32,
1e-4 of the largest acceleration as documented for the path; h stops within one iteration of the
oracle's, and successive iterations at the end differ by less than h_converge = 0.01.  With the
tabulated kernel FP32 rounding can move a pair by one of the table's 1000 entries: 1e-3."""
import numpy as np
import pytest

import oracle as O
from gandalf_amd import ic as ICS

pytestmark = pytest.mark.gpu

KERNELS = {"m4": ("m4", 0), "quintic": ("quintic", 0), "m4_tab": ("m4", 1)}
# particles, largest walk group
CLOUDS = [(33, 64), (65, 64), (300, 64), (2500, 64), (2500, 7), (5003, 2)]


def relmax(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


def passes(g, precision, gmax):
    from gandalf_amd.gpu import GpuSim
    s = GpuSim(g["params"], precision=precision, group_max=gmax)
    s.set_particles(g["r"], g["v"], g["m"], g["u"])
    s.setup()
    return s


def check(g, precision, gmax, grav):
    s = passes(g, precision, gmax)
    p = O.params_from_dict(g["params"])
    r, m = s.get("r"), s.get("m")
    h0 = s.get("h")
    s.density()                      # from the settled smoothing lengths
    st = {k: s.get(k) for k in ("h", "rho", "invomega", "zeta", "pressure", "sound", "hfactor")}
    ref = O.compute_h(p, r, m, h0, s.get("u"))
    for k in ("h", "rho", "invomega", "zeta"):
        if precision == "fp64":
            if k != "zeta" or grav:
                assert relmax(st[k], ref[k]) < 1e-12, k
        elif k == "h":
            assert np.max(np.abs(st[k] / ref[k] - 1.0)) < 0.01, k
    (s.all_forces if grav else s.hydro_forces)()
    tol = 1e-11 if precision == "fp64" else 1e-3 if p.tabulated else 1e-4
    a, dudt, _ = O.hydro_forces(p, int(grav), r, s.get("v"), m, st)
    if grav:
        at, gp = O.direct_gravity(p, r, m, st)
        a = a + at
        assert relmax(s.get("gpot"), gp) < tol
    e = np.linalg.norm(s.get("a") - a, axis=1)
    assert np.max(e) < tol * np.max(np.linalg.norm(a, axis=1))
    if precision == "fp64" and not grav:     # the clouds turn rigidly: their dudt is zero
        assert relmax(s.get("dudt"), dudt) < 1e-10


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kern", list(KERNELS))
@pytest.mark.parametrize("N,gmax", CLOUDS)
def test_cloud_passes_match_oracle(N, gmax, kern, precision):
    g = ICS.rotating_m2_cloud(N=N, seed=11)
    # every cell opened: the walk is the exact kernel-softened sum
    g["params"].update(kernel=KERNELS[kern][0], tabulated_kernel=KERNELS[kern][1],
                       thetamaxsqd=1e-12, gas_eos="energy_eqn")
    check(g, precision, gmax, True)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_gravity_walk_of_many_groups_matches_oracle(precision):
    """More than 8192 walk groups: one wavefront a group in the gravity walk (the clouds above
    have two and four)."""
    g = ICS.rotating_m2_cloud(N=17011, seed=12)
    g["params"].update(kernel="m4", thetamaxsqd=1e-12, gas_eos="energy_eqn")
    s = passes(g, precision, 2)
    assert s.tree_arrays()["group_first"].size > 8192
    check(g, precision, 2, True)


# The mixed path takes a candidate's image about the group's centre for all of its targets, so it
# has no cases where a group's extent and range pass half the box, and none with the tabulated
# kernel, where a lattice's nearly cancelling sums leave no bound on the effect of a shifted entry.
@pytest.mark.parametrize("side,gmax,kern,precision", [
    (7, 64, "m4", "fp64"), (7, 64, "m4_tab", "fp64"),
    (11, 64, "m4", "fp64"), (11, 64, "quintic", "fp64"), (11, 64, "m4_tab", "fp64"),
    (11, 64, "m4", "mixed"),
    (13, 3, "m4", "fp64"), (13, 3, "quintic", "fp64"), (13, 3, "m4_tab", "fp64"),
    (13, 3, "m4", "mixed"), (13, 3, "quintic", "mixed")])
def test_periodic_box_passes_match_oracle(side, gmax, kern, precision):
    g = ICS.jittered_lattice_box(n_side=side, seed=5, vamp=1.0)
    g["params"].update(kernel=KERNELS[kern][0], tabulated_kernel=KERNELS[kern][1])
    check(g, precision, gmax, False)
