"""The direct sums at the edges of their work division: one star, a partly filled block, one
source tile and one more star, both sides of the change from 4 to 8 targets a block, and larger
counts with a remainder, against the oracle.  The sums add up to 8200 terms in another order, with a few ulps
each: 1e-12 of the maximum; the smoothed jerk carries the reference's single-precision cube, one
float ulp (1.2e-7) of its near terms, which cancel at most tenfold: 1e-6."""
import numpy as np
import pytest

import oracle as O
from gandalf_amd import ic as ICS

pytestmark = pytest.mark.gpu


def relmax(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


@pytest.mark.parametrize("smoothed", [0, 1])
@pytest.mark.parametrize("N", [1, 3, 257, 4095, 4097, 8191, 8193])
def test_direct_sums_at_edge_sizes(N, smoothed):
    from gandalf_amd.gpu import GpuSim
    g = ICS.plummer_sphere(N=max(N, 8), seed=31)
    r, v, m, u = (np.ascontiguousarray(g[k][:N]) for k in "rvmu")
    h = 0.05 + 0.05 * np.random.default_rng(N).random(N)
    g["params"].update(nbody_eps=0.0, nbody_softening=smoothed, kernel="quintic")
    s = GpuSim(g["params"], precision="fp64")
    s.set_particles(r, v, m, u, h=h)
    s.nbody_direct(smoothed=bool(smoothed))
    if smoothed:
        a, ad, gp = O.nbody_direct_smoothed(O.params_from_dict(g["params"]), r, v, m, h)
    else:
        a, ad, gp = O.nbody_direct(r, v, m)
    if N == 1:
        assert not s.get("a").any() and not s.get("adot").any()
        return
    assert relmax(s.get("a"), a) < 1e-12
    assert relmax(s.get("gpot"), gp) < 1e-12
    assert relmax(s.get("adot"), ad) < (1e-6 if smoothed else 1e-12)
