"""The mixed path with tabulated kernels, whose density sums keep to one order (a lone wavefront, a
batch at a time): h and rho against the FP64 path from the same first guesses, also where the search
radii grow.  A pair takes another entry of the 1000 where FP32 moves it across, about one in 10^4,
which changes a density by less than 1e-3: at most a few per cent of the particles, 1e-4 rms.  Where that decides whether a
particle iterates once more its h moves by up to the iteration's own tolerance, 1e-2."""
import numpy as np
import pytest

from gandalf_amd import ic as ICS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [13, 27, 40])
@pytest.mark.parametrize("kernel", ["m4", "quintic"])
@pytest.mark.parametrize("factor", [1.0, 0.8])
def test_mixed_tabulated_density_follows_fp64(side, kernel, factor):
    from gandalf_amd.gpu import GpuSim
    g = ICS.jittered_lattice_box(n_side=side, seed=7)
    g["params"].update(kernel=kernel, tabulated_kernel=1)
    got = {}
    for precision in ("fp64", "mixed"):
        s = GpuSim(g["params"], precision=precision)
        s.set_particles(g["r"], g["v"], g["m"], g["u"])
        s.setup()
        if precision == "fp64":
            h0 = s.get("h") * factor
        s.set("h", h0)
        s.build_tree()
        s.density()
        got[precision] = s.get("h"), s.get("rho")
    for a, b in zip(got["mixed"], got["fp64"]):
        d = np.abs(a / b - 1.0)
        assert np.sqrt(np.mean(d * d)) < 1e-4
        assert d.max() < 3e-2          # rho goes with the cube of h
