"""Search radii that have to grow: the h-rho pass from a first guess several times too small, whose
particles need many of the reference's 1.05 steps, ends at the same h as the oracle's, and beyond the
reference's number of retries it fails as before.  FP64: h to 1e-12, as sums of up to a hundred terms
of one sign in another order."""
import numpy as np
import pytest

import oracle as O
from gandalf_amd import ic as ICS

pytestmark = pytest.mark.gpu


def first_guess_pass(factor):
    from gandalf_amd.gpu import GpuSim
    g = ICS.rotating_m2_cloud(N=3001, seed=17)
    g["params"].update(kernel="m4", gas_eos="energy_eqn")
    s = GpuSim(g["params"], precision="fp64")
    s.set_particles(g["r"], g["v"], g["m"], g["u"])
    s.setup()
    h0 = s.get("h") * factor
    s.set("h", h0)
    s.build_tree()
    s.density()
    return s, O.compute_h(O.params_from_dict(g["params"]), s.get("r"), s.get("m"), h0, s.get("u"))


@pytest.mark.parametrize("factor", [0.9, 0.5, 0.2])
def test_small_first_guess_reaches_the_same_h(factor):
    s, ref = first_guess_pass(factor)
    assert np.max(np.abs(s.get("h") / ref["h"] - 1.0)) < 1e-12
    assert np.max(np.abs(s.get("rho") / ref["rho"] - 1.0)) < 1e-12


def test_too_small_first_guess_is_refused():
    from gandalf_amd.gpu import GdfError
    with pytest.raises(GdfError, match="did not settle"):
        first_guess_pass(0.01)
