"""Block timesteps: active flags that change between the density pass and the forces.

The density pass's candidate lists hold the sets of the particles that were active in it.  Forces of
particles flagged active only afterwards - by setting the flags, by SetActiveParticles or by
CheckTimesteps - come from lists made for them: equal to the forces after the lists have been
dropped.  Both evaluate the same pairs in another order: FP64 1e-11 of the largest acceleration
(a few hundred terms, cancelling by up to a hundred), mixed the path's documented 1e-4."""
import numpy as np
import pytest

from gandalf_amd import ic as ICS

pytestmark = pytest.mark.gpu


def activate(s, how):
    one = np.ones(s.N)
    if how == "set":
        s.set("active", one)
    elif how == "set_active_particles":
        s.set("nlast", 0 * one)
        s.set("nstep", one)
        s.set_active_particles(1)
    else:
        # every neighbour five levels deeper: all end their step of four early
        for name, value in (("level", 0), ("levelneib", 5), ("nlast", 0), ("nstep", 4)):
            s.set(name, value * one)
        assert s.check_timesteps(1, 4, 1, 1.0e-4) == s.N
    assert np.all(s.get("active") == 1)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("how", ["set", "set_active_particles", "check_timesteps"])
def test_forces_of_particles_activated_after_the_density_pass(how, precision):
    from gandalf_amd.gpu import GpuSim
    g = ICS.rotating_m2_cloud(N=5003, seed=29, nlevels=4)
    sparse = (np.random.default_rng(3).random(5003) < 0.02).astype(float)
    acc = []
    for fresh in (False, True):
        s = GpuSim(g["params"], precision=precision)
        s.set_particles(g["r"], g["v"], g["m"], g["u"])
        s.setup()
        s.set("active", sparse)
        s.density()
        activate(s, how)
        if fresh:
            s.set("v", s.get("v"))
        s.all_forces()
        acc.append(s.get("a"))
    top = np.max(np.linalg.norm(acc[1], axis=1))
    e = np.max(np.linalg.norm(acc[0] - acc[1], axis=1)) / top
    assert e < (1e-11 if precision == "fp64" else 1e-4), e
