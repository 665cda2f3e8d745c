"""A force pass that fails while its gravity walk runs on the second stream (forced from the host:
GDF_FAULT_HYDRO makes the hydro pass report a failure) returns with the walk finished: the context
takes other particles and gives their forces as a fresh context does, bit for bit."""
import numpy as np
import pytest

from gandalf_amd import ic as ICS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_context_after_a_failed_force_pass(precision, monkeypatch):
    from gandalf_amd.gpu import GdfError, GpuSim
    N = 60000
    first, second = (ICS.rotating_m2_cloud(N=N, seed=s) for s in (41, 42))

    def forces(s):
        s.set_particles(second["r"], second["v"], second["m"], second["u"])
        s.setup()
        return s.get("a"), s.get("gpot")

    s = GpuSim(first["params"], precision=precision)
    s.set_particles(first["r"], first["v"], first["m"], first["u"])
    s.setup()
    s.build_tree()
    s.density()
    monkeypatch.setenv("GDF_FAULT_HYDRO", "1")
    with pytest.raises(GdfError, match="injected failure"):
        s.all_forces()
    monkeypatch.delenv("GDF_FAULT_HYDRO")
    for x, y in zip(forces(s), forces(GpuSim(first["params"], precision=precision))):
        assert np.array_equal(x, y)
