"""Lists of the walk groups that hold active particles, over the number of groups a workgroup of the
compaction takes (1024): the gravity walk of a force pass counts interactions for exactly those
groups, and the counts of a group do not depend on which other groups are listed."""
import numpy as np
import pytest

from gandalf_amd import ic as ICS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65, 20011, 70001, 140009])
@pytest.mark.parametrize("share", [0.0005, 0.02, 1.0])
def test_walked_groups_are_those_with_active_particles(n, share):
    from gandalf_amd.gpu import GpuSim
    g = ICS.rotating_m2_cloud(N=n, seed=23, nlevels=4)
    s = GpuSim(g["params"], precision="mixed")
    s.set_particles(g["r"], g["v"], g["m"], g["u"])
    s.setup()
    rng = np.random.default_rng(n)
    act = (rng.random(s.N) < share).astype(float)
    act[rng.integers(s.N)] = 1.0
    a = s.tree_arrays()
    counts = []
    for flags in (np.ones(s.N), act):
        s.set("active", flags)
        s.all_forces()
        counts.append(s.gravity_group_counts())
    on = np.add.reduceat(act[a["perm"]], a["group_first"]) > 0
    for full, some in zip(*counts):
        assert np.array_equal(some, np.where(on, full, 0))
    assert np.all(counts[0][1] > 0)
