"""Block timesteps, FP64: the neighbour sets after a step are those of the step's last force pass,
for its targets (NeighbourManager.h:521), though the step's end has cleared the active flags; with
the flags set since, a fresh walk's for the flagged particles.  Exactly the oracle's brute-force
sets."""
import numpy as np
import pytest

import oracle as O
from conftest import load_golden

pytestmark = pytest.mark.gpu


def rows(off, ids, which):
    return [ids[off[i]:off[i + 1]].tolist() for i in np.flatnonzero(which)]


def test_sets_after_block_steps():
    from gandalf_amd.gpu import GpuSim
    d = load_golden("cloud4k_quintic_blk")
    p = O.params_from_dict(d["meta"]["params"])
    s = GpuSim(d["meta"]["params"], precision="fp64")
    s.set_particles(d["in_r"], d["in_v"], d["in_m"], d["in_u"])
    s.setup()
    sparse = 0
    for k in range(6):
        for mode in (1, 0):
            off, ids = s.neighbour_sets(mode)
            ref = O.neighbour_sets(p, s.get("r"), s.get("h"), mode)
            tgt = np.diff(off) > 0
            assert tgt.all() if k == 0 else tgt.any(), k
            assert rows(off, ids, tgt) == rows(*ref, tgt), (k, mode)
        sparse += tgt.sum() < s.N // 4
        s.step(1)
    assert sparse > 0
    flags = np.zeros(s.N)
    flags[::7] = 1
    s.set("active", flags)
    off, ids = s.neighbour_sets(1)
    assert np.array_equal(np.diff(off) > 0, flags > 0)
    assert rows(off, ids, flags > 0) == rows(*O.neighbour_sets(p, s.get("r"), s.get("h"), 1), flags > 0)
