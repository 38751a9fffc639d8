"""Read-backs packed by one launch: every array, and any subset of them, comes
back as it was set, for sizes around the launch's 256-word blocks."""
import ctypes

import numpy as np
import pytest

from remcdockingsimulator_amd import _native as nat
from remcdockingsimulator_amd import forcefield as ffm
from remcdockingsimulator_amd import model
from remcdockingsimulator_amd.engine import Engine

pytestmark = pytest.mark.gpu


def beads(n, rng):
    """n one-bead bodies at arbitrary places."""
    pos = rng.uniform(0.0, 90.0, (n, 3)).astype(np.float32)
    return model.SystemArrays(
        body_start=np.arange(n + 1, dtype=np.int32), type=np.zeros(n, np.int32), charge=np.zeros(n, np.float32),
        sigma=np.full(n, 6.0, np.float32), crowder=np.ones(n, np.uint8), box=90.0, pos=pos,
        rel=np.zeros((n, 3), np.float32), center=pos.copy(), quat=np.tile([1.0, 0.0, 0.0, 0.0], (n, 1)))


@pytest.mark.parametrize("n", [1, 2, 15, 16, 255, 257, 1031])
def test_state_reads_back_whole_and_in_part(n):
    rng = np.random.default_rng(n)
    e = Engine(0)
    e.set_forcefield(ffm.ForceField.synthetic(1))
    e.add_replicas(e.add_system(beads(n, rng)), [300.0, 310.0, 320.0], 2.0, 0.2)
    want = []
    for r in range(3):
        st = dict(pos=rng.normal(size=(n, 3)).astype(np.float32), rel=rng.normal(size=(n, 3)).astype(np.float32),
                  center=rng.normal(size=(n, 3)).astype(np.float32), quat=rng.normal(size=(n, 4)))
        e.set_state(r, **st)
        want.append(st)
    for r in (2, 0, 1):
        got = e.state(r)
        for k in want[r]:
            assert np.array_equal(got[k], want[r][k]), (r, k)
            assert got[k].flags["C_CONTIGUOUS"]
    # any pointer may be null
    y, cz, q = np.empty(n, np.float32), np.empty(n, np.float32), np.empty((n, 4))
    null = ctypes.c_void_p()
    e._chk(e.lib.remc_get_state(e.ctx, 1, null, nat.fptr(y), null, null, null, null, null, null, nat.fptr(cz),
                                nat.dptr(q)), "remc_get_state")
    assert np.array_equal(y, want[1]["pos"][:, 1]) and np.array_equal(cz, want[1]["center"][:, 2])
    assert np.array_equal(q, want[1]["quat"])
    e._chk(e.lib.remc_get_state(e.ctx, 1, *[null] * 10), "remc_get_state")
    e.close()
