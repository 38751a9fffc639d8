"""The adjoint's sums hold every pair's contribution to the same precision: a
body midway between pairs of equal beads feels exactly no force, since the two
contributions of a pair are the same number with opposite signs.  (Added in
single precision before the 64-bit sum, the two leave the rounding of one.)
Coordinates are such that both displacements are exact in every form."""
import numpy as np
import pytest

from remcdockingsimulator_amd import forcefield as ffm
from remcdockingsimulator_amd.engine import Engine
from remcdockingsimulator_amd.model import SystemArrays

pytestmark = pytest.mark.gpu

F = np.float32


@pytest.mark.parametrize("box", [0.0, 64.0, 4096.0])
@pytest.mark.parametrize("pairs,charge", [(8, 0.0), (8, 1.0), (40, 1.0), (33, 1.0)])
def test_no_force_between_equal_beads(pairs, charge, box):
    rng = np.random.default_rng(pairs)
    at = np.array([24.0, 32.0, 16.0])
    d = np.rint(rng.uniform(3.0, 7.0, (pairs, 3)) * 2.0 ** 17) / 2.0 ** 17 * rng.choice([-1.0, 1.0], (pairs, 3))
    other = np.stack([at + d, at - d], 1).reshape(-1, 3)  # bead 2 k opposite bead 2 k + 1
    n, rows = 64 + 2 * pairs, 64
    pos = np.concatenate([np.tile(at, (rows, 1)), other]).astype(F)
    assert np.array_equal(pos[rows::2].astype(float) - at, at - pos[rows + 1::2].astype(float))
    types = np.concatenate([rng.integers(0, 20, rows), np.repeat(rng.integers(0, 20, pairs), 2)]).astype(np.int32)
    q = np.concatenate([np.full(rows, charge), np.repeat(rng.choice([-1.0, 0.0, 1.0], pairs) * charge, 2)]).astype(F)
    center = np.stack([at, at]).astype(F)
    rel = (pos - center[0]).astype(F)
    sa = SystemArrays(body_start=np.array([0, rows, n], np.int32), type=types, charge=q, sigma=np.full(n, 6.0, F),
                      crowder=np.zeros(2, np.uint8), box=box, pos=pos, rel=rel, center=center,
                      quat=np.tile([1.0, 0, 0, 0], (2, 1)))
    e = Engine(0)
    e.set_forcefield(ffm.ForceField.synthetic(3, low=-0.6, high=0.3))
    e.add_replicas(e.add_system(sa), [300.0], 2.0, 0.2)
    (ft,), _ = e.adjoint_all()
    one, _ = e.adjoint(0)
    e.close()
    assert np.all(ft[0] == 0.0) and np.all(one[0] == 0.0), (ft[0], one[0])
