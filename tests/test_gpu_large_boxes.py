"""Full energy, non-crowder energy and adjoint in large boxes against the FP64
oracle: on both sides of the box edge up to which distances come from 32-bit
fractions of the box (1024 A) and far above it, with the bodies near the origin,
where single precision holds coordinates finely, and far from it.

Bars from the terms' magnitudes, as in test_gpu_pairs_tiles: 2e-6 of an energy
term.  Of a derivative: 3.5 units in the last place of the reciprocal, 16 of the
sixth power, 33.5 of x6 (2 x6 - 1), 3 for the constants, and two each for the
displacement's product and its sum: 42 units, 2.6e-6.  A difference of two
floats boxes apart is rounded by 2^-24 of its size, a fraction of the box to
2^-32 of it per coordinate: up to 12 (energies) or 14 (derivatives) times that
over r more."""
import numpy as np
import pytest

from remcdockingsimulator_amd import forcefield as ffm
from remcdockingsimulator_amd import synth
from remcdockingsimulator_amd.engine import Engine

pytestmark = pytest.mark.gpu

# chains (n > 0 beads) and crowders (n < 0) that share a few dozen contacts; more
# beads than the 256 up to which energies take another form
SIZES = {"chains": [40, 24, 30, 8, 56, 24, 40, 20, 24],
         "mixed": [24, 30] + [-1] * 40 + [20, 40, -3, 30, -1, 56, 24, 40, 20, 10]}


def build(sizes, rng):
    bodies = []
    for n in sizes:
        local = synth.saw_chain(abs(n), rng) if abs(n) > 1 else np.zeros((1, 3))
        bodies.append(synth.Body(local, rng.integers(0, 20, abs(n)), n < 0))
    return synth.build_system(bodies, 60.0, rng)


def bars(sa, ff, pos):
    """Error bars: full and non-crowder energy, force and torque (bodies x 6)."""
    body = np.repeat(np.arange(sa.n_bodies), np.diff(sa.body_start))
    i, j = np.triu_indices(sa.n_beads, 1)
    keep = body[i] != body[j]
    i, j = i[keep], j[keep]
    d = pos[i].astype(np.float64) - pos[j]
    raw = np.abs(d).sum(1)
    d -= sa.box * np.round(d / sa.box)
    r = np.sqrt((d * d).sum(1))
    # coordinates as given, and those of fractions in the boxes that take them
    coarse = 2.0 ** -24 * raw + (np.sqrt(3.0) * 2.0 ** -32 * sa.box if sa.box <= 1024.0 else 0.0)
    part, slope = 2e-6 + 12.0 * coarse / r, 2.6e-6 + 14.0 * coarse / r
    crow = (sa.crowder[body[i]] != 0) | (sa.crowder[body[j]] != 0)
    eij = np.abs(ff.eij()[sa.type[i], sa.type[j]])
    x6 = (0.5 * (sa.sigma[i].astype(np.float64) + sa.sigma[j]) / r) ** 6
    lj_c, dh_c = ff.lj_cf * ff.kbt_cf, ff.dh_cf * ff.kbt_cf
    dh = np.abs(sa.charge[i].astype(np.float64) * sa.charge[j]) * np.exp(-r / ff.xi) / r * dh_c
    c = np.where(r < ff.crowder_cutoff, (ff.crowder_sigma / r) ** 6, 0.0) * lj_c
    e = np.where(crow, c, (4.0 * eij * (x6 * x6 + x6) + 2.0 * eij * (x6 > 0.5)) * lj_c + dh)
    g = np.where(crow, 6.0 * c / r, 24.0 * eij * (2.0 * x6 * x6 + x6) / r * lj_c + dh * (1.0 / ff.xi + 1.0 / r))
    f = (slope * g / r)[:, None] * np.abs(d)
    force = np.zeros((sa.n_beads, 3))
    np.add.at(force, i, f)
    np.add.at(force, j, f)
    a = np.abs(sa.rel.astype(np.float64))
    turn = np.stack([a[:, 1] * force[:, 2] + a[:, 2] * force[:, 1], a[:, 2] * force[:, 0] + a[:, 0] * force[:, 2],
                     a[:, 0] * force[:, 1] + a[:, 1] * force[:, 0]], 1)
    ft = np.zeros((sa.n_bodies, 6))
    np.add.at(ft, body, np.concatenate([force, turn], 1))
    return (part * e).sum(), (part * e)[~crow].sum(), ft


@pytest.mark.parametrize("box", [1000.0, 1024.0, 1025.0, 2.0e4, 1.0e6])
@pytest.mark.parametrize("place", ["origin", "across", "far"])
@pytest.mark.parametrize("name", sorted(SIZES))
def test_energies_and_adjoint_in_large_boxes(oracle, name, place, box):
    rng = np.random.default_rng(6)
    sa = build(SIZES[name], rng)
    sa.box = float(np.float32(box))
    body = np.repeat(np.arange(sa.n_bodies), np.diff(sa.body_start))
    if place == "across":  # what lies below the middle of the system wraps to the far side
        sa.center = np.where(sa.center < 30.0, sa.center + np.float32(sa.box), sa.center).astype(np.float32)
    elif place == "far":
        sa.center = (sa.center + 0.7 * sa.box).astype(np.float32)
    sa.pos = (sa.rel + sa.center[body]).astype(np.float32)
    if place == "far" and name == "mixed":
        sa.sigma = rng.uniform(4.5, 6.5, sa.n_beads).astype(np.float32)  # sigma per bead
    ff = ffm.ForceField.synthetic(5, low=-0.6, high=0.3)
    e = Engine(0)
    e.set_forcefield(ff)
    e.add_replicas(e.add_system(sa), [300.0, 320.0], 2.0, 0.2)
    full, free = e.energy_all(), e.energy_noncrowder_all()
    fts, _ = e.adjoint_all()
    bar, bar_free, bar_ft = bars(sa, ff, sa.pos)
    osys = oracle.OracleSystem(sa, ff)
    assert abs(full[0] - osys.energy(sa.pos)) <= bar
    assert abs(free[0] - osys.energy_noncrowder(sa.pos)) <= bar_free
    _, ft, _ = osys.gradient(sa.pos.astype(np.float64), sa.rel.astype(np.float64))
    assert np.all(np.abs(fts[0] - ft) <= bar_ft + 1e-12)
    assert np.array_equal(fts[1], fts[0]) and full[1] == full[0]
    e.close()
