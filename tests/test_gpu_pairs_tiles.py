"""Full energy, non-crowder energy and adjoint around the edges of the tiles
(64 rows) and groups (16 columns) of the all-pairs kernels, against the FP64
oracle: bead counts at the edges, chains and crowders of one and more beads in
any order, systems without a box, bodies several boxes away, positive contact
energies (the repulsive flip), sigma per type and per bead.

The pair energies of these systems have both signs, so a sum's error is
measured against the sum of the terms' magnitudes: r^2 carries at most 2.5 units
in the last place (three differences, three roundings of squares and sums), the
sixth power of the inverse three times that and two more units from the
reciprocal and sigma^2 each time, its square twice that: 27 units, 1.6e-6 of a
term, and the contact energy's own rounding; 2e-6 in all.  A difference of two
floats that lie boxes apart is itself rounded, by 2^-24 of its size before the
minimum image, and a term has up to twelve times the relative error of r: that
much more for each pair.  The adjoint's bar is test_gpu_adjoint's (1e-4 of the
largest component)."""
import numpy as np
import pytest

from remcdockingsimulator_amd import forcefield as ffm
from remcdockingsimulator_amd import synth
from remcdockingsimulator_amd.engine import Engine

pytestmark = pytest.mark.gpu

# bodies in order: n > 0 a chain of n beads, n < 0 a crowder of -n beads
SYSTEMS = {
    "63 beads": [40, 23],
    "64 beads": [33, 31],
    "65 beads, a crowder last": [40, 24, -1],
    "crowders first": [-1] * 20 + [30, 50],
    "crowders between": [17, -1, -1, -1, 30, -1, 48, -1],
    "crowders of several beads": [16, -3, 16, -16, 16, -2, 61],
    "129 beads": [100, 29],
    "crowders only": [-1] * 130,
    "one body": [70],
    "many small chains": [3] * 50 + [-1] * 30,
    "chains of one bead": [1] * 40 + [-1] * 40 + [20],
}


def build(sizes, box, rng):
    bodies = []
    for n in sizes:
        local = synth.saw_chain(abs(n), rng) if abs(n) > 1 else np.zeros((1, 3))
        bodies.append(synth.Body(local, rng.integers(0, 20, abs(n)), n < 0))
    return synth.build_system(bodies, box, rng)


def bars(sa, ff, pos):
    """The error bars of the full and the non-crowder energy."""
    body = np.repeat(np.arange(sa.n_bodies), np.diff(sa.body_start))
    i, j = np.triu_indices(sa.n_beads, 1)
    keep = body[i] != body[j]
    i, j = i[keep], j[keep]
    d = pos[i].astype(np.float64) - pos[j]
    raw = np.abs(d).sum(1)
    if sa.box > 0:
        d -= sa.box * np.round(d / sa.box)
    r = np.sqrt((d * d).sum(1))
    part = 2e-6 + 12.0 * 2.0 ** -24 * raw / r
    crow = (sa.crowder[body[i]] != 0) | (sa.crowder[body[j]] != 0)
    eij = ff.eij()[sa.type[i], sa.type[j]]
    x6 = (0.5 * (sa.sigma[i].astype(np.float64) + sa.sigma[j]) / r) ** 6
    dh = sa.charge[i].astype(np.float64) * sa.charge[j] * np.exp(-r / ff.xi) / r * ff.dh_cf * ff.kbt_cf
    contact = (4.0 * np.abs(eij) * (x6 * x6 + x6) + 2.0 * np.abs(eij) * (x6 > 0.5)) * ff.lj_cf * ff.kbt_cf + np.abs(dh)
    c = np.where(r < ff.crowder_cutoff, (ff.crowder_sigma / r) ** 6, 0.0) * ff.lj_cf * ff.kbt_cf
    free = (part * contact)[~crow].sum()
    return free + (part * c)[crow].sum(), free


@pytest.mark.parametrize("name", sorted(SYSTEMS))
@pytest.mark.parametrize("form", ["box", "no box", "images", "sigma per bead"])
def test_energies_and_adjoint_at_tile_edges(oracle, name, form):
    rng = np.random.default_rng(len(name) + 7)
    sa = build(SYSTEMS[name], 75.0, rng)
    ff = ffm.ForceField.synthetic(5, low=-0.6, high=0.3)  # some pairs repel
    body = np.repeat(np.arange(sa.n_bodies), np.diff(sa.body_start))
    if form == "no box":
        sa.box = 0.0
    elif form == "images":
        shift = (75.0 * rng.integers(-3, 4, (sa.n_bodies, 3))).astype(np.float32)
        sa.center = sa.center + shift
        sa.pos = (sa.rel + sa.center[body]).astype(np.float32)
    elif form == "sigma per bead":
        sa.sigma = rng.uniform(4.5, 6.5, sa.n_beads).astype(np.float32)
    e = Engine(0)
    e.set_forcefield(ff)
    e.add_replicas(e.add_system(sa), [300.0, 320.0, 340.0], 2.0, 0.2)
    confs = []
    for r in range(3):
        center = (sa.center + rng.uniform(-0.5, 0.5, sa.center.shape)).astype(np.float32)
        pos = (sa.rel + center[body]).astype(np.float32)
        e.set_state(r, pos=pos, center=center)
        confs.append(pos)
    osys = oracle.OracleSystem(sa, ff)
    full, free = e.energy_all(), e.energy_noncrowder_all()
    assert np.array_equal(e.energy_all_noalloc(), full)
    fts, dps = e.adjoint_all()
    for r, pos in enumerate(confs):
        bar, bar_free = bars(sa, ff, pos)
        want = osys.energy(pos)
        assert abs(full[r] - want) <= bar, (r, full[r], want, bar)
        want = osys.energy_noncrowder(pos)
        assert abs(free[r] - want) <= bar_free, (r, free[r], want, bar_free)
        _, ft, dp = osys.gradient(pos.astype(np.float64), sa.rel.astype(np.float64))
        scale = np.max(np.abs(ft))
        for got, gdp in ((fts[r], dps[r]), e.adjoint(r)):
            assert np.max(np.abs(got - ft)) <= 1e-4 * scale + 1e-9, (r, np.max(np.abs(got - ft)), scale)
            for k in range(3):
                assert abs(gdp[k] - dp[k]) <= 1e-4 * max(abs(dp[k]), 1e-6), (r, k, gdp[k], dp[k])
    e.close()


def test_unequal_systems_in_one_launch(oracle):
    """Systems whose tile counts differ share the launch's grid."""
    rng = np.random.default_rng(3)
    ff = ffm.ForceField.synthetic(6)
    e = Engine(0)
    e.set_forcefield(ff)
    systems = [build(s, b, rng) for s, b in (([20, 9], 60.0), ([150, 100, 90] + [-1] * 60, 130.0), ([-1], 50.0))]
    for sa in systems:
        e.add_replicas(e.add_system(sa), [300.0, 330.0], 2.0, 0.2)
    full = e.energy_all()
    fts, _ = e.adjoint_all()
    for s, sa in enumerate(systems):
        osys = oracle.OracleSystem(sa, ff)
        want = osys.energy(sa.pos)
        _, ft, _ = osys.gradient(sa.pos.astype(np.float64), sa.rel.astype(np.float64))
        for r in (2 * s, 2 * s + 1):
            assert abs(full[r] - want) <= bars(sa, ff, sa.pos)[0]
            assert np.max(np.abs(fts[r] - ft)) <= 1e-4 * np.max(np.abs(ft)) + 1e-9
    e.close()
