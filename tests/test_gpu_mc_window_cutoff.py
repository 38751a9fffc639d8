"""Windows without the partner cache at the crowder cutoff.  Slot a of a window
moves a crowder (of one bead, or three) into another's reach by less than FP32
resolves: in box units, in which the single steps and these windows form the
distances of a one-bead crowder's move, the pair lies inside the cutoff, in
Angstrom outside.  Slot b, which moves the other crowder away, must then see
slot a's move: its dE is minus the term at the cutoff, as single steps have it.
The places are searched for on the host with the two forms' operations; dE is
compared for equality."""
import numpy as np
import pytest

from remcdockingsimulator_amd import forcefield as ffm
from remcdockingsimulator_amd.engine import Engine
from remcdockingsimulator_amd.model import SystemArrays

pytestmark = pytest.mark.gpu

BOX, N, F = 90.0, 8, np.float32
PARKED = np.array([[x, y, 70.0] for x in (5.0, 35.0, 65.0) for y in (5.0, 35.0, 65.0)])[:N]  # out of each other's reach


def engine(pos, seed, window, steps, tail):
    """One replica of crowders of one bead, the last of `tail` beads at one place."""
    sizes, center = [1] * (N - 1) + [tail], np.asarray(pos, F)
    body = np.repeat(np.arange(len(sizes)), sizes)
    rel = np.zeros((len(body), 3), F)
    n = len(body)
    sa = SystemArrays(body_start=np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32), type=np.zeros(n, np.int32),
                      charge=np.zeros(n, F), sigma=np.full(n, 6.0, F), crowder=np.ones(len(sizes), np.uint8),
                      box=BOX, pos=(rel + center[body]).astype(F), rel=rel, center=center,
                      quat=np.tile([1.0, 0, 0, 0], (len(sizes), 1)))
    e = Engine(0)
    e.set_forcefield(ffm.ForceField.synthetic(1))
    e.set_seed(seed)
    e.add_replicas(e.add_system(sa), [300.0], 2.0, 0.2)
    e.set_mc_block(256)
    e.set_mc_coop(1)
    e.set_mc_tuning(lds_cache=False)
    e.set_mc_window(window)
    e.set_recording(steps)
    e.mc_steps(steps)
    rec, center = e.records(0), e.state(0)["center"]
    e.close()
    return rec, center


def r2(dx, dy, dz):
    """fma(dx, dx, fma(dy, dy, dz dz)) in float32."""
    w = np.longdouble
    z = (dz.astype(w) * dz).astype(F)
    y = (dy.astype(w) * dy + z).astype(F)
    return (dx.astype(w) * dx + y).astype(F)


def straddling(na, ta, tb, rng, cut):
    """A place b about the cutoff from na, inside it in box units only, beyond
    reach of na - ta and, moved by tb, of both."""
    ib = F(1.0) / F(BOX)
    cut2 = F(cut) * F(cut)
    cut2u = cut2 * (ib * ib)
    for _ in range(200):
        u = rng.normal(size=(20000, 3))
        u /= np.linalg.norm(u, axis=1)[:, None]
        u = u[(u @ ta > 0.8) & (u @ tb > 0.8)]
        b = (na + u * (cut * (1.0 + rng.uniform(-2e-7, 2e-7, (len(u), 1))))).astype(F)
        d = (na.astype(F) - b).astype(F)
        du = (d * ib).astype(F)
        ok = (r2(*d.T) >= cut2) & (r2(*du.T) < cut2u) & np.all((b > 3.0) & (b < BOX - 3.0), axis=1)
        if ok.any():
            return b[np.argmax(ok)]
    return None


@pytest.mark.parametrize("tail", [1, 3])
def test_windows_see_what_single_steps_see_at_the_cutoff(tail):
    cut = ffm.ForceField.synthetic(1).crowder_cutoff
    rng = np.random.default_rng(2)
    found = 0
    for seed in range(1, 400):
        if found == 6:
            break
        rec, first = engine(PARKED, seed, False, 1, tail)
        a = int(rec["body"][0])
        if rec["move"][0] != 0 or (a == N - 1) != (tail > 1):  # the crowder of several beads moves first
            continue
        rec, both = engine(PARKED, seed, False, 2, tail)
        b = int(rec["body"][1])
        if rec["move"][1] != 0 or b == a or np.any(rec["delta"]):
            continue
        ta, tb = (first[a] - PARKED[a]).astype(float), (both[b] - PARKED[b]).astype(float)
        pos = PARKED.astype(F)
        pos[a] = [45.0, 40.0, 30.0]
        na = engine(pos, seed, False, 1, tail)[1][a]
        pb = straddling(na.astype(float), ta, tb, rng, cut)
        if pb is None:
            continue
        pos[b] = pb
        single, windows = engine(pos, seed, False, 2, tail)[0], engine(pos, seed, True, 2, tail)[0]
        print("seed", seed, "bodies", a, b, "dE", single["delta"], windows["delta"], flush=True)
        # slot a's own dE is the term at the cutoff or none, by a rounding of its own
        # (a window has that of several beads in Angstrom)
        if not single["accepted"][0] or not windows["accepted"][0]:
            continue
        assert tail > 1 or windows["delta"][0] == single["delta"][0]
        assert single["delta"][1] < 0.0 and windows["delta"][1] == single["delta"][1]
        found += 1
    assert found == 6
