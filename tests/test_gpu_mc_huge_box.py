"""MC steps in a box of 1e7 A, whose sixth power is beyond single precision (the
crowder term of a large move takes a sixth power of the distance), against the
FP64 oracle at the MC parity tests' bars with steep contacts.  The bodies stay a
hundred Angstrom and more from the boundary, so that no pair's difference is one
of coordinates of the box's size, which single precision holds to 1 A."""
import numpy as np
import pytest

from helpers import compare_decisions, engine_for, kT, say
from remcdockingsimulator_amd import forcefield as ffm
from remcdockingsimulator_amd import synth

pytestmark = pytest.mark.gpu

SEED = 0x0B0C
STEPS = 200


@pytest.mark.parametrize("lds_cache,window", [(True, True), (False, True), (True, False)])
@pytest.mark.parametrize("box", [1.0e7, 9.0e5])
def test_mc_parity_in_a_huge_box(oracle, box, lds_cache, window):
    rng = np.random.default_rng(11)
    bodies = [synth.chain_body(n, rng) for n in (40, 24, 33, 5)] + [synth.crowder_body() for _ in range(24)]
    sa = synth.build_system(bodies, 55.0, rng)
    sa.box = float(np.float32(box))
    body = np.repeat(np.arange(sa.n_bodies), np.diff(sa.body_start))
    sa.center = np.rint(sa.center + 400.0).astype(np.float32)
    sa.pos = (sa.rel + sa.center[body]).astype(np.float32)
    ladder = synth.geometric_ladder(290.0, 420.0, 4)
    wl = synth.Workload("huge box", [sa], [ladder], 2.0, 0.2, ffm.ForceField.synthetic(9))
    e = engine_for(wl, seed=SEED, block=256)
    e.set_mc_coop(1)
    e.set_mc_tuning(lds_cache=lds_cache)
    e.set_mc_window(window)
    e.set_recording(STEPS)
    e.mc_steps(STEPS)
    e.synchronize()
    o = oracle.OracleSystem(sa, wl.ff)
    energies, diverged = e.energies(), 0
    for r, T in enumerate(ladder):
        say("box", box, "cache", lds_cache, "window", window, "replica", r)
        orep = oracle.OracleReplica(o, T, wl.translate_step, wl.rotate_step, r)
        orec = orep.mc(seed=SEED, nsteps=STEPS, mode=0)
        _, div = compare_decisions(e.records(r), orec, T, rel_tol=1e-5)
        st = e.state(r)
        assert 300.0 < st["pos"].min() and st["pos"].max() < 600.0
        want = o.energy(st["pos"])
        assert abs(energies[r] - want) <= 1e-4 * kT(T) + 1e-5 * abs(want)
        if div:
            diverged += 1
            continue
        for k, v in (("pos", orep.pos), ("rel", orep.rel), ("center", orep.center), ("quat", orep.quat)):
            assert np.array_equal(st[k], v), (r, k)
    assert diverged <= 1
    e.close()
