"""MC steps of systems without a box against the FP64 oracle: bodies and moves
identical, dE within 1e-4 kT and 1e-5 of |dE| (the bars of the MC parity tests
with steep contacts), positions bit-identical while the decisions agree, and the
tracked energy that of the conformation reached.  Chains and crowders close
together, so that moves meet contacts, crowders and both."""
import numpy as np
import pytest

from helpers import compare_decisions, engine_for, kT, say
from remcdockingsimulator_amd import forcefield as ffm
from remcdockingsimulator_amd import synth

pytestmark = pytest.mark.gpu

SEED = 0x0B0C
STEPS = 400


def workload(crowders, per_bead):
    rng = np.random.default_rng(11)
    bodies = [synth.chain_body(n, rng) for n in (40, 24, 33, 5)] + [synth.crowder_body() for _ in range(crowders)]
    sa = synth.build_system(bodies, 55.0, rng)
    sa.box = 0.0
    if per_bead:
        sa.sigma = rng.uniform(5.0, 6.5, sa.n_beads).astype(np.float32)
    ladder = synth.geometric_ladder(290.0, 420.0, 4)
    return synth.Workload("boxes", [sa], [ladder], 2.0, 0.2, ffm.ForceField.synthetic(9))


@pytest.mark.parametrize("coop", [1, 2])
@pytest.mark.parametrize("crowders,per_bead,lds_cache,window", [(0, False, True, True), (24, False, True, True),
                                                                (24, True, False, True), (24, False, True, False)])
def test_mc_parity_without_a_box(oracle, crowders, per_bead, lds_cache, window, coop):
    wl = workload(crowders, per_bead)
    sa, ladder = wl.systems[0], wl.temperatures[0]
    e = engine_for(wl, seed=SEED, block=256)
    e.set_mc_coop(coop)
    e.set_mc_tuning(lds_cache=lds_cache, split_min_pairs=64)
    e.set_mc_window(window)
    e.set_recording(STEPS)
    e.mc_steps(STEPS)
    e.synchronize()
    o = oracle.OracleSystem(sa, wl.ff)
    energies, diverged, moved = e.energies(), 0, 0
    for r, T in enumerate(ladder):
        say("crowders", crowders, "cache", lds_cache, "window", window, "members", coop, "replica", r)
        orep = oracle.OracleReplica(o, T, wl.translate_step, wl.rotate_step, r)
        orec = orep.mc(seed=SEED, nsteps=STEPS, mode=0)
        rec = e.records(r)
        _, div = compare_decisions(rec, orec, T, rel_tol=1e-5)
        moved += int(np.count_nonzero(orec["delta"]))
        st = e.state(r)
        want = o.energy(st["pos"])
        assert abs(energies[r] - want) <= 1e-4 * kT(T) + 1e-5 * abs(want)
        if div:
            diverged += 1
            continue
        for k, v in (("pos", orep.pos), ("rel", orep.rel), ("center", orep.center), ("quat", orep.quat)):
            assert np.array_equal(st[k], v), (r, k)
    assert diverged <= 1 and moved > STEPS
    e.close()
