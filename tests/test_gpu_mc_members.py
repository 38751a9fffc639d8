"""MC launches whose replicas have different numbers of workgroups: a context
of one costly system of two replicas and a light one of 290, where as many
workgroups for every replica is at most two each and the costly replicas alone
decide the launch's time.  The members (up to 32) share each large move and
each window; with and without the partner cache; and again after host-protocol
steps have changed the canonical state only.  Bars as in the other MC parity
tests: bodies and moves identical, dE within 1e-4 kT of the FP64 oracle
(and 1e-5 of |dE| for steep contacts, where an error of r^2 of a few 2^-24 in
FP32 counts six times), positions bit-identical while the decisions agree."""
import numpy as np
import pytest

from helpers import compare_decisions, engine_for, kT, say
from remcdockingsimulator_amd import forcefield as ffm
from remcdockingsimulator_amd import synth

pytestmark = pytest.mark.gpu

SEED = 0xBA1A


def workload():
    rng = np.random.default_rng(77)
    ff = ffm.ForceField.synthetic(7)
    heavy = synth.build_system([synth.chain_body(n, rng) for n in (97, 130, 64, 111, 65, 96, 128)]
                               + [synth.crowder_body() for _ in range(29)], 210.0, rng)
    light = synth.build_system([synth.chain_body(33, rng), synth.chain_body(7, rng)]
                               + [synth.crowder_body() for _ in range(11)], 90.0, rng)
    return synth.Workload("members", [light, heavy], [synth.geometric_ladder(290.0, 420.0, 290), [300.0, 330.0]], 2.0,
                          0.2, ff)


@pytest.mark.parametrize("block,lds_cache,window", [(256, True, True), (256, False, True), (1024, False, True),
                                                    (512, True, False)])
def test_members_by_cost(oracle, block, lds_cache, window):
    wl = workload()
    e = engine_for(wl, seed=SEED, block=block)
    e.set_mc_tuning(lds_cache=lds_cache, split_min_pairs=64)
    e.set_mc_window(window)
    n1, n2, n3 = 120, 9, 90
    heavy = 290  # the first replica of the costly system
    e.mc_steps(n1)
    e.mc_steps_plain(heavy, n2)
    e.set_recording(n3)
    e.mc_steps(n3)
    e.synchronize()
    energies = e.energies()
    diverged = 0
    for r, sys in ((heavy, 1), (heavy + 1, 1), (0, 0), (289, 0)):
        say("block", block, "cache", lds_cache, "window", window, "replica", r)
        T = float(np.concatenate(wl.temperatures)[r])
        o = oracle.OracleSystem(wl.systems[sys], wl.ff)
        first = oracle.OracleReplica(o, T, wl.translate_step, wl.rotate_step, r)
        before = n1 + (n2 if r == heavy else 0)
        first.mc(seed=SEED, nsteps=before, mode=0)
        orep = oracle.OracleReplica(o, T, wl.translate_step, wl.rotate_step, r, pos=first.pos, rel=first.rel,
                                    center=first.center, quat=first.quat, energy=first.energy, step=before)
        orec = orep.mc(seed=SEED, nsteps=n3, mode=0)
        n_eq, div = compare_decisions(e.records(r), orec, T, rel_tol=1e-5)
        if div:
            diverged += 1
            continue
        st = e.state(r)
        for k, want in (("pos", orep.pos), ("rel", orep.rel), ("center", orep.center), ("quat", orep.quat)):
            assert np.array_equal(st[k], want), (r, k)
        assert abs(energies[r] - orep.energy) < 1e-4 * kT(T) + 1e-5 * abs(orep.energy)
    e.close()
    assert diverged <= 1
