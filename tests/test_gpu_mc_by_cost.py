"""MC workgroups by the systems' cost, asked for and carried to another context:
the costly replicas have more than eight members (two polls of a slot row), the
decisions are the FP64 oracle's (bars of test_gpu_mc_members), and a context set
to another's configuration takes the same steps bit for bit without tuning."""
import numpy as np
import pytest

from helpers import compare_decisions, engine_for, kT, say
from remcdockingsimulator_amd import synth
from remcdockingsimulator_amd.engine import Engine
from test_gpu_mc_members import SEED
from test_gpu_mc_members import workload as members_workload

pytestmark = pytest.mark.gpu


def workload(light=290):
    """That of test_gpu_mc_members with `light` replicas of the light system."""
    wl = members_workload()
    wl.temperatures[0] = synth.geometric_ladder(290.0, 420.0, light)
    return wl


# 1024 threads: one workgroup per CU, so 256 for all members of all replicas
@pytest.mark.parametrize("block,lds_cache,window,light", [(256, True, True, 290), (256, False, True, 290),
                                                          (1024, False, True, 120), (512, True, False, 290)])
def test_parity_of_a_plan_by_cost(oracle, block, lds_cache, window, light):
    wl = workload(light)
    e = engine_for(wl, seed=SEED, block=block)
    e.set_mc_by_cost()
    e.set_mc_tuning(lds_cache=lds_cache, split_min_pairs=64)
    e.set_mc_window(window)
    n1, n2, heavy = 90, 60, light  # heavy: the first replica of the costly system
    e.mc_steps(n1)
    by_cost, most = e.mc_by_cost()
    say("block", block, "cache", lds_cache, "window", window, "largest number of members", most)
    assert by_cost and 8 < most <= 32 and e.mc_block() == block and e.mc_coop() == 1
    e.mc_steps_plain(heavy, 5)  # host steps change the canonical state only
    e.set_recording(n2)
    e.run(2, n2 // 2)
    e.synchronize()
    assert e.mc_by_cost() == (True, most)
    diverged = 0
    for r, sys in ((heavy, 1), (light - 1, 0)):
        # (up to the first exchange, at the rung's own temperature)
        T = float(np.concatenate(wl.temperatures)[r])
        o = oracle.OracleSystem(wl.systems[sys], wl.ff)
        first = oracle.OracleReplica(o, T, wl.translate_step, wl.rotate_step, r)
        before = n1 + (5 if r == heavy else 0)
        first.mc(seed=SEED, nsteps=before, mode=0)
        orep = oracle.OracleReplica(o, T, wl.translate_step, wl.rotate_step, r, pos=first.pos, rel=first.rel,
                                    center=first.center, quat=first.quat, energy=first.energy, step=before)
        orec = orep.mc(seed=SEED, nsteps=n2 // 2, mode=0)
        n_eq, div = compare_decisions(e.records(r)[:n2 // 2], orec, T, rel_tol=1e-5)
        diverged += div
    full, tracked = e.energy_all(), e.energies()
    assert np.all(np.abs(full - tracked) <= 1e-4 * kT(290.0) + 1e-5 * np.abs(full))
    e.close()
    assert diverged <= 1


def test_a_configuration_is_carried_over():
    wl = workload()
    a = engine_for(wl, seed=SEED)
    assert a.mc_by_cost() == (False, 0)
    a.set_mc_by_cost()
    a.mc_steps(40)
    assert a.mc_by_cost()[0]
    b = engine_for(wl, seed=SEED)
    b.set_mc_block(a.mc_block())
    b.set_mc_coop(a.mc_coop())
    assert not b.mc_by_cost()[0]
    b.set_mc_by_cost(a.mc_by_cost()[0])
    b.mc_steps(40)
    assert b.mc_by_cost() == a.mc_by_cost() and b.mc_block() == a.mc_block()
    assert np.array_equal(a.energies(), b.energies()) and np.array_equal(a.counters(), b.counters())
    for r in (0, 289, 290, 291):
        sa, sb = a.state(r), b.state(r)
        assert all(np.array_equal(sa[k], sb[k]) for k in sa)
    # a number of its own, or none, ends it
    b.set_mc_coop(1)
    b.mc_steps(4)
    assert b.mc_by_cost() == (False, 1)
    b.set_mc_by_cost(False)
    b.mc_steps(4)
    assert b.mc_by_cost()[1] >= 1
    a.close()
    b.close()


def test_one_system_is_tuned_as_ever():
    wl = synth.config(1)
    e = Engine(0)
    synth.load_engine(e, wl, seed=SEED)
    e.set_mc_by_cost()
    e.mc_steps(8)
    on, most = e.mc_by_cost()
    assert not on and most == e.mc_coop() >= 1
    e.close()
