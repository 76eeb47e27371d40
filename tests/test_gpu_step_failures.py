"""Runs in which a wait of the stepping kernel runs out of time (a bound of 0 ends
every launch at its first wait): the same bits as without.  The complexes are
above the line from which plain runs step by the kernel, which the counts of timed
launches show: the kernel counts every step and the initial pass, launches 1 step
in 16."""
import ctypes as C

import numpy as np
import pytest

import geauxdock_amd as g
from geauxdock_amd import abi
from geauxdock_amd.host import ReplicaOut

pytestmark = pytest.mark.gpu

FIELDS = ("energy", "movematrix", "idx_tmp", "n_accept", "n_exchange", "best_energy", "is_accept", "n_swap_lig",
          "n_swap_prt")
FOUR = (4001, 46, 5, 11, 4)    # four blocks, 960 items
SEVEN = (3000, 40, 10, 11, 4)  # seven blocks


def _same(a, b):
    for f in FIELDS:
        assert np.array_equal(getattr(a, f), getattr(b, f)), f


def _job(ene, shape, seed=4):
    return g.synth_complex(*shape, floor_temp=0.05, ceiling_temp=0.3, seed=seed, ene=ene)


def _batch(devs, mcs, stats=False):
    outs = [ReplicaOut(d.n_rep) for d in devs]
    arr = (C.c_void_p * len(devs))(*[d.h for d in devs])
    oc = (abi.gd_replica_out * len(devs))(*[o.c for o in outs])
    st = abi.gd_stats()
    g.check(g.lib().gd_batch_dock(arr, len(devs), (abi.gd_mc_param * len(devs))(*mcs), oc,
                                  C.byref(st) if stats else None), "gd_batch_dock")
    return outs, st


# launches of one step, two and five follow the one that failed
@pytest.mark.parametrize("spe", [1, 2, 5])
@pytest.mark.parametrize("shape", [FOUR, SEVEN])
def test_plain(ene, shape, spe):
    dev = g.DeviceJob(_job(ene, shape))
    mc = g.make_mc(16, steps_per_exchange=spe, seed=3, axes=("temp", "lig", "prt"))
    want, st = dev.dock(mc)
    assert st.n_pair_launch == 17
    dev.set_step_wait(0.0)
    for _ in range(2):
        out, st = dev.dock(mc)
        _same(want, out)
        assert 0 < st.n_pair_launch < 16
    dev.set_step_wait(2.0)
    out, st = dev.dock(mc)
    _same(want, out)
    assert st.n_pair_launch == 17
    dev.close()


@pytest.mark.parametrize("spe", [1, 3])
def test_batch(ene, spe):
    devs = [g.DeviceJob(_job(ene, s, seed=k + 1)) for k, s in enumerate([FOUR, (300, 9, 3, 2, 1), SEVEN])]
    mcs = [g.make_mc(9 + 4 * k, steps_per_exchange=spe, seed=3, job_id=k, axes=("temp", "lig")) for k in range(3)]
    want, st = _batch(devs, mcs, stats=True)
    assert st.n_pair_launch == 18
    devs[1].set_step_wait(0.0)
    got, st = _batch(devs, mcs, stats=True)
    assert 0 < st.n_pair_launch < 17
    for a, b in zip(want, got):
        _same(a, b)
    for d in devs:
        d.close()


def _serve(jobs, mcs, wait, sweep=7, calls=80):
    s = C.c_void_p()
    cfg = abi.gd_server_config(hbm_budget=64 << 30, max_active=len(jobs), sweep_steps=sweep)
    g.check(g.lib().gd_server_create(C.byref(cfg), C.byref(s)), "create")
    outs = [ReplicaOut(j.n_rep) for j in jobs]
    for j, mc, o in zip(jobs, mcs, outs):
        t = C.c_int64()
        g.check(g.lib().gd_server_submit(s, C.byref(j.desc), C.byref(mc), C.byref(o.c), C.byref(t)), "submit")
    done = 0
    for k in range(calls):
        if k in wait:
            g.check(g.lib().gd_server_set_step_wait(s, wait[k]), "wait")
        na, nd, n, res = C.c_int(), C.c_int(), C.c_int(), (abi.gd_job_result * 8)()
        g.check(g.lib().gd_server_step(s, C.byref(na), C.byref(nd)), "step")
        g.lib().gd_server_results(s, res, 8, C.byref(n))
        assert all(res[i].status == 0 for i in range(n.value))
        done += n.value
        if done == len(jobs):
            break
    g.lib().gd_server_destroy(s)
    assert done == len(jobs)
    return outs, k + 1


@pytest.mark.parametrize("spe", [1, 4])
@pytest.mark.parametrize("at", [0, 2])
def test_server(ene, spe, at):
    """The bound is set before the first sweep, and before the third."""
    jobs = [_job(ene, s, seed=k + 1) for k, s in enumerate([FOUR, (300, 9, 3, 2, 1), (700, 21, 13, 5, 4)])]
    mcs = [g.make_mc(20 + 9 * k, steps_per_exchange=spe, seed=3, job_id=k, axes=("temp", "lig")) for k in range(3)]
    want, _ = _serve(jobs, mcs, {})
    got, _ = _serve(jobs, mcs, {at: 0.0})
    for a, b in zip(want, got):
        _same(a, b)
