"""Runs in which a wait of the stepping kernel runs out of time (a bound of 0 ends
every launch at its first wait): the same bits as without.  The complexes are
above the line from which plain runs step by the kernel, which the counts of timed
launches show: the kernel counts every step and the initial pass, launches 1 step
in 16."""
import ctypes as C
import threading
import time

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


@pytest.mark.parametrize("blocking", [False, True])
@pytest.mark.parametrize("dump,spe", [(5, 4), (1, 0), (7, 7), (20, 3)])
def test_streamed(ene, dump, spe, blocking):
    """Every dump is handed over once, and is that of a run by launches: whole runs
    that fail in their first dump, on a job that steps by the kernel before and
    after."""
    dev = g.DeviceJob(_job(ene, FOUR))
    mc = g.make_mc(20, steps_per_dump=dump, steps_per_exchange=spe, seed=3, axes=("temp", "lig"))
    runs = []
    for way in ("kernel", "failing", "kernel", "launches"):
        dev.set_step_wait(0.0 if way == "failing" else 2.0)
        if way == "launches":
            dev.set_streams(1)
        dumps = []
        out, st = dev.dock_stream(mc, lambda k, s0, rec, cnt: dumps.append((k, s0, rec, cnt)), blocking=blocking)
        assert (st.n_pair_launch == 21) == (way == "kernel"), (way, st.n_pair_launch)
        runs.append((out, dumps))
    assert [d[:2] for d in runs[0][1]] == [(k, s) for k, s in enumerate(range(0, 20, dump))]
    for out, dumps in runs[1:]:
        _same(runs[0][0], out)
        assert [d[:2] for d in dumps] == [d[:2] for d in runs[0][1]]
        for a, b in zip(dumps, runs[0][1]):
            keep = np.arange(a[2].shape[1])[None, :] < a[3][:, None]
            assert np.array_equal(a[3], b[3]) and np.array_equal(a[2][keep], b[2][keep])
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
    want, calls = _serve(jobs, mcs, {})
    got, more = _serve(jobs, mcs, {at: 0.0})
    for a, b in zip(want, got):
        _same(a, b)
    assert more == calls + 1  # only the sweep that failed is taken again


def test_server_tries_again(ene):
    """256 sweeps by launches, then the stepping kernel again (which fails again)."""
    jobs = [_job(ene, (700, 21, 13, 5, 4))]
    mcs = [g.make_mc(300, steps_per_exchange=7, seed=3, axes=("temp", "lig"))]
    want, calls = _serve(jobs, mcs, {}, sweep=1, calls=400)
    assert calls == 300
    got, more = _serve(jobs, mcs, {5: 0.0}, sweep=1, calls=400)
    _same(want[0], got[0])
    assert more == 302


@pytest.mark.parametrize("wait", [{}, {2: 0.0}])
def test_converging_server(ene, wait):
    """A sweep that is taken again counts once towards convergence."""
    jobs = [_job(ene, FOUR), _job(ene, (700, 21, 13, 5, 4), seed=5)]
    mcs = [g.make_mc(4000, steps_per_exchange=5, seed=3, job_id=k) for k in range(2)]
    steps = []
    for w in ({}, wait):
        s = C.c_void_p()
        cfg = abi.gd_server_config(hbm_budget=64 << 30, max_active=2, sweep_steps=10, converge_sweeps=3,
                                   converge_tol=0.02)
        g.check(g.lib().gd_server_create(C.byref(cfg), C.byref(s)), "create")
        for j, mc in zip(jobs, mcs):
            g.check(g.lib().gd_server_submit(s, C.byref(j.desc), C.byref(mc), None, None), "submit")
        got = {}
        for k in range(450):
            if k in w:
                g.check(g.lib().gd_server_set_step_wait(s, w[k]), "wait")
            n, res = C.c_int(), (abi.gd_job_result * 8)()
            g.check(g.lib().gd_server_step(s, None, None), "step")
            g.lib().gd_server_results(s, res, 8, C.byref(n))
            for r in res[:n.value]:
                assert r.status == 0
                got[r.ticket] = r.replica_steps
            if len(got) == 2:
                break
        g.lib().gd_server_destroy(s)
        steps.append(got)
    assert steps[0] == steps[1] and len(steps[0]) == 2
    assert all(v < 4000 * j.n_rep for v, j in zip(steps[0].values(), jobs))


# Runs that fail after a state was kept (once in about 0.2 s): they go on from it.


@pytest.mark.parametrize("blocking", [False, True])
def test_streamed_run_goes_on(ene, blocking):
    """The bound is set to 0 once dump 5 of 10 was handed over, when 12,000 or
    14,000 of 20,000 steps were launched and states were kept: every dump
    is handed over once and is that of a run by launches."""
    dev = g.DeviceJob(_job(ene, FOUR))
    mc = g.make_mc(20000, steps_per_dump=2000, steps_per_exchange=100, seed=3, axes=("temp", "lig", "prt"))
    runs = []
    for fail in (False, True):
        dumps = []

        def take(k, s0, rec, cnt):
            keep = np.arange(rec.shape[1])[None, :] < cnt[:, None]
            dumps.append((k, s0, cnt, rec[keep].copy()))
            if fail and k == 5:
                dev.set_step_wait(0.0)

        out, st = dev.dock_stream(mc, take, blocking=blocking)
        runs.append((out, dumps))
        if fail:  # timed launches, 1 step in 16 on two streams: of 12,000 steps at most
            assert 0 < st.n_pair_launch <= 2 * (12000 // 16 + 1), st.n_pair_launch
        else:
            assert st.n_pair_launch == 20001
    _same(runs[0][0], runs[1][0])
    assert [d[:2] for d in runs[1][1]] == [(k, 2000 * k) for k in range(10)]
    for a, b in zip(runs[0][1], runs[1][1]):
        assert np.array_equal(a[2], b[2]) and np.array_equal(a[3], b[3])
    dev.set_step_wait(2.0)
    out, st = dev.dock(g.make_mc(20, seed=3))  # the kept state is of that run only
    assert st.n_pair_launch == 21
    dev.set_step_wait(0.0)
    again, _ = dev.dock(g.make_mc(20, seed=3))
    _same(out, again)
    dev.close()


def _timed(run):
    t = time.perf_counter()
    return run(), time.perf_counter() - t


def _fail_after(devs, run, seconds):
    t = threading.Timer(seconds, lambda: [d.set_step_wait(0.0) for d in devs])
    t.start()
    try:
        return run()
    finally:
        t.cancel()
        t.join()


def test_plain_run_goes_on(ene):
    """More launches than the device's queue holds, so that the bound, set to 0 after
    half the time, counts for the later ones."""
    dev = g.DeviceJob(_job(ene, FOUR))
    mc = g.make_mc(30000, steps_per_exchange=2, seed=3, axes=("temp", "lig", "prt"))
    (want, st), seconds = _timed(lambda: dev.dock(mc))
    assert st.n_pair_launch == 30001
    out, st = _fail_after([dev], lambda: dev.dock(mc), seconds / 2)
    _same(want, out)
    assert 0 < st.n_pair_launch <= 2 * (22000 // 16 + 1), st.n_pair_launch
    dev.close()


# the same lengths (captured launches); unlike ones, of which the shortest ends before
# the failure
@pytest.mark.parametrize("steps,stats", [((12000, 12000, 12000), False), ((12000, 900, 11000), True)])
def test_batch_goes_on(ene, steps, stats):
    devs = [g.DeviceJob(_job(ene, s, seed=k + 1)) for k, s in enumerate([SEVEN, (300, 9, 3, 2, 1), SEVEN])]
    mcs = [g.make_mc(n, steps_per_exchange=48, seed=3, job_id=k, axes=("temp", "lig")) for k, n in enumerate(steps)]
    (want, _), seconds = _timed(lambda: _batch(devs, mcs))
    got, st = _fail_after(devs[:1], lambda: _batch(devs, mcs, stats=stats), 0.6 * seconds)
    for a, b in zip(want, got):
        _same(a, b)
    if stats:  # by launches from a kept state on
        assert 0 < st.n_pair_launch <= 10000 // 16, st.n_pair_launch
    for d in devs:
        d.close()


def test_batch_fails_before_its_list_shrinks(ene):
    """Only the job that ends at step 9,000 bounds the waits to 0, from step 6,000 or so
    on: the launches after it has left the list run in time, on a state that is not
    to be kept."""
    devs = [g.DeviceJob(_job(ene, SEVEN, seed=k + 1)) for k in range(2)]
    mcs = [g.make_mc(n, steps_per_exchange=48, seed=3, job_id=k, axes=("temp", "lig"))
           for k, n in enumerate((26000, 9000))]
    _, first = _timed(lambda: _batch(devs, [mcs[1], mcs[1]]))
    want, _ = _batch(devs, mcs)
    got, st = _fail_after(devs[1:], lambda: _batch(devs, mcs, stats=True), 0.7 * first)
    assert 0 < st.n_pair_launch < 26000 // 16
    for a, b in zip(want, got):
        _same(a, b)
    for d in devs:
        d.close()
