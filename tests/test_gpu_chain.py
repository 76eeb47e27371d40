"""The stepping kernel (all MC steps between exchange points in one launch)
against stepping by launches (gd_job_set_streams): the same bits."""
import numpy as np
import pytest

import geauxdock_amd as g

pytestmark = pytest.mark.gpu

FIELDS = ("energy", "movematrix", "idx_tmp", "n_accept", "n_exchange", "best_energy", "is_accept", "n_swap_lig",
          "n_swap_prt")


def _same(a, b):
    for f in FIELDS:
        assert np.array_equal(getattr(a, f), getattr(b, f)), f


# one block (launches), two and many; fewer and more tickets than resident
# groups; one-chunk and two-atom ligands; a tile count over the common reduce
# shapes; whole tiles without points
@pytest.mark.parametrize("P,L,nl,np_,nt,steps,spe,axes", [
    (1200, 24, 16, 4, 1, 20, 0, ("temp",)),
    (37, 2, 13, 5, 1, 9, 4, ("temp", "lig", "prt")),
    (400, 5, 13, 5, 1, 12, 5, ("lig",)),
    (4001, 46, 5, 11, 4, 12, 5, ("temp", "lig", "prt")),
    (3000, 40, 20, 11, 8, 9, 4, ("temp", "lig", "prt")),
    (9000, 80, 5, 11, 4, 5, 2, ("prt",)),
])
def test_chain_matches_launches(ene, P, L, nl, np_, nt, steps, spe, axes):
    job = g.synth_complex(P, L, nl, np_, nt, floor_temp=0.05, ceiling_temp=0.3, seed=P + L, ene=ene)
    res = []
    for by_launches in (False, True):
        dev = g.DeviceJob(job)
        if by_launches:
            dev.set_streams(1)
        for n, record in ((0, False), (steps, False), (steps, True)):
            mc = g.make_mc(n, steps_per_dump=max(1, n // 2), steps_per_exchange=spe, seed=3, axes=axes,
                           record=record, move_mode="gaussian" if record else "reference")
            out, _ = dev.dock(mc)
            res.append((out, dev.records(max(1, n // 2)) if record else None))
        dev.close()
    for (a, ra), (b, rb) in zip(res[:3], res[3:]):
        _same(a, b)
        if ra is not None:
            assert np.array_equal(ra[1], rb[1])
            keep = np.arange(ra[0].shape[1])[None, :] < ra[1][:, None]
            assert np.array_equal(ra[0][keep], rb[0][keep])


# a wait bound of 0 ends every launch at its first wait: the run is repeated by
# launches, and a streamed run hands every dump over once
def test_out_of_time_repeats_by_launches(ene):
    job = g.synth_complex(400, 5, 13, 5, 1, floor_temp=0.05, ceiling_temp=0.3, seed=4, ene=ene)
    mc = g.make_mc(20, steps_per_dump=5, steps_per_exchange=4, seed=3, axes=("temp", "lig"), record=True)
    res = []
    for wait in (0.0, 2.0, 0.0):
        dev = g.DeviceJob(job)
        dev.set_step_wait(wait)
        for blocking in (False, True):
            dumps = []

            def take(k, s0, rec, cnt):
                dumps.append((k, s0, [r[:n].copy() for r, n in zip(rec, cnt)]))

            out, _ = dev.dock_stream(mc, take, blocking=blocking)
            res.append((out, dumps))
        dev.set_step_wait(2.0)
        res.append((dev.dock(mc)[0], res[-1][1]))  # the same job after a failed launch
        dev.close()
    assert [d[0] for d in res[0][1]] == [0, 1, 2, 3]
    for out, dumps in res[1:]:
        _same(res[0][0], out)
        assert [d[:2] for d in dumps] == [d[:2] for d in res[0][1]]
        for a, b in zip(dumps, res[0][1]):
            assert all(np.array_equal(x, y) for x, y in zip(a[2], b[2]))


def test_threads_dock_side_by_side(ene):
    import threading
    jobs = [g.synth_complex(900 + 50 * k, 20, 13, 10, 1, seed=k, ene=ene) for k in range(3)]
    mc = g.make_mc(60, steps_per_exchange=20, seed=3)
    want = []
    for job in jobs:
        dev = g.DeviceJob(job)
        dev.set_streams(1)
        want.append(dev.dock(mc)[0])
        dev.close()
    got = [None] * 3

    def run(k):
        dev = g.DeviceJob(jobs[k])
        got[k] = [dev.dock(mc)[0] for _ in range(5)]
        dev.close()

    t = [threading.Thread(target=run, args=(k,)) for k in range(3)]
    [x.start() for x in t]
    [x.join() for x in t]
    for k in range(3):
        for out in got[k]:
            _same(want[k], out)


# lists of jobs: one block (launches), many small ones, jobs of unlike sizes whose
# lengths and exchange intervals differ, more blocks than finishers
LISTS = {
    "one block": [(300, 9, 3, 2, 1)],
    "small": [(500 + 7 * k, 8 + k, 5, 5, 1) for k in range(12)],
    "unlike": [(37, 2, 1, 1, 1), (3000, 40, 10, 11, 4), (700, 30, 13, 5, 1), (1200, 24, 5, 5, 2)],
    "blocks": [(150, 6, 16, 8, 5) for _ in range(7)],
}


def _batch(devs, mcs, stats=False):
    import ctypes as C
    from geauxdock_amd import abi
    outs = [g.host.ReplicaOut(d.n_rep) for d in devs]
    arr = (C.c_void_p * len(devs))(*[d.h for d in devs])
    oc = (abi.gd_replica_out * len(devs))(*[o.c for o in outs])
    st = abi.gd_stats()
    g.check(g.lib().gd_batch_dock(arr, len(devs), (abi.gd_mc_param * len(devs))(*mcs), oc,
                                  C.byref(st) if stats else None), "gd_batch_dock")
    return outs, st


@pytest.mark.parametrize("name", list(LISTS))
@pytest.mark.parametrize("steps,spe", [(0, 0), (11, 4), (30, 0)])
def test_batch_chain_matches_launches(ene, name, steps, spe):
    """A wait bound of 0 has the batch repeated by launches."""
    jobs = [g.synth_complex(*s, seed=k + 1, ene=ene) for k, s in enumerate(LISTS[name])]
    devs = [g.DeviceJob(j) for j in jobs]
    ragged = name == "unlike"
    mcs = [g.make_mc(steps + (3 * k if ragged and steps else 0), steps_per_exchange=spe + (k if ragged and spe else 0),
                     seed=3, job_id=k, move_mode="gaussian", axes=("temp", "lig", "prt")) for k in range(len(jobs))]
    a, st = _batch(devs, mcs, stats=True)
    b, _ = _batch(devs, mcs)
    devs[-1].set_step_wait(0.0)
    c, _ = _batch(devs, mcs)
    devs[-1].set_step_wait(2.0)
    d, _ = _batch(devs, mcs)
    for k in range(len(jobs)):
        for o in (b, c, d):
            _same(a[k], o[k])
    assert steps == 0 or st.n_pair_launch > 0
    for x in devs:
        x.close()


def test_server_chain_matches_launches(ene):
    import ctypes as C
    from geauxdock_amd import abi
    jobs = [g.synth_complex(*s, seed=k + 1, ene=ene) for k, s in enumerate(LISTS["unlike"])]
    mcs = [g.make_mc(20 + 9 * k, steps_per_exchange=4 + k, seed=3, job_id=k, axes=("temp", "lig")) for k in range(4)]
    got = []
    for wait in (2.0, 0.0):
        s = C.c_void_p()
        cfg = abi.gd_server_config(hbm_budget=64 << 30, max_active=3, sweep_steps=13)
        g.check(g.lib().gd_server_create(C.byref(cfg), C.byref(s)), "create")
        g.check(g.lib().gd_server_set_step_wait(s, wait), "wait")
        outs = [g.host.ReplicaOut(j.n_rep) for j in jobs]
        for j, mc, o in zip(jobs, mcs, outs):
            t = C.c_int64()
            g.check(g.lib().gd_server_submit(s, C.byref(j.desc), C.byref(mc), C.byref(o.c), C.byref(t)), "submit")
        done = 0
        for _ in range(60):
            na, nd, n, res = C.c_int(), C.c_int(), C.c_int(), (abi.gd_job_result * 8)()
            g.check(g.lib().gd_server_step(s, C.byref(na), C.byref(nd)), "step")
            g.lib().gd_server_results(s, res, 8, C.byref(n))
            assert all(res[i].status == 0 for i in range(n.value))
            done += n.value
            if done == 4:
                break
        assert done == 4
        g.lib().gd_server_destroy(s)
        got.append(outs)
    for a, b in zip(*got):
        _same(a, b)


@pytest.mark.parametrize("bad", [-1.0, 61.0, float("nan")])
def test_bad_wait(ene, bad):
    dev = g.DeviceJob(g.synth_complex(40, 4, 2, 2, 1, seed=1, ene=ene))
    with pytest.raises(g.GDError):
        dev.set_step_wait(bad)
    dev.close()
