"""Runs whose HIP calls are refused part of the way: an error or another path, and
the next call as if nothing had been."""
import pytest

from tests import hip_refuse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("after", [0, 1, 2])
def test_refused_stepping_launch(tmp_path, after):
    """The first, second or third launch of the stepping kernel is refused: an
    error, and the next run of the job steps by it again (with stats, the steps it
    took and the initial pass; launches would have 1 in 16 of them timed)."""
    hip_refuse.run(tmp_path, """
job = g.synth_complex(4001, 46, 5, 11, 4, floor_temp=0.05, ceiling_temp=0.3, seed=4, ene=ene)
dev = g.DeviceJob(job)
mc = g.make_mc(30, steps_per_exchange=10, seed=3)
want, st = dev.dock(mc)
assert st.n_pair_launch == 31
shim.refuse_stepping_after(%d)
try:
    dev.dock(mc)
    raise SystemExit("a refused launch went unnoticed")
except g.GDError:
    pass
for _ in range(2):
    out, st = dev.dock(mc)
    same(want, out)
    assert st.n_pair_launch == 31, st.n_pair_launch
""" % after)


_SERVE = """
jobs = [g.synth_complex(700 + 40 * k, 21 + k, 13, 5, 2, floor_temp=0.05, ceiling_temp=0.3, seed=k + 1, ene=ene)
        for k in range(3)]
mcs = [g.make_mc(40 + 9 * k, steps_per_exchange=7 + k, seed=3, job_id=k, axes=("temp", "lig")) for k in range(3)]

def serve(refuse):
    s = C.c_void_p()
    cfg = abi.gd_server_config(hbm_budget=64 << 30, max_active=3, sweep_steps=13)
    g.check(g.lib().gd_server_create(C.byref(cfg), C.byref(s)), "create")
    outs = [g.host.ReplicaOut(j.n_rep) for j in jobs]
    for j, mc, o in zip(jobs, mcs, outs):
        t = C.c_int64()
        g.check(g.lib().gd_server_submit(s, C.byref(j.desc), C.byref(mc), C.byref(o.c), C.byref(t)), "submit")
    done = errors = 0
    for k in range(40):
        if k in refuse:
            refuse[k](s)
        na, nd, n, res = C.c_int(), C.c_int(), C.c_int(), (abi.gd_job_result * 8)()
        errors += g.lib().gd_server_step(s, C.byref(na), C.byref(nd)) != 0
        shim.refuse_device_over(NONE)
        g.lib().gd_server_results(s, res, 8, C.byref(n))
        assert all(res[i].status == 0 for i in range(n.value))
        done += n.value
        if done == 3:
            break
    assert done == 3
    g.lib().gd_server_destroy(s)
    return outs, errors

want, errors = serve({})
assert errors == 0
"""


@pytest.mark.parametrize("after", [0, 1])
def test_refused_sweep(tmp_path, after):
    """The first or second stepping launch of a sweep is refused: the call is an
    error, and the next ones take the steps that it did not."""
    hip_refuse.run(tmp_path, _SERVE + """
got, errors = serve({1: lambda s: shim.refuse_stepping_after(%d)})
assert errors == 1
for a, b in zip(want, got):
    same(a, b)
""" % after)


def test_refused_sweep_after_a_time_out(tmp_path):
    """The first stepping launch of a sweep runs out of time and the second is refused:
    the sweep is taken again from its start."""
    hip_refuse.run(tmp_path, _SERVE + """
def both(s):
    g.check(g.lib().gd_server_set_step_wait(s, 0.0), "wait")
    shim.refuse_stepping_after(1)

got, errors = serve({1: both, 2: lambda s: g.check(g.lib().gd_server_set_step_wait(s, 2.0), "wait")})
assert errors == 1
for a, b in zip(want, got):
    same(a, b)
""")


def test_refused_lists(tmp_path):
    """No memory for the lists of a sweep whose jobs have changed: an error, and
    the lists are made by the next call."""
    hip_refuse.run(tmp_path, _SERVE + """
got, errors = serve({k: lambda s: shim.refuse_device_over(0) for k in range(1, 8)})
assert errors >= 1
for a, b in zip(want, got):
    same(a, b)
""")


def test_no_pinned_memory(tmp_path):
    """No pinned memory at all from the first call on: evaluations, runs, batches,
    the served requests and the read-back give what they give with it."""
    hip_refuse.run(tmp_path, _SERVE.replace("want, errors = serve({})\nassert errors == 0", "") + """
from tests.oracle_ffi import random_poses
ip, fp = C.POINTER(C.c_int), C.POINTER(C.c_float)
small = g.synth_complex(300, 9, 3, 2, 1, seed=1, ene=ene)
large = g.synth_complex(4001, 46, 5, 11, 4, floor_temp=0.05, ceiling_temp=0.3, seed=4, ene=ene)

def everything():
    got = []
    for job in (small, large):
        dev = g.DeviceJob(job)
        for n in (1, 130, 2500):
            conf, pose = random_poses(job, n, seed=n, trans=2.0)
            conf, pose = np.ascontiguousarray(conf, np.int32), np.ascontiguousarray(pose, np.float32)
            got += list(dev.eval(conf, pose, want_coords=True))
            terms, raw = np.zeros((n, 10), np.float32), np.zeros((n, 9), np.float32)
            for r in (raw.ctypes.data_as(fp), None):
                g.check(g.lib().gd_energy_eval_noalloc(dev.h, n, conf.ctypes.data_as(ip), pose.ctypes.data_as(fp),
                                                       terms.ctypes.data_as(fp), r), "noalloc")
            got += [terms, raw]
        for wait in (2.0, 0.0):  # 0: the failure word comes by a copy, too
            dev.set_step_wait(wait)
            out, st = dev.dock(g.make_mc(24, steps_per_exchange=7, seed=3, axes=("temp", "lig", "prt")))
            back = dev.replicas()
            for o in (out, back):
                got += [getattr(o, f).copy() for f in FIELDS]
        outs = [g.host.ReplicaOut(job.n_rep)]
        mc = g.make_mc(9, steps_per_exchange=4, seed=3)
        g.check(g.lib().gd_batch_dock(C.byref(dev.h), 1, C.byref(mc), C.byref(outs[0].c), None), "batch")
        got += [getattr(outs[0], f).copy() for f in FIELDS]
        dev.close()
    outs, errors = serve({})
    assert errors == 0
    return got + [getattr(o, f).copy() for o in outs for f in FIELDS]

shim.refuse_pinned_over(0)
a = everything()
assert shim.refused_pinned() > 0
shim.refuse_pinned_over(NONE)
b = everything()
assert len(a) == len(b)
for x, y in zip(a, b):
    assert np.array_equal(x, y)
""")
