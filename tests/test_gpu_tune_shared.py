"""The shared sweep measures what a batch takes."""
import ctypes as C
import time

import pytest

import geauxdock_amd as g
from geauxdock_amd import abi

pytestmark = pytest.mark.gpu


def test_sweep_times_the_path_of_batches(ene):
    """The table's tile is one of the candidates, so the best time is at most that of
    the batch as it is (a tenth for noise; by launches it is a third longer)."""
    jobs = [g.synth_complex(1200, 24, 5, 5, 1, seed=k + 1, ene=ene) for k in range(64)]
    devs = [g.DeviceJob(j) for j in jobs]
    lc, pt, _ = g.host.tiling_lookup(24, 1200, 25, True)
    assert lc == 4 and pt in (32, 40, 48, 64, 80, 96, 128)
    arr = (C.c_void_p * 64)(*[d.h for d in devs])
    mc = [g.make_mc(400, move_mode="gaussian", seed=1, job_id=k) for k in range(64)]
    mcs = (abi.gd_mc_param * 64)(*mc)
    times = []
    for _ in range(6):
        t = time.perf_counter()
        g.check(g.lib().gd_batch_dock(arr, 64, mcs, None, None), "batch")
        times.append(1e3 * (time.perf_counter() - t))
    best, ms = abi.gd_tiling(), C.c_double()
    g.check(g.lib().gd_autotune_shared(arr, 64, 400, C.byref(best), C.byref(ms)), "tune")
    print("batch %s ms, sweep %.2f ms at %d points, %d waves" % (["%.2f" % x for x in times], ms.value,
                                                                  best.tile_points, best.waves_per_cu))
    assert ms.value <= 1.1 * sorted(times)[len(times) // 2]
    for d in devs:
        assert d.tiling() == (lc, pt)
        d.close()
