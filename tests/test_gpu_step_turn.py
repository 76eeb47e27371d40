"""The turn at the stepping kernel, which one run of the process has at a time: with
stats a run by it counts every step and the initial pass, one by launches 1 step in
16."""
import threading

import numpy as np
import pytest

import geauxdock_amd as g

pytestmark = pytest.mark.gpu

FIELDS = ("energy", "movematrix", "idx_tmp", "n_accept", "n_exchange", "best_energy", "is_accept", "n_swap_lig",
          "n_swap_prt")


def _together(fns):
    errors = []

    def call(f):
        try:
            f()
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    t = [threading.Thread(target=call, args=(f,)) for f in fns]
    [x.start() for x in t]
    [x.join() for x in t]
    assert not errors, errors


def test_runs_that_do_not_step_by_it_leave_it(ene):
    """Runs of a one-block job, which is stepped by launches, beside those of a
    large one: every run of the large one has the turn."""
    small = g.DeviceJob(g.synth_complex(300, 9, 3, 2, 1, seed=1, ene=ene))
    large = g.DeviceJob(g.synth_complex(4001, 46, 5, 11, 4, seed=2, ene=ene))
    mc = g.make_mc(40, steps_per_exchange=20, seed=3)
    want, st = large.dock(mc)
    assert st.n_pair_launch == 41
    stop, counts = threading.Event(), []

    def one():
        while not stop.is_set():
            small.dock(g.make_mc(400, seed=3))

    def other():
        try:
            for _ in range(20):
                out, st = large.dock(mc)
                counts.append(st.n_pair_launch)
                assert np.array_equal(out.energy, want.energy)
        finally:
            stop.set()

    _together([one, other])
    assert counts == [41] * 20
    small.close()
    large.close()


def test_large_runs_side_by_side(ene):
    """Three threads' jobs that all suit the kernel: the same bits by either way of
    stepping."""
    jobs = [g.synth_complex(4001 - 100 * k, 46 - k, 5, 11, 4, floor_temp=0.05, ceiling_temp=0.3, seed=k, ene=ene)
            for k in range(3)]
    devs = [g.DeviceJob(j) for j in jobs]
    mc = g.make_mc(40, steps_per_exchange=20, seed=3, axes=("temp", "lig", "prt"))
    want = []
    for d in devs:
        out, st = d.dock(mc)
        assert st.n_pair_launch == 41
        want.append(out)

    def run(k):
        for _ in range(8):
            out, _ = devs[k].dock(mc)
            for f in FIELDS:
                assert np.array_equal(getattr(out, f), getattr(want[k], f)), f

    _together([lambda k=k: run(k) for k in range(3)])
    for d in devs:
        d.close()


def test_default_streams(ene):
    """Two streams are the default: setting them changes nothing, and after another
    number they bring the default back."""
    dev = g.DeviceJob(g.synth_complex(4001, 46, 5, 11, 4, seed=2, ene=ene))
    mc = g.make_mc(24, steps_per_exchange=20, seed=3)
    want, st = dev.dock(mc)
    assert st.n_pair_launch == 25
    for n, launches in ((2, 25), (1, 2), (2, 25), (4, 8), (3, 6), (2, 25)):
        dev.set_streams(n)
        out, st = dev.dock(mc)
        assert np.array_equal(out.energy, want.energy)
        assert st.n_pair_launch == launches, (n, st.n_pair_launch)
    dev.close()
