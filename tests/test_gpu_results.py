"""Start state and results of runs: written and gathered on the device for one
job and for lists of jobs (40 to a launch)."""
import ctypes as C

import numpy as np
import pytest

import geauxdock_amd as g
from geauxdock_amd import abi
from geauxdock_amd.host import ReplicaOut

pytestmark = pytest.mark.gpu

FIELDS = ("energy", "movematrix", "idx_tmp", "n_accept", "n_exchange", "best_energy", "is_accept", "n_swap_lig",
          "n_swap_prt")


def _batch(devs, mcs, outs):
    arr = (C.c_void_p * len(devs))(*[d.h for d in devs])
    oc = (abi.gd_replica_out * len(devs))(*[o.c for o in outs])
    g.check(g.lib().gd_batch_dock(arr, len(devs), (abi.gd_mc_param * len(devs))(*mcs), oc, None), "gd_batch_dock")


# one replica, a block less one, whole blocks, one more
@pytest.mark.parametrize("nl,np_,nt", [(1, 1, 1), (7, 9, 1), (8, 2, 4), (13, 5, 1), (16, 2, 4)])
def test_start_state(ene, nl, np_, nt):
    """No step: every replica at the zero pose and its own temperature, the
    energies those of the evaluation at that pose."""
    job = g.synth_complex(150, 7, nl, np_, nt, seed=nl, ene=ene)
    dev = g.DeviceJob(job)
    n = nl * np_ * nt
    for _ in range(2):  # a used state starts over
        out, _ = dev.dock(g.make_mc(0))
        r = np.arange(n)
        lig, t, p = r % nl, r // nl % nt, r // (nl * nt)
        assert np.array_equal(out.idx_tmp, t)
        assert not out.movematrix.any() and not out.n_exchange.any() and not out.n_swap_lig.any()
        terms, _, _ = dev.eval(np.stack([lig, p], 1).astype(np.int32), np.zeros((n, 6), np.float32))
        assert np.array_equal(out.energy, terms)
        dev.dock(g.make_mc(6, steps_per_exchange=2, seed=1, axes=("temp", "lig", "prt")))
    dev.close()


def test_results_of_long_lists(ene):
    """41 jobs, more than one launch gathers, each as in a batch of its own;
    an array that is not asked for is left out."""
    jobs = [g.synth_complex(100 + k, 4 + k % 5, 1 + k % 4, 2, 3, seed=k, ene=ene) for k in range(41)]
    devs = [g.DeviceJob(j) for j in jobs]
    mcs = [g.make_mc(8, steps_per_exchange=3, seed=2, job_id=k, axes=("temp", "lig")) for k in range(41)]
    outs = [ReplicaOut(j.n_rep) for j in jobs]
    outs[3].c.energy = None
    _batch(devs, mcs, outs)
    assert not outs[3].energy.any()
    for k in (0, 3, 39, 40):
        one = [ReplicaOut(jobs[k].n_rep)]
        _batch([devs[k]], [mcs[k]], one)
        for f in FIELDS:
            if (k, f) != (3, "energy"):
                assert np.array_equal(getattr(one[0], f), getattr(outs[k], f)), (k, f)
    for d in devs:
        d.close()


def test_large_results(ene):
    """196,608 replicas, whose results (18 MB) are copied row by row: every replica's
    energies are those of the evaluation at its pose, and the ladders hold each
    temperature once."""
    nl, np_, nt = 64, 32, 96
    job = g.synth_complex(16, 2, nl, np_, nt, floor_temp=0.05, ceiling_temp=0.3, seed=6, ene=ene)
    dev = g.DeviceJob(job)
    n = nl * np_ * nt
    out, _ = dev.dock(g.make_mc(3, steps_per_exchange=1, seed=2, axes=("temp", "lig")))
    r = np.arange(n)
    lig, p = r % nl, r // (nl * nt)
    terms, _, _ = dev.eval(np.stack([lig, p], 1).astype(np.int32), out.movematrix)
    assert np.array_equal(out.energy, terms)
    assert (out.best_energy <= out.energy[:, 9]).all()
    assert 0 < out.n_accept.sum() <= 3 * n and set(np.unique(out.is_accept)) <= {0, 1}
    assert out.n_exchange.sum() > 0 and out.n_swap_lig.sum() > 0 and not out.n_swap_prt.any()
    ladders = np.sort(out.idx_tmp.reshape(np_, nt, nl).transpose(0, 2, 1), axis=2)
    assert (ladders == np.arange(nt)).all()
    dev.close()
