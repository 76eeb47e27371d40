"""Batches whose jobs take unlike numbers of steps, none among them: every job as
in a batch of its own (the same bits), and the energies of a job without steps
those of the evaluation at the zero pose."""
import ctypes as C

import numpy as np
import pytest

import geauxdock_amd as g
from geauxdock_amd import abi
from geauxdock_amd.host import ReplicaOut

pytestmark = pytest.mark.gpu

FIELDS = ("energy", "movematrix", "idx_tmp", "n_accept", "n_exchange", "best_energy", "is_accept", "n_swap_lig",
          "n_swap_prt")
ONE = (300, 9, 3, 2, 1)        # one 64-replica block
MANY = (700, 21, 13, 5, 4)     # five
BIG = (3000, 40, 10, 11, 4)    # seven


def _batch(devs, mcs, stats=False):
    outs = [ReplicaOut(d.n_rep) for d in devs]
    arr = (C.c_void_p * len(devs))(*[d.h for d in devs])
    oc = (abi.gd_replica_out * len(devs))(*[o.c for o in outs])
    st = abi.gd_stats()
    g.check(g.lib().gd_batch_dock(arr, len(devs), (abi.gd_mc_param * len(devs))(*mcs), oc,
                                  C.byref(st) if stats else None), "gd_batch_dock")
    return outs


# without steps beside jobs with them: two one-block jobs, of which one is left; a
# one-block job left of many blocks; many blocks left; several that stop in turn,
# the first to stop with one step; all without steps
@pytest.mark.parametrize("sizes,steps", [
    ([ONE, ONE], [0, 100]), ([MANY, ONE], [0, 30]), ([MANY, BIG], [0, 12]), ([ONE, BIG, MANY], [12, 0, 0]),
    ([ONE, MANY, ONE, BIG, ONE], [1, 7, 0, 9, 20]), ([MANY, ONE], [0, 0])])
@pytest.mark.parametrize("spe", [0, 4])
def test_lengths(ene, sizes, steps, spe):
    jobs = [g.synth_complex(*s, floor_temp=0.05, ceiling_temp=0.3, seed=k + 1, ene=ene)
            for k, s in enumerate(sizes)]
    devs = [g.DeviceJob(j) for j in jobs]
    mcs = [g.make_mc(n, steps_per_exchange=spe, seed=3, job_id=k, move_mode="gaussian", axes=("temp", "lig", "prt"))
           for k, n in enumerate(steps)]
    runs = [_batch(devs, mcs), _batch(devs, mcs, stats=True)]
    for k, (job, dev) in enumerate(zip(jobs, devs)):
        alone, = _batch([dev], [mcs[k]])
        for outs in runs:
            for f in FIELDS:
                assert np.array_equal(getattr(outs[k], f), getattr(alone, f)), (k, f)
        if steps[k] == 0:
            nl, nt = sizes[k][2], sizes[k][4]
            r = np.arange(job.n_rep)
            conf = np.stack([r % nl, r // (nl * nt)], 1).astype(np.int32)
            terms, _, _ = dev.eval(conf, np.zeros((job.n_rep, 6), np.float32))
            assert np.array_equal(runs[0][k].energy, terms)
            assert np.array_equal(runs[0][k].best_energy, terms[:, 9])
        dev.close()
