"""Energy evaluation in passes of any number of 64-lane blocks: fewer and more
poses than the job has lanes, its own buffers, the workspace and the static
scratch, against evaluating the poses one block at a time: the same bits."""
import ctypes as C

import numpy as np
import pytest

import geauxdock_amd as g
from tests.oracle_ffi import random_poses

pytestmark = pytest.mark.gpu

_fp = C.POINTER(C.c_float)
_ip = C.POINTER(C.c_int)


# one block and several; more poses than lanes; more than a workspace pass; a
# job whose own lanes are the pass; wide ligand chunks; a tiny complex
@pytest.mark.parametrize("P,L,nl,np_,nt,n,lc", [
    (300, 9, 3, 2, 1, 1, 4), (300, 9, 3, 2, 1, 64, 4), (300, 9, 3, 2, 1, 65, 4), (300, 9, 3, 2, 1, 2100, 4),
    (700, 21, 5, 11, 4, 129, 4), (700, 21, 5, 11, 4, 257, 8), (90, 6, 16, 8, 8, 1100, 16), (37, 2, 1, 1, 1, 130, 4)])
def test_passes(ene, P, L, nl, np_, nt, n, lc):
    job = g.synth_complex(P, L, nl, np_, nt, seed=n, ene=ene)
    dev = g.DeviceJob(job)
    dev.set_tiling(lc, 16)
    conf, pose = random_poses(job, n, seed=5, trans=2.0)
    conf, pose = np.ascontiguousarray(conf, np.int32), np.ascontiguousarray(pose, np.float32)
    terms, raw, co = dev.eval(conf, pose, want_coords=True)
    t2, r2 = np.full_like(terms, np.nan), np.full_like(raw, np.nan)
    for _ in range(2):
        g.check(g.lib().gd_energy_eval_noalloc(dev.h, n, conf.ctypes.data_as(_ip), pose.ctypes.data_as(_fp),
                                               t2.ctypes.data_as(_fp), r2.ctypes.data_as(_fp)), "noalloc")
        assert np.array_equal(terms, t2) and np.array_equal(raw, r2)
    for at in list(range(0, n, 64))[:3] + [max(0, n - 3)]:
        t, r, c = dev.eval(conf[at:at + 64], pose[at:at + 64], want_coords=True)
        assert np.array_equal(t, terms[at:at + 64]) and np.array_equal(r, raw[at:at + 64])
        assert np.array_equal(c, co[at:at + 64])
    # the replica state is not touched
    mc = g.make_mc(8, seed=2, steps_per_exchange=3)
    a, _ = dev.dock(mc)
    dev.eval(conf, pose)
    b = dev.replicas()
    assert np.array_equal(a.energy, b.energy) and np.array_equal(a.movematrix, b.movematrix)
    dev.close()
