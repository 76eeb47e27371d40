"""Launch shape of the stepping kernel (CPU only)."""
import ctypes as C

import pytest

import geauxdock_amd as g
from geauxdock_amd import abi


# whole devices and partitions of them
@pytest.mark.parametrize("n_cu", [1, 16, 32, 64, 128, 256])
def test_finishers_leave_room_for_workers(n_cu):
    """The groups that stay for a whole launch are at most a quarter of those the
    device holds, so those of three processes leave room for workers."""
    lib = g.lib()
    for n_jobs in (1, 2, 3, 8, 30, 64, 65, 256):
        for n_rep in (25, 64, 65, 220, 512, 513, 1760, 64 * 64, 64 * 1000):
            for chunks, groups in ((1, 1), (1, 3), (6, 3), (10, 5), (20, 9), (20, 60)):
                f, s = C.c_int(), C.c_int()
                g.check(lib.gd_stepping_shape(n_cu, n_jobs, n_rep, chunks, groups, C.byref(f), C.byref(s)), "shape")
                assert s.value in (n_cu, 2 * n_cu, 3 * n_cu, 4 * n_cu)
                assert 1 <= f.value <= max(1, s.value // 4), (n_jobs, n_rep, chunks, groups, f.value, s.value)


def test_arguments():
    f = C.c_int()
    assert g.lib().gd_stepping_shape(0, 1, 1, 1, 1, C.byref(f), C.byref(f)) == abi.GD_ERR_ARG
    assert g.lib().gd_stepping_shape(1, 1, 1, 1, 1, None, C.byref(f)) == abi.GD_ERR_ARG
    assert g.lib().gd_stepping_shape(256, 1, 1 << 26, 1 << 20, 1, C.byref(f), C.byref(f)) == abi.GD_ERR_SIZE
