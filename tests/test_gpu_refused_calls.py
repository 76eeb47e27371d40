"""Runs whose HIP calls are refused part of the way: an error or another path, and
the next call as if nothing had been."""
import pytest

from tests import hip_refuse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("after", [1, 3, 5])
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
shim.refuse_launch_after(%d)  # start kernel, stepping kernel, exchange, ...
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
