"""A refused allocation is reported by the call that made it, and by no later one."""
import pytest

import geauxdock_amd as g

pytestmark = pytest.mark.gpu


# one block (launches), five (the stepping kernel)
@pytest.mark.parametrize("shape", [(300, 9, 3, 2, 1), (700, 21, 13, 5, 4)])
def test_next_call_is_well(ene, shape):
    dev = g.DeviceJob(g.synth_complex(*shape, seed=1, ene=ene))
    mc = g.make_mc(12, seed=2, steps_per_exchange=4)
    want, _ = dev.dock(mc)
    with pytest.raises(g.GDError):
        g.check(g.lib().gd_device_copy(1 << 50, 1, None), "gd_device_copy")
    out, _ = dev.dock(mc)
    assert (out.energy == want.energy).all()
    dev.close()
