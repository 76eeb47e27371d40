"""Pair passes of few items (three work groups to an item) against passes of many
(one): the same bits for the same poses, on both sides of the item count where the
library changes over, and energies within 1e-5 of FP64 on the oracle."""
import numpy as np
import pytest

import geauxdock_amd as g
from tests.oracle_ffi import random_poses, rel_err

pytestmark = pytest.mark.gpu


# items of a 64-pose block = ceil(L / 4) * tile groups.  256 items are four blocks of
# 64, so that 256 poses and 257 lie on the two sides for 256 CUs; then a last chunk
# of one atom, tiles with no or few points of a class, tiles of more than 64 points,
# a complex smaller than its tiles
@pytest.mark.parametrize("P,L,tile,n_few,n_many", [
    (2048, 4, 4, 256, 257), (2048, 4, 4, 1, 2048), (1201, 5, 2, 64, 512), (5003, 21, 90, 65, 1024),
    (700, 62, 16, 63, 1500), (19, 3, 4, 1, 64)])
def test_same_bits(ene, oracle, P, L, tile, n_few, n_many):
    job = g.synth_complex(P, L, 5, 3, 2, seed=P + L, ene=ene)
    dev = g.DeviceJob(job)
    dev.set_tiling(4, tile)
    conf, pose = random_poses(job, n_many, seed=7, trans=2.0)
    terms, raw, _ = dev.eval(conf, pose)
    for at in (0, n_many - n_few):
        t, r, coords = dev.eval(conf[at:at + n_few], pose[at:at + n_few], want_coords=True)
        assert np.array_equal(t, terms[at:at + n_few]) and np.array_equal(r, raw[at:at + n_few])
        k = min(n_few, 64)
        _, r_raw, r_scale, _ = oracle.energy(job, conf[at:at + k], pose[at:at + k], mode=2, coords=coords[:k])
        assert rel_err(r[:k], r_raw, r_scale).max() <= 1e-5
    dev.close()
