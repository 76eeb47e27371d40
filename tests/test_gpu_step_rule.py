"""Plain runs on both sides of the item counts where stepping changes over from
launches on one stream to the stepping kernel: the same bits as launches, as the
default steps them, with a wait bound that ends every stepping launch at once (the
run is repeated by launches), and again on the same job."""
import numpy as np
import pytest

import geauxdock_amd as g

pytestmark = pytest.mark.gpu

FIELDS = ("energy", "movematrix", "idx_tmp", "n_accept", "n_exchange", "best_energy", "is_accept", "n_swap_lig",
          "n_swap_prt")


# (points, atoms, conformers, conformers, temperatures, tile points): two blocks of
# about 560 items and 640 and of 2,240; four of 128 and 132; six of 42 and 44; one-chunk and
# two-atom ligands with many tiles; a last chunk of one atom
@pytest.mark.parametrize("P,L,nl,np_,nt,tile", [
    (1120, 80, 13, 5, 1, 5), (8960, 80, 13, 5, 1, 10), (1280, 80, 13, 5, 1, 5), (1024, 32, 5, 11, 4, 8), (1056, 32, 5, 11, 4, 8),
    (1344, 8, 13, 5, 5, 8), (1408, 8, 13, 5, 5, 8), (900, 4, 10, 11, 4, 2), (500, 2, 13, 5, 5, 1),
    (800, 21, 13, 5, 5, 4)])
def test_same_bits(ene, P, L, nl, np_, nt, tile):
    job = g.synth_complex(P, L, nl, np_, nt, floor_temp=0.05, ceiling_temp=0.3, seed=P + L, ene=ene)
    dev = g.DeviceJob(job)
    dev.set_tiling(4, tile)
    mc = g.make_mc(11, steps_per_dump=6, steps_per_exchange=4, seed=3, axes=("temp", "lig", "prt"), record=True,
                   move_mode="gaussian")
    runs = []
    for wait in (2.0, 0.0, 2.0):
        dev.set_step_wait(wait)
        runs.append((dev.dock(mc)[0], dev.records(6)))
    dev.set_streams(1)
    want, (rec, cnt) = dev.dock(mc)[0], dev.records(6)
    for out, (r, c) in runs:
        for f in FIELDS:
            assert np.array_equal(getattr(out, f), getattr(want, f)), f
        assert np.array_equal(c, cnt)
        keep = np.arange(rec.shape[1])[None, :] < cnt[:, None]
        assert np.array_equal(r[keep], rec[keep])
    dev.close()
