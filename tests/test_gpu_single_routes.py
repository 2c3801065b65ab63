"""Alignment of each image to its own reference: in one pass from the pixels where there are
many shifts or images, else with the ring spectra in memory.  The same images in one call
and in small calls give the same records, bit for bit."""
import numpy as np
import pytest

from isac_amd import binding, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,D,R,rng,empty", [
    (350, 32, 1, 1.0, False),     # one ring
    (700, 40, 9, 1.0, True),      # 9 shifts in three groups, odd ring count, some images all 0
    (342, 96, 40, 1.0, False),    # just enough groups
])
def test_single_routes_agree(gpu, P, D, R, rng, empty):
    ds = synth.make_dataset(P, 3, D, max(7.0, 0.4 * D), 0.5, max(rng, 1.0), False, seed_refs=P, seed_particles=R)
    order = np.argsort(ds.ref_idx, kind="stable")
    x, cid = ds.sbj[order], ds.ref_idx[order].astype(np.int32)
    if empty:
        x[::7] = 0.0
    acc = np.random.default_rng(R).uniform(-0.7, 0.7, (P, 2)).astype(np.float32)
    whole = binding.ref_free_align(x, cid, ds.ref, R, rng, 1, acc_xy=acc)
    n = (P + 6) // 7
    for a in range(0, P, n):
        ids, local = np.unique(cid[a:a + n], return_inverse=True)
        part = binding.ref_free_align(x[a:a + n], local.astype(np.int32), ds.ref[ids], R, rng, 1, acc_xy=acc[a:a + n])
        for key in ("angle", "shift_x", "shift_y", "mirror"):
            np.testing.assert_array_equal(whole[key][a:a + n], part[key], err_msg=key)
