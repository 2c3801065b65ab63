"""Ring spectra at the edges of their launch shapes, through searches against the FP64
oracle: ring pairs split over wavefronts and not, rows that leave part of a group of
four, one ring, odd ring counts, all of a reference's ring pairs in one workgroup."""
import numpy as np
import pytest

from isac_amd import binding, synth
from oracle import coracle
from parity import compare_mref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,N,D,R,rng", [
    (2, 3, 32, 1, 0.0),       # half a ring pair, one row of a group
    (3, 2, 40, 9, 1.0),       # five pairs over five wavefronts, 9 rows in three groups
    (40, 2, 48, 17, 3.0),     # nine pairs over seven wavefronts
    (600, 2, 40, 8, 1.0),     # pairs split in two
    (2100, 1, 36, 7, 0.0),    # not split, one row per wavefront
    (100, 2, 120, 5, 4.0),    # not split, 21 groups, one workgroup per CU
    (5, 1, 128, 63, 0.0),     # 32 pairs over 16 wavefronts
])
def test_polar_row_edges(gpu, P, N, D, R, rng):
    ds = synth.make_dataset(P, N, D, 0.4 * D, 0.5, max(rng, 1.0), False, seed_refs=P + N,
                            seed_particles=R, seed_noise=D)
    acc = np.random.default_rng(R).uniform(-0.4, 0.4, (P, 2)).astype(np.float32)
    peak, d = binding.multi_ref_align(ds.sbj, ds.ref, R, 1.0, rng, rng, acc_xy=acc)
    ref = coracle.mref(ds.sbj, ds.ref, acc, R, rng, rng, 1.0)
    print(compare_mref(peak, d, ref, f"{P} x {N}, {D} px, {R} rings"))
