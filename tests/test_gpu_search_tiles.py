"""FP32 search kernel at the edges of its tiles against the FP64 oracle: reference
counts around a tile of 8, shift counts and particle counts that leave partial blocks
of 8 rows (several particles in one block, a particle ending inside one), ring counts
around the rings that stay in registers and the unrolled ring groups of 4."""
import numpy as np
import pytest

from isac_amd import binding, synth
from oracle import coracle
from parity import compare_mref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,N,D,R,rng,step", [
    (1, 1, 32, 3, 0.0, 1.0),      # one row, one reference, fewer rings than stay resident
    (13, 9, 32, 4, 0.0, 1.0),     # one shift: eight particles in one block of rows
    (5, 7, 40, 5, 1.0, 1.0),      # 9 shifts
    (18, 8, 40, 7, 1.0, 1.0),     # a full tile, runs of more than one particle
    (300, 17, 48, 8, 1.0, 1.0),   # three tiles, the last with one reference
    (9, 16, 64, 29, 2.0, 0.5),    # 81 shifts of half a pixel
    (3, 3, 128, 62, 4.0, 1.0),
])
def test_search_tile_edges(gpu, P, N, D, R, rng, step):
    ds = synth.make_dataset(P, N, D, 0.4 * D, 0.5, max(rng, 1.0), False, seed_refs=P + N,
                            seed_particles=R, seed_noise=D)
    acc = np.random.default_rng(R).uniform(-0.4, 0.4, (P, 2)).astype(np.float32)
    peak, d = binding.multi_ref_align(ds.sbj, ds.ref, R, step, rng, rng, acc_xy=acc)
    ref = coracle.mref(ds.sbj, ds.ref, acc, R, rng, rng, step)
    print(compare_mref(peak, d, ref, f"{P} x {N}, {D} px, {R} rings"))
