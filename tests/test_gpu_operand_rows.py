"""16-bit operand rows built from the FP32 spectra (more than 40 rings) at the edges of
their layout: a last step of 8 and of 16 rings, full and partly filled, none, padding
rows of few shifts, rows past the last image, more LDS than a kernel has by default."""
import numpy as np
import pytest

from isac_amd import binding, synth
from oracle import coracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,rel", [("fp16", 2e-3), ("bf16", 2e-2)])
@pytest.mark.parametrize("P,D,R,rng", [
    (17, 96, 41, 1.0),      # 9 of the last 16 rings, 9 shifts on 16 rows, 15 images of padding
    (16, 104, 48, 2.0),     # no last step
    (3, 110, 49, 1.0),      # 1 of the last 8 rings
    (5, 118, 56, 0.0),      # all of the last 8 rings, one shift
    (4, 128, 121, 1.0),     # 32 pieces a slot
])
def test_operand_row_edges(gpu, P, D, R, rng, precision, rel):
    import torch
    ds = synth.make_dataset(P, 5, D, 0.42 * D, 0.5, max(rng, 1.0), True, seed_refs=D, seed_particles=R)
    x, ref = torch.from_numpy(ds.sbj).cuda(), torch.from_numpy(ds.ref).cuda()
    _, d = binding.mref_align_mixed_device(x, ref, R, 1.0, rng, rng, precision)
    want = coracle.mref(ds.sbj, ds.ref, np.zeros((P, 2), np.float32), R, rng, rng, 1.0)["d"]
    # the form's bound on its maxima, of the largest of a particle: a smaller one carries its error
    err = np.abs(d.cpu().numpy() - want) / np.abs(want).max(0, keepdims=True)
    print(precision, P, D, R, float(err.max()))
    assert err.max() <= rel
