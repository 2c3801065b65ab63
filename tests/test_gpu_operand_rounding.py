"""FP16 operands past 40 rings are products rounded to FP32 first: the approximate maxima of a
search, as that rounding gives them, bit for bit (in one rounding to FP16 six of the 768
differ, and a peak between two nearly equal samples can move)."""
import os

import numpy as np
import pytest

from isac_amd import binding, synth

pytestmark = pytest.mark.gpu


def test_fp16_rows_are_rounded_twice(gpu):
    import torch
    want = np.load(os.path.join(os.path.dirname(__file__), "golden", "golden_fp16_rows.npz"))["d"]
    ds = synth.make_dataset(96, 8, 96, 38.0, 0.1, 1.0, False, seed_refs=3, seed_particles=23)
    _, d = binding.mref_align_mixed_device(torch.from_numpy(ds.sbj).cuda(), torch.from_numpy(ds.ref).cuda(), 43, 1.0,
                                           1.0, 1.0, "fp16")
    np.testing.assert_array_equal(d.cpu().numpy(), want)
