"""Bands of the 3x3 convolution with resident weights at the edges of the rule for their
height, bit for bit the unbanded kernel's: whole images, rows of which the smallest bands
hold one or none, the widest rows that any band holds and the first that none does."""
import numpy as np
import pytest

from test_gpu_posenet_tiles import _bf16, _call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,cin,cout", [
    (13, 13, 64, 64), (14, 14, 64, 16),              # whole images past 31 KB
    (16, 17, 64, 32), (22, 22, 32, 64), (23, 23, 32, 16),   # about 52 KB
    (9, 53, 64, 16), (5, 54, 64, 64), (6, 68, 64, 16),      # two rows in 31, 39 and 52 KB
    (4, 71, 64, 16), (7, 72, 64, 128), (3, 97, 64, 32), (3, 147, 64, 64), (2, 148, 64, 16),
    (3, 130, 32, 64), (5, 131, 32, 16), (4, 200, 32, 128), (3, 266, 32, 64), (2, 268, 32, 16),
])
def test_band_heights(gpu, H, W, cin, cout):
    import torch
    rng = np.random.default_rng(H + W + cin)
    x, w = _bf16(rng, 3, H, W, cin), _bf16(rng, 208, 9 * cin)
    b = torch.from_numpy(rng.standard_normal(208).astype(np.float32)).cuda()
    got, want = (torch.empty((3, H, W, c), dtype=torch.bfloat16, device="cuda") for c in (cout, 208))
    _call("isac_nn_conv_fwd", x, 3, H, W, cin, w, b, 1, cout, 3, 1, 0, got)
    _call("isac_nn_conv_fwd", x, 3, H, W, cin, w, b, 1, 208, 3, 1, 0, want)
    torch.cuda.synchronize()
    assert torch.equal(got, want[..., :cout].contiguous())
