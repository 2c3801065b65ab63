"""Tile edges of the proposal network's kernels where a rule chooses between two of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _call(name, *args):
    import torch
    from isac_amd import posenet
    args = [a.data_ptr() if torch.is_tensor(a) else a for a in args]
    posenet._call(posenet._lib(), name, *args, torch.cuda.current_stream().cuda_stream)


def _bf16(rng, *shape):
    import torch
    return torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).cuda().to(torch.bfloat16)


@pytest.mark.parametrize("n", [1, 16, 63, 130])
@pytest.mark.parametrize("cin,cout,relu,f32", [(16, 16, 0, 1), (176, 48, 1, 0), (192, 16, 1, 1), (400, 304, 0, 0)])
def test_dense_rows_equal_the_large_batch(gpu, n, cin, cout, relu, f32):
    """Few rows run in 16 x 16 tiles, many (33 * 256 here) in 64 x 64 ones, bit for bit alike."""
    import torch
    rng = np.random.default_rng(n + cin)
    big = 33 * 256
    x, w = _bf16(rng, big, cin), _bf16(rng, cout, cin)
    b = torch.from_numpy(rng.standard_normal(cout).astype(np.float32)).cuda()
    dt = torch.float32 if f32 else torch.bfloat16
    want, got = (torch.empty((m, cout), dtype=dt, device="cuda") for m in (big, n))
    _call("isac_nn_conv_fwd", x, big, 1, 1, cin, w, b, 1, cout, 1, relu, f32, want)
    _call("isac_nn_conv_fwd", x, n, 1, 1, cin, w, b, 1, cout, 1, relu, f32, got)
    torch.cuda.synchronize()
    assert torch.equal(got, want[:n])
    ref = x[:n].double() @ w.double().T + b.double()
    ref = (ref.clamp_min(0.0) if relu else ref).cpu().numpy()
    # sums of cin products in FP32, and the output's rounding
    np.testing.assert_allclose(got.double().cpu().numpy(), ref, rtol=2.0 ** -23 if f32 else 2.0 ** -8,
                               atol=cin * 2.0 ** -22)
