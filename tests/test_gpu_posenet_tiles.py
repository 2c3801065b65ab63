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


@pytest.mark.parametrize("n,H,W,cin,cout,ks,parts", [
    (1, 1, 1, 16, 16, 1, 4),        # one pixel, one part
    (129, 1, 1, 24, 40, 1, 4),      # images of one pixel, several to a stage
    (70, 7, 5, 1, 32, 3, 3),        # one channel, images across stages, a short last range
    (3, 61, 67, 1, 32, 3, 40),      # more parts than a workgroup of the sum has wavefronts
    (2, 33, 32, 24, 72, 3, 2),      # partial column and channel tiles, ranges that end in a stage
    (5, 2, 300, 64, 20, 3, 1),      # channels not a multiple of 8
    (700, 2, 1, 16, 136, 1, 17),
])
def test_weight_gradient_edges(gpu, n, H, W, cin, cout, ks, parts):
    """Against 64-bit sums over the pixels; a product is exact in FP32, so a sum of m of
    them is within m 2^-24 of the sum of their magnitudes."""
    import torch
    rng = np.random.default_rng(n + cin + H)
    x, dz = _bf16(rng, n, H, W, cin), _bf16(rng, n, H, W, cout)
    K1 = ks * ks * cin + 1
    g = torch.full((cout, K1), float("nan"), device="cuda")
    part = torch.empty(parts * cout * K1, device="cuda")
    _call("isac_nn_conv_wgrad", x, dz, n, H, W, cin, cout, ks, g, part, part.numel() * 4)
    torch.cuda.synchronize()
    r = ks // 2
    xp = torch.nn.functional.pad(x.double().cpu(), (0, 0, r, r, r, r))
    cols = torch.cat([xp[:, i:i + H, j:j + W] for i in range(ks) for j in range(ks)], -1).reshape(n * H * W, -1)
    cols = torch.cat([cols, torch.ones(n * H * W, 1, dtype=torch.float64)], 1)
    d = dz.double().cpu().reshape(n * H * W, cout)
    want, mag = d.T @ cols, d.abs().T @ cols.abs()
    err = (g.double().cpu() - want).abs()
    assert bool((err <= n * H * W * 2.0 ** -24 * mag + 1e-30).all()), float((err / (mag + 1e-30)).max())


@pytest.mark.parametrize("H,W,cin,cout", [(19, 19, 64, 128), (9, 9, 32, 192), (5, 3, 128, 64), (1, 1, 32, 16),
                                          (38, 37, 32, 32), (2, 65, 128, 128)])
def test_resident_conv_channel_tiles(gpu, H, W, cin, cout):
    """Tiles of 64 output channels and several pixel blocks at a time, bit for bit the
    unbanded kernel's (run at 208 channels, which is no multiple of 64)."""
    import torch
    rng = np.random.default_rng(H + W + cin)
    x, w = _bf16(rng, 3, H, W, cin), _bf16(rng, 208, 9 * cin)
    b = torch.from_numpy(rng.standard_normal(208).astype(np.float32)).cuda()
    got, want = (torch.empty((3, H, W, c), dtype=torch.bfloat16, device="cuda") for c in (cout, 208))
    _call("isac_nn_conv_fwd", x, 3, H, W, cin, w, b, 1, cout, 3, 1, 0, got)
    _call("isac_nn_conv_fwd", x, 3, H, W, cin, w, b, 1, 208, 3, 1, 0, want)
    torch.cuda.synchronize()
    assert torch.equal(got, want[..., :cout].contiguous())
