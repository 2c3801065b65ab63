"""The FP32 search gives the same bits through every entry, however an entry cuts the
particles into launches: the sums that normalise a row of rings are added in one order.
Images whose variance is a small difference of large sums show any other order: a mean of
1000 over a deviation of 1, and a constant with noise in its last bits."""
import numpy as np
import pytest

from isac_amd import binding

pytestmark = pytest.mark.gpu


def _images(kind, n, D, seed):
    g = np.random.default_rng(seed)
    if kind == "offset":
        return (1000.0 + g.standard_normal((n, D, D))).astype(np.float32)
    level = g.uniform(0.05, 3.0, (n, 1, 1)).astype(np.float32)
    return (level * (1.0 + 2.0 ** -23 * g.integers(0, 2, (n, D, D)))).astype(np.float32)


# the ring pairs of a row group go over 4096 // (images x groups of four shifts) wavefronts,
# at most the pairs and 16; the host entry runs quarters of the particles
@pytest.mark.parametrize("kind", ["offset", "constant"])
@pytest.mark.parametrize("P,N,D,R,rng", [
    (600, 2, 40, 8, 1.0),     # whole: 2 wavefronts, quarters: 4
    (1500, 2, 40, 17, 1.0),   # whole: not split, quarters: 3
    (300, 3, 100, 47, 1.0),   # whole: 4, quarters: 16, three batches of the static scratch: 9
    (90, 2, 128, 61, 4.0),    # whole: 2, quarters: 8, batches of 12 and 6: 16
    (3, 1, 32, 4, 0.0),       # one image a quarter, a reference alone
    (229, 5, 32, 3, 1.0),     # odd counts through the halves of the host's staging
])
def test_entries_give_the_same_bits(gpu, P, N, D, R, rng, kind):
    import torch
    x, r = _images(kind, P, D, P + R), _images("offset", N, D, R)
    acc = np.random.default_rng(D).uniform(-0.4, 0.4, (P, 2)).astype(np.float32)
    xd, rd, ad = (torch.from_numpy(v).cuda() for v in (x, r, acc))
    peak, d = (v.clone() for v in binding.mref_align_device(xd, rd, R, 1.0, rng, rng, acc_xy=ad))

    def same(what, p2, d2):
        torch.cuda.synchronize()
        p2, d2 = (torch.as_tensor(v).cpu() for v in (p2, d2))
        diff = int((d2 != d.cpu()).any(0).sum())
        assert diff == 0, f"{what}: d of {diff} of {P} particles differs"
        assert torch.equal(p2, peak.cpu()), f"{what}: peak_list differs"

    same("host pointers", *binding.multi_ref_align(x, r, R, 1.0, rng, rng, acc_xy=acc))
    p2, d2 = torch.empty_like(peak), torch.empty_like(d)
    binding.mref_align_device_noalloc(xd, rd, R, 1.0, rng, rng, p2, d2, acc_xy=ad)
    same("static scratch", p2, d2)
    sub = [{"sbj": xd, "ref": rd, "ring_num": R, "shift_rng": rng, "acc_xy": ad}]
    same("batched graph", *binding.BatchedMref(sub).run(binding.BATCH_GRAPH)[0])
    one = [binding.mref_align_device(xd[i:i + 1], rd, R, 1.0, rng, rng, acc_xy=ad[i:i + 1]) for i in (0, P // 2)]
    torch.cuda.synchronize()
    for i, (_, d1) in zip((0, P // 2), one):
        assert torch.equal(d1[:, 0], d[:, i]), f"one image: d of particle {i} differs"


@pytest.mark.parametrize("kind", ["offset", "constant"])
@pytest.mark.parametrize("P,D,R", [(700, 40, 9), (350, 96, 44), (490, 128, 61)])
def test_single_routes_give_the_same_bits(gpu, P, D, R, kind):
    """All images in one pass from the pixels, sevenths of them through ring spectra in memory."""
    x, ref = _images(kind, P, D, P + R), _images("offset", 3, D, R)
    cid = np.sort(np.arange(P) % 3).astype(np.int32)
    acc = np.random.default_rng(R).uniform(-0.7, 0.7, (P, 2)).astype(np.float32)
    whole = binding.ref_free_align(x, cid, ref, R, 1.0, 1, acc_xy=acc)
    for a in range(0, P, P // 7):
        e = slice(a, a + P // 7)
        ids, local = np.unique(cid[e], return_inverse=True)
        part = binding.ref_free_align(x[e], local.astype(np.int32), ref[ids], R, 1.0, 1, acc_xy=acc[e])
        for key in ("angle", "shift_x", "shift_y", "mirror"):
            np.testing.assert_array_equal(whole[key][e], part[key], err_msg=key)
