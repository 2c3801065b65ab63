"""FP32 search in the forms that large calls run: ring pairs spread over lanes or not, one or
several workgroups a CU, runs of 2, 4 and 8 particles a workgroup that begin and end inside
a block of 8 rows, a last run that is shorter.  Against one-particle calls, which run
other forms, bit for bit, and a few particles against the FP64 oracle."""
import numpy as np
import pytest

from isac_amd import binding, synth
from oracle import coracle
from parity import compare_mref

pytestmark = pytest.mark.gpu


# ring spectra: form, wavefronts a workgroup (passes); particles a search workgroup
@pytest.mark.parametrize("P,N,D,R,rng", [
    (901, 9, 76, 34, 3.0),      # unspread, 7 (2); 8
    (701, 30, 76, 34, 2.0),     # unspread, 7 (1); 4
    (333, 17, 96, 40, 3.0),     # unspread, 7 (2); 4
    (257, 5, 110, 51, 3.0),     # unspread, 13 (1), one workgroup a CU; 2
    (130, 9, 128, 61, 4.0),     # unspread, 11 (2), one workgroup a CU; 2
    (1501, 5, 40, 17, 1.0),     # spread, 4; 8
    (1501, 2, 128, 61, 1.0),    # spread, 16; 8
    (2101, 1, 36, 7, 0.0),      # spread, 1: four pairs; 8 of one row
    (2101, 9, 100, 46, 0.0),    # spread, 8; 8 of one row
    (600, 2, 128, 60, 2.0),     # spread, 16; 1
    (901, 17, 32, 9, 1.0),      # spread, 4; 4
    (2103, 1, 32, 1, 1.0),      # unspread, one ring, 3 (1); 4
    (515, 9, 50, 3, 2.0),       # unspread, two pairs, 7 (1); 1
    (100, 17, 40, 15, 1.0),     # few images; 2
])
def test_large_calls(gpu, P, N, D, R, rng):
    import torch
    ds = synth.make_dataset(P, N, D, max(7.0, 0.4 * D), 0.5, max(rng, 1.0), False, seed_refs=P + N, seed_particles=R)
    acc = np.random.default_rng(R).uniform(-0.4, 0.4, (P, 2)).astype(np.float32)
    x, r, a = (torch.from_numpy(v).cuda() for v in (ds.sbj, ds.ref, acc))
    peak, d = (v.clone() for v in binding.mref_align_device(x, r, R, 1.0, rng, rng, acc_xy=a))
    peak = peak.view(N, P, 4)
    some = sorted({0, 1, 2, 3, 5, 7, 8, P // 2, P // 2 + 1, P - 9, P - 2, P - 1})
    for p in some:
        e = slice(p, p + 1)
        p1, d1 = binding.mref_align_device(x[e], r, R, 1.0, rng, rng, acc_xy=a[e])
        torch.cuda.synchronize()
        assert torch.equal(d[:, e], d1), f"d of particle {p}"
        assert torch.equal(peak[:, e], p1.view(N, 1, 4)), f"peak_list of particle {p}"
    few = [0, 7, P - 1]
    want = coracle.mref(ds.sbj[few], ds.ref, acc[few], R, rng, rng, 1.0)
    print(compare_mref(peak[:, few].reshape(N, -1).cpu().numpy(), d[:, few].cpu().numpy(), want, f"{P} x {N}, {D} px"))


@pytest.mark.parametrize("D,R,rng,hw", [
    (76, 34, 3.0, 1),     # one window: spread over 8 wavefronts; eight: not spread
    (76, 33, 3.0, 0),     # one row
    (128, 61, 3.0, 1),    # 16 wavefronts and 13
    (40, 17, 1.0, 0),     # 3 and 4
    (64, 29, 2.0, 2),
    (32, 1, 2.0, 1),
])
def test_masked_forms_agree(gpu, D, R, rng, hw):
    """The same proposal once and eight times over: other launch shapes and items, one result."""
    import torch
    P, N, n = 300, 4, 2 * int(rng) + 1
    ds = synth.make_dataset(P, N, D, max(7.0, 0.4 * D), 0.5, rng, False, seed_refs=D, seed_particles=R)
    g = np.random.default_rng(D + hw)
    one = np.stack([g.integers(0, m, (P, 1)) for m in (N, 2, 72, n * n)], 2).astype(np.int32)
    x, r, prop = (torch.from_numpy(v).cuda() for v in (ds.sbj, ds.ref, one))

    def run(q):
        out = binding.mref_proposal_device(x, r, R, 1.0, rng, rng, q.contiguous(), -1e30, shift_half=hw,
                                           edge_fallback=False)
        torch.cuda.synchronize()
        return {k: out[k].clone() for k in ("best_ref", "best_val", "best_peak")}

    a, b = run(prop), run(prop.expand(P, 8, 4))
    far = torch.randint(0, n * n, (P, 7), device="cuda", dtype=torch.int32)   # seven others, with no reference
    others = torch.stack([torch.full_like(far, -1), torch.zeros_like(far), torch.zeros_like(far), far], 2)
    c = run(torch.cat([prop, others], 1))
    for k in a:
        assert torch.equal(a[k], b[k]), k
        assert torch.equal(a[k], c[k]), k
