"""Workloads of the alignment library, each a pass through its public entry points.

Kinds of case:
  search      multi-reference search of device images (binding.mref_align_device)
  host        the same search through the reference's host-pointer ABI
  best        16-bit MFMA search with the exact best reference per particle
  narrowed    search around proposals, with its fallbacks
  prealign    the pre-alignment loop (shift steps x iterations) on the device
  reffree     reference-free iterations through the host-pointer ABI
  generation  what follows a search: equal-size assignment, reference update
  network     one training step of the proposal network
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-isac_amd"))
from isac_amd import binding, learned, posenet, synth  # noqa: E402

L = binding.RING_LEN
BOXES = (64, 76, 96, 128)


def rings(D):
    return D // 2 - 3


def listed():
    return [
        # the smallest call: a handful of class averages against a few references
        {"name": "search_24x5_d64", "kind": "search", "P": 24, "N": 5, "D": 64, "R": 29, "rng": 2, "snr": 0.1,
         "integer": True, "acc": True},
        # the small workload of the benchmark: latency still counts
        {"name": "search_1000x8_d64", "kind": "search", "P": 1000, "N": 8, "D": 64, "R": 29, "rng": 2, "snr": 0.1,
         "integer": True, "acc": False},
        # the headline workload: one generation's search on one GPU
        {"name": "search_20000x100_d76", "kind": "search", "P": 20000, "N": 100, "D": 76, "R": 35, "rng": 3,
         "snr": 0.05, "integer": False, "acc": False},
        # the largest box and shift range that a subset has
        {"name": "search_1500x60_d128", "kind": "search", "P": 1500, "N": 60, "D": 128, "R": 60, "rng": 4,
         "snr": 0.1, "integer": False, "acc": True},
        # the reference's drivers: one uneven subset from host images, odd box and counts
        {"name": "host_3001x57_d75", "kind": "host", "P": 3001, "N": 57, "D": 75, "R": 33, "rng": 3, "snr": 0.1,
         "integer": False, "acc": True},
        # callers that need each particle's best reference only
        {"name": "best_fp16_8000x100_d76", "kind": "best", "P": 8000, "N": 100, "D": 76, "R": 35, "rng": 3,
         "snr": 0.05, "integer": False, "acc": False, "precision": "fp16"},
        # the same in bf16 with more rings than the direct operand kernel takes
        {"name": "best_bf16_1201x85_d96", "kind": "best", "P": 1201, "N": 85, "D": 96, "R": 44, "rng": 3,
         "snr": 0.1, "integer": False, "acc": True, "precision": "bf16"},
        # search with proposals, as the learned form runs it
        {"name": "narrowed_10000x100_d76", "kind": "narrowed", "P": 10000, "N": 100, "D": 76, "R": 35, "rng": 3,
         "snr": 0.1, "integer": True, "hit": 0.9, "unsure": 0.1},
        # pre-alignment of a stack to its own average
        {"name": "prealign_5000_d76", "kind": "prealign", "P": 5000, "D": 76, "R": 35, "rng": 3, "iters": 3,
         "snr": 0.2, "center": -1, "cutoff": 0.3, "falloff": 0.1},
        # reference-free alignment inside the classes of one generation
        {"name": "reffree_3000x30_d76", "kind": "reffree", "P": 3000, "N": 30, "D": 76, "R": 35, "rng": 2,
         "iters": 3, "snr": 0.1, "cutoff": 0.3, "falloff": 0.2},
        # from scores to new references, headline sizes
        {"name": "generation_20000x100_d76", "kind": "generation", "P": 20000, "N": 100, "D": 76, "snr": 0.05,
         "cutoff": 0.25, "falloff": 0.2},
        # the proposal network's training step at the learned form's settings
        {"name": "network_256_d76", "kind": "network", "B": learned.TRAIN["batch"], "N": 100, "D": 76, "rng": 3},
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["search", "search", "search", "host", "best", "best", "narrowed", "prealign", "reffree",
                       "generation", "network"])
    if kind == "network":
        return {"kind": kind, "B": rng.randint(32, 512), "N": rng.randint(20, 200), "D": rng.choice((64, 76)),
                "rng": rng.randint(2, 3)}
    D = rng.choice(BOXES + (rng.randint(32, 128), rng.randint(32, 128)))
    R = rings(D) - rng.randint(0, 3)
    shift = rng.randint(1, 4 if D > 100 else 3)
    c = {"kind": kind, "D": D}
    if kind == "generation":
        N = rng.randint(5, 150)
        return c | {"P": _log(rng, max(200, N), 20000), "N": N, "snr": rng.uniform(0.05, 0.2), "cutoff": 0.25,
                    "falloff": 0.2}
    c |= {"R": R, "rng": shift, "snr": rng.uniform(0.05, 0.2)}
    # work per pair relative to the headline's, so that no draw costs more than it
    rel = (2 * shift + 1) ** 2 * R / (49 * 35)
    if kind in ("prealign", "reffree"):
        c |= {"P": _log(rng, 100, max(200, min(6000, int(6000 / rel)))), "iters": rng.randint(2, 4),
              "cutoff": rng.choice((0.0, 0.3)), "falloff": 0.2}
        if kind == "prealign":
            return c | {"center": rng.choice((0, -1))}
        return c | {"N": rng.randint(2, 40)}
    N = rng.randint(2, 200)
    c |= {"N": N, "P": _log(rng, 16, max(32, min(20000, int(1.2e6 / (N * max(rel, 0.2)))))),
          "integer": rng.random() < 0.5}
    if kind == "narrowed":
        return c | {"rng": min(shift, 3), "hit": rng.uniform(0.8, 1.0), "unsure": rng.uniform(0.0, 0.2)}
    c["acc"] = rng.random() < 0.5
    if kind == "best":
        c["precision"] = rng.choice(("fp16", "bf16"))
    return c


def _images(c, seed, n_ref):
    D, r = c["D"], c.get("rng", 3)
    sbj, ref, ds = synth.make_dataset_torch(c["P"], n_ref, D, float(rings(D) - 1), c["snr"], float(r),
                                            bool(c.get("integer", False)), "cuda", seed_refs=seed,
                                            seed_particles=seed + 1, seed_noise=seed + 2)
    return sbj.contiguous(), ref.contiguous(), ds


def _acc(c, seed):
    """Shifts accumulated by earlier iterations (none in the first one)."""
    if not c.get("acc"):
        return None
    return np.random.default_rng(seed + 3).uniform(-1.0, 1.0, (c["P"], 2)).astype(np.float32)


def _score_scale(R):
    """CCF value of a normalised image with itself."""
    return L * L * R * (R + 1) / 2.0


def prepare(case, seed):
    c, k = case, case["kind"]
    s = {"c": c}
    if k == "network":
        g = torch.Generator(device="cuda").manual_seed(seed)
        n_shift = (2 * c["rng"] + 1) ** 2
        net = posenet.PoseNet(c["N"], n_shift, D=c["D"], seed=seed % 1000, **learned.NET)
        x, _, _ = _images({"P": c["B"], "D": c["D"], "rng": c["rng"], "snr": 0.1, "integer": True}, seed, c["N"])
        y = torch.stack([torch.randint(0, m, (c["B"],), generator=g, device="cuda")
                         for m in (c["N"], 144, n_shift)], 1).to(torch.int32).contiguous()
        return s | {"net": net, "x": x, "y": y}
    if k == "prealign":
        x, _, _ = _images(c, seed, 1)
        # the driver subtracts each image's mean first
        return s | {"x": (x - x.mean((1, 2), keepdim=True)).contiguous()}
    if k == "reffree":
        x, ref, ds = _images(c, seed, c["N"])
        cid = np.sort(ds.ref_idx)
        # particles in class order; the first averages are those of the unaligned members
        order = torch.from_numpy(np.argsort(ds.ref_idx, kind="stable")).cuda()
        x = x[order].cpu().numpy()
        cid = np.unique(cid, return_inverse=True)[1].astype(np.int32)
        avg = np.stack([x[cid == i].mean(0) for i in range(int(cid[-1]) + 1)]).astype(np.float32)
        return s | {"x": x, "cid": cid, "avg": avg}
    x, ref, ds = _images(c, seed, c["N"])
    P, N = c["P"], c["N"]
    if k == "generation":
        # scores of particles that resemble their own class and, less, its neighbours
        g = torch.Generator(device="cuda").manual_seed(seed)
        f = torch.randn(N, 6, generator=g, device="cuda")
        cls = torch.from_numpy(ds.ref_idx).cuda()
        sim = torch.exp(-0.2 * torch.cdist(f, f) ** 2)
        q = 0.7 + 0.6 * torch.rand(P, generator=g, device="cuda")
        d = 1e7 * (sim[:, cls] * q + 0.15 * torch.randn(N, P, generator=g, device="cuda") + 0.8)
        peak = torch.empty(N, P, 4, device="cuda")
        peak[..., 0] = 360.0 * torch.rand(N, P, generator=g, device="cuda")
        peak[..., 1:3] = torch.randint(-3, 4, (N, P, 2), generator=g, device="cuda").float()
        peak[..., 3] = torch.randint(0, 2, (N, P), generator=g, device="cuda").float()
        return s | {"x": x, "d": d.contiguous(), "peak": peak.view(N, 4 * P)}
    if k == "narrowed":
        rs = np.random.default_rng(seed + 4)
        ny, K = 2 * c["rng"] + 1, 8
        prop = np.empty((P, K, 4), np.int32)
        for j, m in enumerate((N, 2, 72, ny * ny)):
            prop[..., j] = rs.integers(0, m, (P, K))
        # the network's best triple is mostly the pose that made the particle
        psi = np.mod(360.0 - ds.phi + 180.0 * ds.mirror, 360.0)
        sh = np.clip(np.rint(ds.shift + c["rng"]).astype(int), 0, ny - 1)
        true = np.stack([ds.ref_idx, ds.mirror, np.minimum((psi / 5.0).astype(int), 71), sh[:, 0] * ny + sh[:, 1]], 1)
        hit = rs.random(P) < c["hit"]
        prop[hit, 0] = true[hit]
        near = true[:, None] + np.stack([np.zeros((P, 2)), np.zeros((P, 2)), rs.integers(-2, 3, (P, 2)),
                                         np.zeros((P, 2))], 2).astype(int)
        near[..., 2] %= 72
        prop[hit, 1:3] = near[hit]
        conf = rs.random(P).astype(np.float32)
        return s | {"x": x, "ref": ref, "prop": torch.from_numpy(prop).cuda(), "conf": torch.from_numpy(conf).cuda(),
                    "threshold": 0.2 * _score_scale(c["R"])}
    acc = _acc(c, seed)
    if k == "host":
        return s | {"x": x.cpu().numpy(), "ref": ref.cpu().numpy(), "acc": acc}
    return s | {"x": x, "ref": ref, "acc": None if acc is None else torch.from_numpy(acc).cuda()}


def run(state):
    c, k = state["c"], state["c"]["kind"]
    if k == "search":
        return binding.mref_align_device(state["x"], state["ref"], c["R"], 1.0, float(c["rng"]), float(c["rng"]),
                                         acc_xy=state["acc"])
    if k == "host":
        return binding.multi_ref_align(state["x"], state["ref"], c["R"], 1.0, float(c["rng"]), float(c["rng"]),
                                       acc_xy=state["acc"])
    if k == "best":
        return binding.mref_best_mixed_device(state["x"], state["ref"], c["R"], 1.0, float(c["rng"]),
                                              float(c["rng"]), c["precision"], acc_xy=state["acc"])
    if k == "narrowed":
        return binding.mref_proposal_device(state["x"], state["ref"], c["R"], 1.0, float(c["rng"]), float(c["rng"]),
                                            state["prop"], state["threshold"], level2=True, conf=state["conf"],
                                            conf_min=c["unsure"], fallback_form="fp16")
    if k == "prealign":
        return binding.pre_align_loop_device(state["x"], c["R"], [float(c["rng"]), 1.0], [1.0, 1.0], c["iters"],
                                             center=c["center"], cutoff=c["cutoff"], falloff=c["falloff"])
    if k == "reffree":
        return binding.ref_free_align(state["x"], state["cid"], state["avg"], c["R"], float(c["rng"]), c["iters"],
                                      cutoff_freq=c["cutoff"], falloff=c["falloff"])
    if k == "generation":
        groups = binding.assign_groups_device(state["d"])
        cls = torch.from_numpy(binding.classes_from_assignment(groups.cpu().numpy(), c["N"])).cuda()
        return (groups,) + binding.update_references_device(state["x"], state["peak"], cls, c["N"], c["cutoff"],
                                                            c["falloff"])
    net, t = state["net"], learned.TRAIN
    logits = net.forward(state["x"], train=True)
    loss = net.backward(state["y"], t["sigma_psi"], t["sigma_shift"])
    net.step(t["lr"] / t["warmup"], t["wd"])
    return {"logits": logits, "loss": loss, "gradients": net.gflat, "weights": net.flat}


def _search_work(P, N, D, R, S):
    """Ring FFTs of every image at every shift, the ring contraction of every pair,
    and one complex inverse FFT per (pair, shift) for both mirrors."""
    fft = 2.5 * L * math.log2(L)
    return P * S * R * fft + P * N * S * (8.0 * R * (L // 2 + 1) + 2.0 * fft)


def work(case):
    c, k = case, case["kind"]
    if k == "network":
        h, ch, f = c["D"], (1,) + learned.NET["channels"], 0.0
        for i in range(4):
            f += 2.0 * 9 * ch[i] * ch[i + 1] * h * h
            h = h // 2 if i < 3 else h
        heads = c["N"] + 144 + (2 * c["rng"] + 1) ** 2
        w = h * h * ch[4] * learned.NET["hidden"] + learned.NET["hidden"] * heads
        # forward, input gradient and weight gradient; AdamW reads and writes its state
        return {"bytes": 4.0 * c["B"] * c["D"] ** 2 + 28.0 * w, "flops": 3.0 * c["B"] * (f + 2.0 * w)}
    P, D, S = c["P"], c["D"], (2 * c.get("rng", 0) + 1) ** 2
    img = 4.0 * P * D * D
    if k == "generation":
        return {"bytes": img + 4.0 * P * c["N"] + 20.0 * P + 4.0 * c["N"] * D * D, "flops": 30.0 * P * D * D}
    if k == "prealign":
        n = [S] * c["iters"] + [9] * (c["iters"] - 1)
        return {"bytes": (2 * c["iters"]) * img + 24.0 * P,
                "flops": sum(_search_work(P, 1, D, c["R"], x) for x in n) + 2 * c["iters"] * 30.0 * P * D * D}
    if k == "reffree":
        return {"bytes": c["iters"] * img + 24.0 * P,
                "flops": c["iters"] * (_search_work(P, 1, D, c["R"], S) + 30.0 * P * D * D)}
    N, R = c["N"], c["R"]
    out = 20.0 * P * N if k != "narrowed" else 28.0 * P
    ref = 4.0 * N * D * D
    if k == "narrowed":
        # up to 8 windows of 3 x 3 shifts, and the exhaustive search of the unsure
        return {"bytes": img + ref + 128.0 * P + out,
                "flops": _search_work(P, 8, D, R, min(9, S)) + _search_work(c["unsure"] * P, N, D, R, S)}
    return {"bytes": img + ref + out, "flops": _search_work(P, N, D, R, S)}


# ------------------------------------------------------------------ 64 bits


def _sample(img, x, y):
    """Bilinear samples of img [n, D, D] at x, y [n, m], coordinates clamped per tap."""
    n, D = img.shape[0], img.shape[-1]
    x0, y0 = torch.floor(x), torch.floor(y)
    fx, fy = x - x0, y - y0
    xa, xb = x0.long().clamp(0, D - 1), (x0.long() + 1).clamp(0, D - 1)
    ya, yb = y0.long().clamp(0, D - 1) * D, (y0.long() + 1).clamp(0, D - 1) * D
    flat = img.reshape(n, D * D)
    at = lambda i: torch.gather(flat, 1, i)  # noqa: E731
    return (1 - fy) * ((1 - fx) * at(ya + xa) + fx * at(ya + xb)) + fy * ((1 - fx) * at(yb + xa) + fx * at(yb + xb))


def _spectra(img, centre, R):
    """Normalised ring spectra [n * s, R, 129] of img [n, D, D] about centre [n, s, 2]."""
    n, s = centre.shape[:2]
    t = torch.arange(L, device=img.device, dtype=torch.float64) * (2 * math.pi / L)
    w = torch.arange(1, R + 1, device=img.device, dtype=torch.float64)
    x = centre[..., 0].reshape(n, s, 1, 1) + w.view(-1, 1) * torch.cos(t)
    y = centre[..., 1].reshape(n, s, 1, 1) + w.view(-1, 1) * torch.sin(t)
    v = _sample(img, x.reshape(n, -1), y.reshape(n, -1)).view(n * s, R, L)
    nn = L * R * (R + 1) / 2.0
    mu = (v * w.view(-1, 1)).sum((1, 2)) / nn
    sd = torch.sqrt(torch.abs((v * v * w.view(-1, 1)).sum((1, 2)) / nn - mu * mu))
    return torch.fft.rfft((v - mu.view(-1, 1, 1)) / (sd.view(-1, 1, 1) + 1e-7))


def _best_ccf(x, ref, acc, R, rng):
    """Largest CCF over mirror, shift and psi of every pair, [N, P]."""
    P, D, N = x.shape[0], x.shape[-1], ref.shape[0]
    w = torch.arange(1, R + 1, device=x.device, dtype=torch.float64).view(-1, 1)
    zero = torch.full((N, 1, 2), float(D // 2), dtype=torch.float64, device=x.device)
    G = (_spectra(ref.double(), zero, R) * w).permute(2, 1, 0).contiguous()      # [129, R, N]
    ax = torch.arange(-rng, rng + 1, device=x.device, dtype=torch.float64)
    grid = torch.stack(torch.meshgrid(ax, ax, indexing="ij"), -1).reshape(-1, 2) + D // 2
    S = grid.shape[0]
    out = torch.empty(N, P, dtype=torch.float64, device=x.device)
    step = max(1, int(6e5 / (S * max(N, R))))
    for p in range(0, P, step):
        n = min(step, P - p)
        c = grid[None].expand(n, -1, -1) + (acc[p:p + n, None].double() if acc is not None else 0.0)
        F = _spectra(x[p:p + n].double(), c, R).permute(2, 0, 1).contiguous()    # [129, nS, R]
        top = None
        for a in (F.conj().resolve_conj(), F):   # R conj(S), and the mirror's conj(R S)
            C = torch.matmul(a, G).permute(1, 2, 0)
            m = torch.fft.irfft(C if top is None else C.conj().resolve_conj(), n=L).amax(-1) * L
            top = m if top is None else torch.maximum(top, m)
        out[:, p:p + n] = top.view(n, S, N).amax(1).T
    return out


def _greedy(d, cap):
    """Class of each particle: pairs by falling score fill classes of cap particles."""
    N, P = d.shape
    order = np.argsort(-d.reshape(-1), kind="stable")
    cls, room, left = np.full(P, -1), [cap] * N, N * cap
    for i in order.tolist():
        k, p = divmod(i, P)
        if room[k] and cls[p] < 0:
            cls[p] = k
            room[k] -= 1
            left -= 1
            if not left:
                break
    # leftovers: the class of their highest pair for the first P mod cap, class 0 for the rest
    rest = np.flatnonzero(cls < 0)
    if rest.size:
        cls[rest] = 0
        cls[rest[:P % cap]] = np.unravel_index(np.argmax(d[:, rest]), (N, rest.size))[0]
    return cls


def _updated(x, peak, cls, N, cutoff, falloff):
    """New references, parameters, counts and average shifts of an assignment."""
    P, D = x.shape[0], x.shape[-1]
    k = torch.from_numpy(cls).to(x.device)
    q = peak.view(N, P, 4)[k, torch.arange(P, device=x.device)].double()
    a, sx, sy, m = torch.deg2rad(q[:, 0]), q[:, 1], q[:, 2], q[:, 3] != 0
    ca, sa = torch.cos(a), torch.sin(a)
    px, py = -sx * ca - sy * sa, sx * sa - sy * ca
    count = torch.bincount(k, minlength=N)
    tot = torch.zeros(N, 2, dtype=torch.float64, device=x.device)
    tot.index_add_(0, k, torch.stack([torch.where(m, -px, px), py], 1))
    avg = tot / count.clamp(min=1).view(-1, 1)
    g = torch.arange(D, device=x.device, dtype=torch.float64)
    yy, xx = torch.meshgrid(g, g, indexing="ij")
    c = float(D // 2)
    refs = torch.zeros(N, D, D, dtype=torch.float64, device=x.device)
    for p in range(0, P, 1000):
        e = slice(p, min(P, p + 1000))
        v = lambda t: t[e].view(-1, 1, 1)  # noqa: E731
        ux = torch.where(v(m), D - xx, xx) - c
        uy = yy - c
        X = ux * v(ca) - uy * v(sa) + c + v(sx)
        Y = ux * v(sa) + uy * v(ca) + c + v(sy)
        n = X.shape[0]
        refs.index_add_(0, k[e], _sample(x[e].double(), X.reshape(n, -1), Y.reshape(n, -1)).view(n, D, D))
    refs /= count.clamp(min=1).view(-1, 1, 1)
    kx = torch.arange(D // 2 + 1, device=x.device, dtype=torch.float64)
    ky = torch.fft.fftfreq(D, device=x.device, dtype=torch.float64) * D
    ky = torch.where(2 * ky == -D, -ky, ky)
    f = torch.sqrt((kx[None] / D) ** 2 + (ky[:, None] / D) ** 2)
    cc = math.pi / (2 * falloff * cutoff)
    h = 0.5 * (torch.tanh(cc * (f + cutoff)) - torch.tanh(cc * (f - cutoff)))
    turn = (kx.view(1, 1, -1) * avg[:, 0].view(-1, 1, 1) + ky.view(1, -1, 1) * avg[:, 1].view(-1, 1, 1)) / D
    F = torch.fft.rfft(refs, dim=2)
    F = torch.fft.ifft(torch.fft.fft(F, dim=1) * h * torch.exp(2j * math.pi * turn), dim=1)
    refs = torch.fft.irfft(F, n=D, dim=2)
    par = torch.stack([q[:, 0], px - torch.where(m, -1.0, 1.0) * avg[k, 0], py - avg[k, 1], q[:, 3]], 1)
    return refs, par, avg


def _logits(net, x):
    """The network's forward pass in 64 bits on its own rounded weights."""
    n = x.shape[0]
    v = x.double()
    v = v - v.mean((1, 2), keepdim=True)
    v = (v / torch.sqrt((v * v).mean((1, 2), keepdim=True))).unsqueeze(1)
    W = [net.master(i).double() for i in range(6)]
    for i in range(4):
        cin, cout, _ = net.layers[i]
        w = W[i][:, :9 * cin].view(cout, 3, 3, cin).permute(0, 3, 1, 2)
        v = torch.relu(torch.nn.functional.conv2d(v, w, W[i][:, -1], padding=1))
        if i < 3:
            v = torch.nn.functional.max_pool2d(v, 2)
    v = v.permute(0, 2, 3, 1).reshape(n, -1)
    v = torch.relu(v @ W[4][:, :-1].T + W[4][:, -1])
    return v @ W[5][:, :-1].T + W[5][:, -1]


def exact(case, seed):
    c, k = case, case["kind"]
    if k in ("prealign", "reffree", "narrowed"):
        return None   # a choice among alignments feeds the next step
    s = prepare(case, seed)
    if k == "network":
        return {"logits": _logits(s["net"], s["x"]), "loss": None, "gradients": None, "weights": None}
    if k == "generation":
        cls = _greedy(s["d"].cpu().numpy(), c["P"] // c["N"])
        refs, par, avg = _updated(s["x"], s["peak"], cls, c["N"], c["cutoff"], c["falloff"])
        return [None, refs, par, None, avg]
    dev = "cuda"
    x, ref, acc = (None if v is None else torch.as_tensor(v).to(dev) for v in (s["x"], s["ref"], s["acc"]))
    d = _best_ccf(x, ref, acc, c["R"], c["rng"])
    if k == "best":
        return {"d": d, "best_val": d.amax(0)}
    return [None, d]
