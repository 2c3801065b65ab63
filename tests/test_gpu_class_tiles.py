"""Reference update at the edges of its tiles: class sizes around the eight members that
are loaded at once and the 64 of a shift sum, image sizes around the 16 x 16 pixel tiles,
particles around a chunk of the member lists."""
import numpy as np
import pytest
import torch

from isac_amd import synth
from test_gpu_update import _check_against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,sizes", [
    (16, (1, 7, 8, 9)),
    (17, (0, 16, 63, 64, 65)),
    (33, (1, 0, 129)),
    (24, (500, 523, 2)),     # 1025 particles
])
def test_class_tile_edges(gpu, D, sizes):
    N, P = len(sizes), sum(sizes)
    ds = synth.make_dataset(P, N, D, max(7.0, 0.4 * D), 0.5, 2.0, False, seed_refs=D, seed_particles=P)
    g = np.random.default_rng(P)
    cls = g.permutation(np.repeat(np.arange(N), sizes)).astype(np.int32)
    peak = np.empty((N, P, 4), np.float32)
    peak[..., 0] = g.uniform(0, 360, (N, P))
    peak[..., 1:3] = g.uniform(-6, 6, (N, P, 2))
    peak[..., 3] = g.integers(0, 2, (N, P))
    _check_against_oracle(torch.from_numpy(ds.sbj).cuda(), torch.from_numpy(peak.reshape(N, 4 * P)).cuda(), cls, N,
                          0.25, 0.2)
