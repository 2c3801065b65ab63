"""Group assignment where the chains of the last free particles matter: all particles
prefer the same classes (more of them free than one workgroup starts from; more proposals
than it makes in one go), classes of one particle, long chains, equal scores."""
import numpy as np
import pytest

from isac_amd import binding
from oracle import isac_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P,kind", [
    (12, 3000, "popular"),    # 1750 free after the rounds
    (700, 700, "popular"),    # 245 000 proposals, classes of one
    (700, 700, "normal"),
    (65, 1365, "ties"),       # more classes than lanes, classes of 21
    (3, 4099, "minus infinity"),
])
def test_assign_chain_edges(gpu, N, P, kind):
    import torch
    g = np.random.default_rng(N + P)
    d = g.standard_normal((N, P)).astype(np.float32)
    if kind == "popular":
        d = (0.4 * g.random((N, P)) - np.arange(N)[:, None]).astype(np.float32)
    elif kind == "ties":
        d = g.integers(0, 3, (N, P)).astype(np.float32)
    elif kind == "minus infinity":
        d[g.random((N, P)) < 0.7] = -np.inf
    got = binding.assign_groups_device(torch.from_numpy(d).cuda()).cpu().numpy()
    np.testing.assert_array_equal(got, O.assign_groups(d))
