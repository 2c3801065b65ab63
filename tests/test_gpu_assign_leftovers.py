"""Group assignment where the particles do not divide evenly into the classes: nearly a
class for each left over, classes of two to nine, scores that resemble a few classes of
each particle (as an alignment's do) and scores in one order for all."""
import numpy as np
import pytest

from isac_amd import binding
from oracle import isac_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P", [(150, 449), (149, 890), (120, 930), (66, 659), (9, 26), (2, 5), (130, 130)])
@pytest.mark.parametrize("kind", ["similar", "one order"])
def test_assign_leftovers(gpu, N, P, kind):
    import torch
    g = np.random.default_rng(N + P)
    if kind == "similar":
        f, own = g.standard_normal((N, 6)), g.integers(0, N, P)
        sim = np.exp(-0.2 * ((f[:, None] - f[None]) ** 2).sum(-1))[:, own]
        d = (sim * (0.7 + 0.6 * g.random(P)) + 0.15 * g.standard_normal((N, P))).astype(np.float32)
    else:
        d = (g.random((N, P)) * 0.3 + g.permutation(N)[:, None]).astype(np.float32)
    got = binding.assign_groups_device(torch.from_numpy(np.ascontiguousarray(d)).cuda()).cpu().numpy()
    np.testing.assert_array_equal(got, O.assign_groups(d))
