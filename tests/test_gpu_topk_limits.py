"""The top-k where its number of candidates changes its path."""
import numpy as np
import pytest

from mmo_amd import ff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2047, 2048, 2049, 4095, 4096, 20_000, (1 << 22) + 1])
@pytest.mark.parametrize("equal", [1, 1023, 1024, 1025, 2046])
@pytest.mark.parametrize("k", [1, 100, 513, 2048])
def test_topk_at_candidate_limits(n, equal, k):
    """`equal` keys tied at the lowest energy and another tie above them, so that the candidates of
    the first digit are just within or beyond the number at which the passes end: exactly the
    (energy, index) order, from one sort (up to 2,048 energies), from the candidates, or from the
    ties in index order."""
    import torch
    ctx = _context()
    rng = np.random.default_rng(n + equal)
    e = 1.0 + rng.integers(0, 50, n) * 0.25
    at = rng.permutation(n)
    e[at[:equal]] = -3.0
    e[at[equal:equal + 1500]] = -2.0
    v, i = ctx.topk(torch.tensor(e, device="cuda:0"), k)
    want = np.argsort(e, kind="stable")[:k]
    assert np.array_equal(i.cpu().numpy(), want)
    assert np.array_equal(v.cpu().numpy(), e[want])


_made = []


def _context():
    if not _made:
        _made.append(ff.Context(0))
    return _made[0]
