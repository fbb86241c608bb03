"""Transmission of bins whose clusters span very little: neighbouring doubles,
a few ulps, zeros next to subnormal values.  With enough bins and m the clusters
take the sum; a midpoint of two such values rounds onto one of them, and the
reciprocal of a subnormal half width overflows.

Tolerance: 1e-13 of each value, as the other transmission tests (cluster nodes
leave 2e-15, sums of < 2e4 positive terms a few roundings)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

REPS = 200                       # copies of a bin: enough workgroups for the clusters


def _both(K, nTr, dTr, kmin=0.0):
    import torch
    from heliosk import engine as E
    n = K.size
    Tr = E.transmission(torch.from_numpy(np.tile(K, REPS)).cuda(), REPS, n, nTr, dTr, kmin=kmin)
    Tr = Tr.cpu().numpy().reshape(REPS, nTr)
    assert np.array_equal(Tr, np.broadcast_to(Tr[:1], Tr.shape))
    return Tr[0], O.transmission(K, 1, n, nTr, dTr, kmin=kmin)[0]


@pytest.mark.parametrize("ulps", [1, 2, 3, 5, 10, 1000])
@pytest.mark.parametrize("base", [1.0, 1e-5, 0.3, 2.0 - 2.0 ** -50])
@pytest.mark.parametrize("shape", ["random", "halves", "one"])
def test_few_ulps(ulps, base, shape):
    """Values a few ulps above a background: random, two equal halves, one value
    apart from all others (the last cluster's only width)."""
    n, rng = 4099, np.random.default_rng(ulps)
    k = {"random": rng.integers(0, ulps + 1, n), "halves": np.where(np.arange(n) < n // 2, 0, ulps),
         "one": np.where(np.arange(n) == n - 1, ulps, 0)}[shape]
    K = np.sort(base + np.spacing(base) * k)
    Tr, To = _both(K, 257, 0.04, kmin=base)
    np.testing.assert_allclose(Tr, To, rtol=1e-13, atol=0.0)


@pytest.mark.parametrize("top", [5e-324, 1e-320, 1e-310, 1e-300, 1e-285])
def test_subnormal_spans(top):
    """Tails that underflow: zeros, subnormals and one cluster of ordinary values."""
    n, rng = 4099, np.random.default_rng(3)
    K = np.where(rng.uniform(0, 1, n) < 0.3, 0.0, rng.uniform(0.0, 1.0, n) * top)
    K[: n // 8] = 10 ** rng.uniform(-3, 1, n // 8)
    Tr, To = _both(np.sort(K), 257, 0.04)
    np.testing.assert_allclose(Tr, To, rtol=1e-13, atol=0.0)
