"""Transmission of bins the clusters of the kernel treat differently: fewer
points than a cluster or a batch of clusters holds, remainders, equal values,
flat and wide bins, unsorted and infinite values.

Tolerance: 1e-13 of each value, as the other transmission tests (cluster nodes
leave 2e-15, sums of < 2e4 positive terms a few roundings)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nxb", [3, 127, 129, 2048, 2049, 10007])
@pytest.mark.parametrize("kind", ["wide", "flat", "steps", "unsorted"])
@pytest.mark.parametrize("nTr, reps", [(5, 1), (257, 1), (257, 67)])
def test_transmission_vs_oracle(Nxb, kind, nTr, reps):
    # three bins, or 67 copies of them: with enough bins of 2048 points or more
    # and enough m the clusters take over from the value-by-value kernel
    import torch
    from heliosk import engine as E
    rng = np.random.default_rng(Nxb)
    nbins = 3
    K = 10 ** rng.uniform(-7, 5, (nbins, Nxb))
    if kind == "flat":
        K = 2.0 + 1e-3 * rng.uniform(0, 1, (nbins, Nxb))
    elif kind == "steps":
        K = np.round(np.log10(K)) + 8.0
        K[:, : Nxb // 3] = 0.0
    if kind != "unsorted":
        K = np.sort(K, axis=1)
    nxmin = rng.integers(0, Nxb + 1, nbins).astype(np.int32)
    dTr = 0.1 if nTr > 100 else 4.0
    Tr = E.transmission(torch.from_numpy(np.tile(K, (reps, 1)).ravel()).cuda(), nbins * reps, Nxb,
                        nTr, dTr, kmin=1e-5, nxmin=np.tile(nxmin, reps)).cpu().numpy()
    Tr = Tr.reshape(reps, nbins, nTr)
    assert np.array_equal(Tr, np.broadcast_to(Tr[:1], Tr.shape))
    Tr = Tr[0]
    To = O.transmission(K.ravel(), nbins, Nxb, nTr, dTr, kmin=1e-5, nxmin=nxmin)
    np.testing.assert_allclose(Tr, To, rtol=1e-13, atol=1e-300)


@pytest.mark.parametrize("nbins", [1, 200])
def test_transmission_infinite_value(nbins):
    """exp(-inf) adds nothing: the other values of its cluster still count."""
    import torch
    from heliosk import engine as E
    n, nTr = 4096, 257
    K = np.sort(10 ** np.random.default_rng(1).uniform(-3, 1, n))
    K[-5:] = np.inf
    Tr = E.transmission(torch.from_numpy(np.tile(K, nbins)).cuda(), nbins, n, nTr, 0.05)
    Tr = Tr.cpu().numpy()[nbins - 1]
    m = np.exp((np.arange(nTr) - nTr // 2) * 0.05)
    e = np.exp(-K[None, :] * m[:, None])
    w = np.ones(n)
    w[:3] += (-5 / 8, 1 / 6, -1 / 24)
    w[-3:] += (-5 / 8, 1 / 6, -1 / 24)
    np.testing.assert_allclose(Tr, e @ w / (n - 1.0), rtol=1e-12)


@pytest.mark.parametrize("nbins", [2, 200])
def test_transmission_undefined_value(nbins):
    """An undefined K makes its bin's transmission undefined, no other's."""
    import torch
    from heliosk import engine as E
    n = 4096
    K = np.sort(10 ** np.random.default_rng(2).uniform(-3, 1, (nbins, n)), axis=1)
    K[1, 300] = np.nan
    Tr = E.transmission(torch.from_numpy(K.ravel()).cuda(), nbins, n, 257, 0.05).cpu().numpy()
    assert np.all(np.isnan(Tr[1]))
    assert np.all(np.isfinite(np.delete(Tr, 1, axis=0)))
