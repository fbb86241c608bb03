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
@pytest.mark.parametrize("nTr", [5, 257])
def test_transmission_vs_oracle(Nxb, kind, nTr):
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
    Tr = E.transmission(torch.from_numpy(K.ravel()).cuda(), nbins, Nxb, nTr, dTr, kmin=1e-5,
                        nxmin=nxmin).cpu().numpy()
    To = O.transmission(K.ravel(), nbins, Nxb, nTr, dTr, kmin=1e-5, nxmin=nxmin)
    np.testing.assert_allclose(Tr, To, rtol=1e-13, atol=1e-300)


def test_transmission_infinite_value():
    """exp(-inf) adds nothing: the other values of its cluster still count."""
    import torch
    from heliosk import engine as E
    K = np.sort(10 ** np.random.default_rng(1).uniform(-3, 1, 1000))
    K[-5:] = np.inf
    Tr = E.transmission(torch.from_numpy(K).cuda(), 1, 1000, 64, 0.2).cpu().numpy()[0]
    m = np.exp((np.arange(64) - 32) * 0.2)
    e = np.exp(-K[None, :] * m[:, None])
    w = np.ones(1000)
    w[:3] += (-5 / 8, 1 / 6, -1 / 24)
    w[-3:] += (-5 / 8, 1 / 6, -1 / 24)
    np.testing.assert_allclose(Tr, e @ w / 999.0, rtol=1e-12)


def test_transmission_undefined_value():
    """An undefined K makes its bin's transmission undefined, no other's."""
    import torch
    from heliosk import engine as E
    K = np.sort(10 ** np.random.default_rng(2).uniform(-3, 1, (2, 700)), axis=1)
    K[1, 300] = np.nan
    Tr = E.transmission(torch.from_numpy(K.ravel()).cuda(), 2, 700, 64, 0.2).cpu().numpy()
    assert np.all(np.isfinite(Tr[0])) and np.all(np.isnan(Tr[1]))
