"""Gradients of the k-coefficients for bins with many equal values, on each
path of the last backward step (bins searched in LDS, by size, and longer
ones), against c = G ln(sorted K) differentiated on the host: with K > kmin
the fit is linear in ln K, dL/dKs = (w G) / Ks, and values equal within a bin
take the mean over their ranks.

Tolerance: G applies ~Nxb products of size max|wG|; the kernel forms u = P1^T w
and sums nC Chebyshev terms per point, each within ~nC eps of the largest; a
tie's mean adds log2(n) roundings.  1e-11 of the largest gradient is three
orders above that."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nxb", [500, 5120, 5121, 10241, 16384, 20000])
@pytest.mark.parametrize("ties", ["none", "pairs", "one value"])
def test_backward_with_equal_values(Nxb, ties):
    import torch
    from heliosk import engine as E
    nbins, nC = 3, 12
    rng = np.random.default_rng(Nxb)
    K = np.exp(rng.uniform(-40.0, -20.0, (nbins, Nxb)))
    if ties == "pairs":
        K[:, 1::2] = K[:, : 2 * (Nxb // 2) : 2]
        K[0, Nxb // 3:Nxb // 3 + 200] = K[0, 0]
    elif ties == "one value":
        K[1] = 3.0e-12
        K[2, ::3] = K[2].min()
    w = rng.uniform(-1.0, 1.0, (nbins, nC))
    grid = E.make_grid(0.0, float(nbins * Nxb), 1.0)
    kt = E.KTable(grid, float(nbins * Nxb), nbins, nC, backward=True)
    Kd = torch.from_numpy(K.reshape(-1)).cuda()
    coeff, nxmin, Ks = kt(Kd, want_sorted=True)
    assert int(nxmin.abs().max()) == 0
    g = kt.backward(Kd, Ks, nxmin, torch.from_numpy(w[None]).cuda()).cpu().numpy()
    P = E.ktable_plan(Nxb, nC)
    x = np.arange(Nxb) * 2.0 / (Nxb - 1.0) - 1.0
    G = P[:, :nC] @ np.polynomial.chebyshev.chebvander(x, nC - 1).T
    G[:, :nC] += P[:, nC:]
    ref = np.empty_like(K)
    for b in range(nbins):
        o = np.argsort(K[b], kind="stable")
        gs = (w[b] @ G) / K[b][o]
        _, inv, cnt = np.unique(K[b][o], return_inverse=True, return_counts=True)
        ref[b, o] = (np.bincount(inv, weights=gs) / cnt)[inv]
    for b in range(nbins):
        d = np.max(np.abs(g.reshape(nbins, Nxb)[b] - ref[b]))
        assert d <= 1e-11 * np.max(np.abs((w[b] @ G)) / K[b].min()), (b, d)
