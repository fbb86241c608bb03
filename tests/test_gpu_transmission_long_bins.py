"""Transmission of bins longer than one batch of the kernel's clusters (128 of 128
values): a whole batch, one value more, three batches with a short one, and the
reference's example bins of 60000 points, with enough copies of a bin that the
clusters take the sum.

Tolerances: those of the value-by-value form's tests, 1e-13 of the oracle and
2e-13 of the reference's printed values."""
import os

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _run(K, copies, nTr, dTr, **kw):
    import torch
    from heliosk import engine as E
    nbins, n = K.shape
    # (the kernel's rule: clusters where every value's exponential takes a fifth longer)
    direct = nbins * copies * n * nTr / 1.24e6
    blocks = nbins * copies * ((nTr + 127) // 128)
    assert direct > 1.2 * (60.0 + 0.0055 * n) * max(1.0, blocks / 512.0)
    if "nxmin" in kw:
        kw = dict(kw, nxmin=np.tile(kw["nxmin"], copies))
    Tr = E.transmission(torch.from_numpy(np.tile(K, (copies, 1)).ravel()).cuda(), nbins * copies, n,
                        nTr, dTr, **kw).cpu().numpy().reshape(copies, nbins, nTr)
    assert np.array_equal(Tr, np.broadcast_to(Tr[:1], Tr.shape))
    return Tr[0]


@pytest.mark.parametrize("Nxb", [16383, 16384, 16385, 16385 + 127, 32769, 40001])
@pytest.mark.parametrize("kind", ["wide", "steps", "unsorted", "infinite"])
def test_batches_of_clusters_vs_oracle(Nxb, kind):
    rng = np.random.default_rng(Nxb)
    K = 10 ** rng.uniform(-7, 5, (2, Nxb))
    if kind == "steps":
        K = np.round(np.log10(K)) + 8.0
        K[:, : Nxb // 3] = 0.0
    elif kind == "infinite":
        K[:, ::5000] = np.inf
    if kind != "unsorted":
        K.sort(axis=1)
    nxmin = np.array([0, Nxb // 2], dtype=np.int32)
    Tr = _run(K, 64, 257, 0.1, kmin=1e-5, nxmin=nxmin)
    To = O.transmission(K.ravel(), 2, Nxb, 257, 0.1, kmin=1e-5, nxmin=nxmin)
    np.testing.assert_allclose(Tr, To, rtol=1e-13, atol=1e-300)


@pytest.mark.parametrize("b", [0, 4])
def test_reference_bins_through_clusters(golden_dir, b):
    Ks = np.load(os.path.join(golden_dir, "p006_bin%d.npz" % b))["K"]
    ref = np.load(os.path.join(golden_dir, "p006_tr%d.npy" % b))
    Tr = _run(Ks[None, :], 16, 1000, 0.05)[0]
    np.testing.assert_allclose(Tr, O.transmission(Ks, 1, Ks.size, 1000, 0.05)[0], rtol=2e-13, atol=0)
    np.testing.assert_allclose(Tr, ref[:, 1], rtol=2e-13, atol=0)
