"""k-table bins longer than one LDS sort, where the number of runs, of merge
rounds and of padded parts of a bucket changes: the sorted spectrum value for
value (zeros of either sign that a splitter equals are copies of it) and a fit
that is known exactly."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def E():
    from heliosk import engine
    return engine


# 16384 + 1 values: 3 runs; 2, 5, 9 and 16 runs and one value past them; runs of
# 16384 from 131073 on (17 of 8192), merged in pairs from 262145 on
@pytest.mark.parametrize("nxb", [16385, 24577, 40960, 40961, 73729, 131072, 131073, 262144, 262145])
@pytest.mark.parametrize("kind", ["random", "rising", "few", "zeros"])
def test_long_bins_sorted(E, nxb, kind):
    nb, dnu = 2, 0.0009765625
    rng = np.random.default_rng(nxb)
    n = nb * nxb
    if kind == "random":
        K = np.exp(rng.normal(0.0, 4.0, n))
    elif kind == "rising":
        K = np.sort(np.exp(rng.normal(0.0, 4.0, n)))
    elif kind == "few":                       # long runs of equal values
        K = rng.integers(1, 6, n).astype(float)
    else:                                     # zeros of both signs and +inf
        K = rng.choice([0.0, -0.0, 1.0e-30, 2.0, np.inf], n)
    grid = E.make_grid(0.0, n * dnu, dnu)
    if grid.nx != n:
        pytest.skip("grid of %d points" % grid.nx)
    kt = E.KTable(grid, n * dnu, nb, 8)
    coeff, nxmin, Ks = kt(torch.as_tensor(K[None, :], device="cuda"), want_sorted=True)
    Ks = Ks.cpu().numpy().reshape(nb, -1)
    for b in range(nb):
        want = np.sort(K[b * nxb:(b + 1) * nxb], kind="stable")
        got = Ks[b][:nxb]
        assert np.array_equal(got, want)
    assert int(nxmin.reshape(-1)[0]) == int((K[:nxb] <= 0.0).sum())


def test_long_bins_fit_does_not_depend_on_the_run_length(E):
    """A spectrum that repeats: bins of 131072 and of 131073 points (16 runs of
    8192, 9 of 16384) drawn from one distribution have coefficients that agree
    as the points' quantiles do (K(y) = e^y at equidistant y, so the fit is
    exact: coefficients 0, 1 and zeros in ln K)."""
    for nxb in (131072, 131073):
        nb, dnu = 2, 0.0009765625
        y = np.tile(np.arange(nxb) / (nxb - 1.0), nb)
        K = np.exp(np.random.default_rng(1).permuted(y.reshape(nb, nxb), axis=1)).reshape(-1)
        grid = E.make_grid(0.0, nb * nxb * dnu, dnu)
        kt = E.KTable(grid, nb * nxb * dnu, nb, 4)
        coeff, nxmin = kt(torch.as_tensor(K[None, :], device="cuda"))[:2]
        # c_0 T_0 + c_1 T_1 at 2 y - 1: ln K = y = 0.5 + 0.5 (2 y - 1)
        want = np.array([0.5, 0.5, 0.0, 0.0])
        got = coeff.cpu().numpy().reshape(nb, -1)[:, :4]
        assert np.all(np.abs(got - want) <= 1e-11)
