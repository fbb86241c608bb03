"""The FP32 form's far field through shared wave sums: tiles and waves at whose
edges a band has no line, one line or only lines that cover some of the waves,
against every pair evaluated."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def E():
    from heliosk import engine
    return engine


def _lines(E, nu):
    n = len(nu)
    rng = np.random.default_rng(n)
    S = 10.0 ** rng.uniform(-24, -20, n)
    one = np.ones(n)
    return E.sort_lines(np.asarray(nu, float), S, 100.0 * one, 0.05 * one, 0.5 * one,
                        A=0.0 * one, delta=0.0 * one, iso_mass=(18.0 / 6.0221412927e23,))


# distances in half widths of a 1024-point tile from the middle of the grid's
# first tile: one line per band, lines at the bands' edges, cut windows that
# end inside the tile, a whole wave of lines and one more
@pytest.mark.parametrize("dist", [[6.0], [3.0], [1.7], [1.49, 1.51, 1.99, 2.01, 3.99, 4.01],
                                  list(np.linspace(1.2, 12.0, 64)), list(np.linspace(1.2, 12.0, 65)),
                                  list(np.linspace(-14.0, 14.0, 700))])
@pytest.mark.parametrize("cut", [25.0, 4.0])
@pytest.mark.parametrize("points", [512, 1024, 2048])
def test_shared_totals_against_every_pair(E, dist, cut, points):
    # bound: the bands' interpolation errors (at most 1e-6 of a line at a
    # point) plus FP32 rounding of the pair-by-pair form (a few 1e-7)
    dnu, nx = 0.002, 3 * 1024 + 17
    grid = E.make_grid(1000.0, 1000.0 + nx * dnu, dnu)
    half = 0.5 * points * dnu
    sp = _lines(E, 1000.0 + half + half * np.asarray(dist))
    st = E.line_params(sp, 500.0, 1.0, Q=[1.0], cut_mode=0, cut=cut)
    K = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP32C, tile_points=points)
    X = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP32C, tile_points=points,
                exact_pairs=True)
    torch.cuda.synchronize()
    K, X = K.cpu().numpy(), X.cpu().numpy()
    assert np.array_equal(K == 0.0, X == 0.0)
    m = X > 0.0
    assert np.all(np.abs(K[m] - X[m]) <= 3e-6 * X[m])
