"""The FP64 form with every pair evaluated: lines that cover a wave with one
wing formula (all its points at once, tiles of 1024 and 2048 points), with two
formulas, with a core and in part, against tiles of 512 points, which take a
segment at a time, and against the oracle.

Tolerance: the same formulas, added in the same order; a point's sum of at most
1500 positive terms carries one rounding a term either way: 1500 * 1.1e-16 =
1.7e-13."""
import numpy as np
import pytest

from helpers import random_lines, rel_err, species_from, state_numpy
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# spans of a wave in Doppler units from well inside a core to far beyond the
# wings' formulas; the last tile full, one point long and one point short
@pytest.mark.parametrize("nx", [2048, 4097, 8191])
@pytest.mark.parametrize("dnu, cut, P", [(0.0005, 3.0, 1.0), (0.01, 20.0, 0.01), (0.05, 200.0, 5.0),
                                         (0.002, 0.0, 1e-5)])
@pytest.mark.parametrize("tile_points", [1024, 2048])
def test_whole_wave_lines_vs_segments(nx, dnu, cut, P, tile_points):
    from heliosk import engine as E
    span = nx * dnu
    d = random_lines(1500, seed=nx, numin=2000.0 - 0.2 * span, numax=2000.0 + 1.2 * span)
    st = E.line_params(species_from(d), 600.0, P, Q=d["iso_Q"], cut_mode=0, cut=cut)
    grid = E.make_grid(2000.0, 2000.0 + span, dnu)
    K = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64, tile_points=tile_points, exact_pairs=True)
    Ks = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64, tile_points=512, exact_pairs=True)
    K, Ks = K.cpu().numpy(), Ks.cpu().numpy()
    np.testing.assert_array_equal(K == 0.0, Ks == 0.0)
    assert rel_err(K, Ks) <= 1.7e-13
    Ko = O.voigt_points(state_numpy(st), grid.numin, grid.dnu, grid.nx)
    assert rel_err(K, Ko) <= 1e-11
