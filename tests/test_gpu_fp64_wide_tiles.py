"""The FP64 form on a grid long enough for every tile width it has (600001
points: 293 tiles of 2048, the last of them short), far lines through nodes and
every pair evaluated, against the oracle and each other, one spectrum and a batch.

Tolerance: that of the FP64 form's other tests, 1e-11 of the oracle and 1e-13
between the ways of adding the same positive terms up."""
import numpy as np
import pytest

from helpers import random_lines, rel_err, species_from, state_numpy
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NX = 600001


# whole waves in the series (x^2 + y^2 >= 1e6), the 4- and the 8-node rule, cores,
# windows that end everywhere
@pytest.mark.parametrize("dnu, cut, P", [(0.0005, 4.0, 1.0), (0.01, 30.0, 0.01), (0.02, 300.0, 5.0),
                                         (0.001, 0.0, 1e-5)])
def test_every_tile_width(dnu, cut, P):
    import torch
    from heliosk import engine as E
    span = NX * dnu
    d = random_lines(200, seed=7, numin=2000.0, numax=2000.0 + span)
    st = E.line_params(species_from(d), 600.0, P, Q=d["iso_Q"], cut_mode=0, cut=cut)
    grid = E.make_grid(2000.0, 2000.0 + span, dnu)
    assert grid.nx == NX
    Ko = O.voigt_points(state_numpy(st), grid.numin, grid.dnu, grid.nx)
    first = None
    for exact in (True, False):
        for tp in (0, 512, 1024, 2048, 4096):
            K = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64, tile_points=tp, exact_pairs=exact)
            B = torch.full_like(K, -1.0)
            E.VoigtBatch([(st, grid, 0.0, B)], mode=E.HK_VOIGT_FP64, tile_points=tp,
                         exact_pairs=exact).launch()
            assert torch.equal(K, B), (exact, tp)
            Kn = K.cpu().numpy()
            np.testing.assert_array_equal(Kn == 0.0, Ko == 0.0)
            assert rel_err(Kn, Ko) <= 1e-11, (exact, tp)
            first = Kn if first is None else first
            assert rel_err(Kn, first) <= 1e-13, (exact, tp)


def test_whole_wave_series_matches_the_node_rules():
    """Lines whose x^2 + y^2 crosses 1e4 and 1e6 inside a wave, at its ends and
    between two waves: sums of one line alone, point by point against the
    oracle (1e-12: one formula against another near their boundary)."""
    from heliosk import engine as E
    dnu = 0.001
    grid = E.make_grid(2000.0, 2000.0 + NX * dnu, dnu)
    for i in range(12):
        d = random_lines(1, seed=i, numin=2000.0 + 300.0 + 0.17 * i, numax=2300.0 + 0.171 * i + 0.1,
                         gamma=(0.02, 0.05))
        st = E.line_params(species_from(d), 600.0, 10.0 ** (-4 + 0.5 * i), Q=d["iso_Q"], cut_mode=0,
                           cut=0.0)
        Ko = O.voigt_points(state_numpy(st), grid.numin, grid.dnu, grid.nx)
        for tp in (1024, 2048):
            K = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64, tile_points=tp, exact_pairs=True)
            K = K.cpu().numpy()
            far = (np.abs(2000.0 + dnu * np.arange(NX) - d["nu"][0]) > 0.5)
            assert float(np.max(np.abs(K - Ko)[far] / Ko[far])) <= 1e-12, (i, tp)
