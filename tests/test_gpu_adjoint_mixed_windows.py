"""The adjoint of short lists whose windows differ: a few long ones among short
ones, on both sides of the bound on the longest window of a list that is taken a
line at a time.

Tolerance: as the adjoint's other oracle tests, 1e-10 of the largest entry."""
import numpy as np
import pytest

from helpers import random_lines, species_from
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# 40011 points: 157 tiles of 256 points in 32 parts are 5 rounds, so the longest window
# may have 0.5 * 5 * 40 + 200 = 300 steps of 64 points, 19200 points
@pytest.mark.parametrize("long_points", [200, 18000, 21000, 60000])
@pytest.mark.parametrize("n", [63, 64, 130, 700])
@pytest.mark.parametrize("every", [1, 16, 64])
def test_mixed_windows_vs_oracle(n, long_points, every):
    import torch
    from heliosk import engine as E
    nx, dnu, T, P, cut = 40011, 0.003, 700.0, 0.3, 200.0
    numax = 2000.0 + nx * dnu
    d = random_lines(n, seed=n + every, numin=1999.0, numax=numax + 1.0, EL=(0.0, 2000.0))
    points = np.full(n, 30.0)
    points[::every] = long_points
    d["vy"] = points * dnu / 2 / cut / P         # the half width is cut times this at 296 K
    d["n"] = np.zeros(n)
    grid = E.make_grid(2000.0, numax, dnu)
    gK = np.random.default_rng(n).uniform(-0.3, 1.0, grid.nx)
    gTP, gS, gv = E.adjoint(species_from(d), T, P, torch.from_numpy(gK).cuda(), grid,
                            Q=d["iso_Q"], cut_mode=1, cut=cut)
    oT, oP, oS, ov = O.voigt_grad(d, T, P, 1, cut, grid.numin, grid.dnu, grid.nx, gK)
    sS = np.sum(np.abs(oS) * d["S"]) + 1e-300
    assert np.max(np.abs(gS.cpu().numpy() - oS)) <= 1e-10 * np.max(np.abs(oS))
    assert np.max(np.abs(gv.cpu().numpy() - ov)) <= 1e-10 * np.max(np.abs(ov))
    gTP = gTP.cpu().numpy()
    assert abs(gTP[0] - oT) <= 1e-10 * max(abs(oT), sS / T)
    assert abs(gTP[1] - oP) <= 1e-10 * max(abs(oP), sS / P)
