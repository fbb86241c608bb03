"""The adjoint of short lists on both sides of the rule that takes a line at a
time: windows short against the tiles they spread over, gaps between windows,
windows that end at the grid's ends, lists of one line and of a workgroup and one
line more, and workspaces that leave one part (each wave many lines).

Tolerance: as the adjoint's other oracle tests, 1e-10 of the largest entry."""
import ctypes

import numpy as np
import pytest

from helpers import random_lines, species_from
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# nx 20011: 78 tiles of 256 points in 32 parts are 3 rounds of 40 steps of 64
# points, so a window of up to 7616 points is taken a line at a time, if the
# lines spread over the whole grid
@pytest.mark.parametrize("nx", [20011, 8191])
@pytest.mark.parametrize("n", [1, 65, 257])
@pytest.mark.parametrize("P, cm, cut", [(0.3, 0, 0.004), (0.3, 0, 0.3), (1e-4, 0, 11.4),
                                        (0.3, 0, 11.7), (2.0, 0, 0.0), (0.05, 1, 30.0),
                                        (1e-3, 2, 50.0)])
@pytest.mark.parametrize("one_part", [False, True])
def test_short_windows_vs_oracle(nx, n, P, cm, cut, one_part):
    import torch
    from heliosk import _lib, engine as E
    dnu, T = 0.003, 700.0
    d = random_lines(n, seed=nx + n, numin=1999.0, numax=2001.0 + nx * dnu, delta=-0.002,
                     EL=(0.0, 2000.0))
    grid = E.make_grid(2000.0, 2000.0 + nx * dnu, dnu)
    gK = np.random.default_rng(n).uniform(-0.3, 1.0, grid.nx)
    g = torch.from_numpy(gK).cuda()
    if one_part:
        sp, nb = species_from(d), 16 * n + 272
        lines, tp, c = sp.lines(), E._tp(T, P, d["iso_Q"]), _lib.Cut(cm, cut)
        ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
        gTP, gS, gv = (torch.empty(k, dtype=torch.float64, device="cuda") for k in (2, n, n))
        E.check(E.lib().hk_voigt_adjoint(ctypes.byref(lines), ctypes.byref(tp), ctypes.byref(c),
                                         ctypes.byref(grid), g.data_ptr(), gS.data_ptr(),
                                         gv.data_ptr(), gTP.data_ptr(), ws.data_ptr(), nb, None))
    else:
        gTP, gS, gv = E.adjoint(species_from(d), T, P, g, grid, Q=d["iso_Q"], cut_mode=cm, cut=cut)
    oT, oP, oS, ov = O.voigt_grad(d, T, P, cm, cut or 1e30, grid.numin, grid.dnu, grid.nx, gK)
    sS = np.sum(np.abs(oS) * d["S"]) + 1e-300
    assert np.max(np.abs(gS.cpu().numpy() - oS)) <= 1e-10 * np.max(np.abs(oS))
    assert np.max(np.abs(gv.cpu().numpy() - ov)) <= 1e-10 * np.max(np.abs(ov))
    gTP = gTP.cpu().numpy()
    assert abs(gTP[0] - oT) <= 1e-10 * max(abs(oT), sS / T)
    assert abs(gTP[1] - oP) <= 1e-10 * max(abs(oP), sS / P)


def test_non_finite_gradient_entry_a_line_at_a_time():
    """An infinite dL/dK reaches the lines whose window holds its point only."""
    import torch
    from heliosk import engine as E
    d = random_lines(300, seed=2, numin=1000.0, numax=1090.0)
    sp = species_from(d)
    grid = E.make_grid(1000.0, 1090.0, 0.003)
    gK = torch.from_numpy(np.random.default_rng(1).uniform(0.0, 1.0, grid.nx)).cuda()
    _, gS0, _ = E.adjoint(sp, 900.0, 0.3, gK, grid, Q=d["iso_Q"], cut_mode=0, cut=0.5)
    gK[15000] = float("inf")
    _, gS, _ = E.adjoint(sp, 900.0, 0.3, gK, grid, Q=d["iso_Q"], cut_mode=0, cut=0.5)
    hit = (sp.nu - (1000.0 + 15000 * 0.003)).abs() < 0.5
    assert 0 < int(hit.sum()) < 50
    assert not torch.isfinite(gS[hit]).any()
    assert torch.equal(gS[~hit], gS0[~hit])
