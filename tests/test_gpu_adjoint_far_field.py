"""The adjoint's far field against the oracle's gradient where it can go
wrong: grids that end inside a tile, a quarter or a segment; windows that end
everywhere; lists of one line, of one workgroup and a little more, and lists
long enough not to be split; low and high pressure; a gradient with an infinite
entry.

Tolerance: as the adjoint's other oracle tests, 1e-10 of the largest entry
(the far field itself leaves 5e-15 of a line; the identity for w' loses
~eps |z|^2 <= 1e-12 below |z|^2 = 1e4)."""
import numpy as np
import pytest

from helpers import random_lines, species_from
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [1, 65, 257, 1024, 3001])
@pytest.mark.parametrize("n", [1, 257])
@pytest.mark.parametrize("T, P, cm, cut", [(900.0, 0.3, 0, 1.3), (300.0, 1e-4, 0, 0.0),
                                           (1500.0, 30.0, 1, 20.0)])
def test_adjoint_edges_vs_oracle(nx, n, T, P, cm, cut):
    import torch
    from heliosk import engine as E
    dnu = 0.003
    d = random_lines(n, seed=nx + n, numin=999.0, numax=1001.0 + nx * dnu, delta=-0.002,
                     EL=(0.0, 2000.0))
    grid = E.make_grid(1000.0, 1000.0 + nx * dnu, dnu)
    gK = np.random.default_rng(n).uniform(-0.3, 1.0, grid.nx)
    gTP, gS, gv = E.adjoint(species_from(d), T, P, torch.from_numpy(gK).cuda(), grid,
                            Q=d["iso_Q"], cut_mode=cm, cut=cut)
    # (cut 0 is the library's "no cut"; the oracle takes the half width itself)
    oT, oP, oS, ov = O.voigt_grad(d, T, P, cm, cut or 1e30, grid.numin, grid.dnu, grid.nx, gK)
    # the totals are sums over the lines: their scale is the sum of magnitudes
    sS = np.sum(np.abs(oS) * d["S"]) + 1e-300
    assert np.max(np.abs(gS.cpu().numpy() - oS)) <= 1e-10 * np.max(np.abs(oS))
    assert np.max(np.abs(gv.cpu().numpy() - ov)) <= 1e-10 * np.max(np.abs(ov))
    gTP = gTP.cpu().numpy()
    assert abs(gTP[0] - oT) <= 1e-10 * max(abs(oT), sS / T)
    assert abs(gTP[1] - oP) <= 1e-10 * max(abs(oP), sS / P)


def test_adjoint_long_list_vs_sums_of_short_ones():
    """A list long enough that one workgroup takes all tiles of its lines
    (no split) against the same lines in pieces (split)."""
    import torch
    from heliosk import engine as E
    n = 256 * 1281 + 3
    d = random_lines(n, seed=5, numin=1000.0, numax=1400.0, EL=(0.0, 2000.0))
    grid = E.make_grid(1190.0, 1210.0, 0.01)
    gK = torch.from_numpy(np.random.default_rng(1).uniform(0.0, 1.0, grid.nx)).cuda()
    gTP, gS, gv = E.adjoint(species_from(d), 700.0, 0.2, gK, grid, Q=d["iso_Q"], cut_mode=0, cut=3.0)
    tot = torch.zeros(2, dtype=torch.float64, device="cuda")
    for a in range(0, n, 100000):
        p = {k: v[a:a + 100000] if isinstance(v, np.ndarray) and v.shape == d["nu"].shape else v
             for k, v in d.items()}
        t, s, v = E.adjoint(species_from(p), 700.0, 0.2, gK, grid, Q=d["iso_Q"], cut_mode=0, cut=3.0)
        tot += t
        b = a + p["nu"].size
        assert float((gS[a:b] - s).abs().max()) <= 1e-13 * float(gS.abs().max())
        assert float((gv[a:b] - v).abs().max()) <= 1e-13 * float(gv.abs().max())
    assert float(((gTP - tot) / gTP).abs().max()) <= 1e-11


def test_adjoint_non_finite_gradient_entry():
    """An infinite dL/dK reaches the lines whose window holds its point only."""
    import torch
    from heliosk import engine as E
    d = random_lines(300, seed=2, numin=1000.0, numax=1030.0)
    sp = species_from(d)
    grid = E.make_grid(1000.0, 1030.0, 0.003)
    gK = torch.from_numpy(np.random.default_rng(1).uniform(0.0, 1.0, grid.nx)).cuda()
    _, gS0, gv0 = E.adjoint(sp, 900.0, 0.3, gK, grid, Q=d["iso_Q"], cut_mode=0, cut=4.0)
    gK[5000] = float("inf")
    _, gS, gv = E.adjoint(sp, 900.0, 0.3, gK, grid, Q=d["iso_Q"], cut_mode=0, cut=4.0)
    hit = (sp.nu - (1000.0 + 5000 * 0.003)).abs() < 4.0
    assert not torch.isfinite(gS[hit]).any()
    assert torch.isfinite(gS[~hit]).all()
    assert float((gS - gS0)[~hit].abs().max()) <= 1e-13 * float(gS0.abs().max())
    assert float((gv - gv0)[~hit].abs().max()) <= 1e-13 * float(gv0.abs().max())
