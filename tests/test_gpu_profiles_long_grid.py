"""Profiles on a grid past the 256-point tiles (600001 points, 512-point tiles, the
last of 449), under a list too dense for the sparse kernels: two segments a lane,
plinths in tiles and waves, sub-Lorentzian ranges that end inside tiles and on tile
edges, against the oracle.

Tolerance: that of the profiles' other oracle tests, 1e-12 of the sum without
plinths."""
import numpy as np
import pytest

from helpers import random_lines, species_from, state_numpy
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NX, DNU = 600001, 0.01
X0 = 2000.0


@pytest.mark.parametrize("cm, cut, P", [(0, 2.0, 0.7), (2, 12.0, 0.2), (0, 40.0, 0.02)])
@pytest.mark.parametrize("profile, plinth, chi", [
    (1, True, None), (1, False, "inside"), (1, True, "edges"), (2, False, None), (2, True, "inside"),
    (2, True, None), (3, False, None), (3, True, "edges"), (3, True, None), (4, False, "inside")])
def test_long_grid_vs_oracle(cm, cut, P, profile, plinth, chi):
    from heliosk import engine as E
    d = random_lines(3000, seed=profile, numin=X0 - 10.0, numax=X0 + NX * DNU + 10.0,
                     gamma=(0.05, 0.2), delta=-0.002)
    st = E.line_params(species_from(d), 500.0, P, Q=d["iso_Q"], cut_mode=cm, cut=cut)
    grid = E.make_grid(X0, X0 + NX * DNU, DNU)
    assert grid.nx == NX and st.nlines > 2 * ((NX + 511) // 512)
    ends = {"inside": (X0 + DNU * (512 * 300 + 77) + 0.4 * DNU, X0 + DNU * (512 * 700 + 200)),
            "edges": (X0 + DNU * 512 * 100, X0 + DNU * (512 * 900 - 1))}.get(chi)
    c = [0.5, 5.0, 20.0, 0.09, 0.05, 0.02, *ends] if chi else None
    args = (state_numpy(st), grid.numin, grid.dnu, grid.nx, profile)
    K = E.profile(st, grid, profile, remove_plinth=plinth, kmin=1e-30, chi=c).cpu().numpy()
    Ko = O.profile_points(*args, remove_plinth=plinth, chi=c, kmin=1e-30)
    Kn = O.profile_points(*args, chi=c, kmin=1e-30) if plinth else Ko
    assert np.max(np.abs(K - Ko) / np.maximum(np.abs(Kn), 1e-12 * np.max(np.abs(Kn)))) <= 1e-12


@pytest.mark.parametrize("cut", [1.5, 4.0])
@pytest.mark.parametrize("n", [3000, 1000])
def test_plinth_inside_a_doppler_line(cut, n):
    """A cut of a few Doppler widths: the plinth does not underflow, so a line takes
    part at all points of its window (dense and sparse lists)."""
    from heliosk import engine as E
    dnu = 0.0005
    d = random_lines(n, seed=9, numin=X0, numax=X0 + NX * dnu)
    st = E.line_params(species_from(d), 500.0, 0.1, Q=d["iso_Q"], cut_mode=2, cut=cut)
    grid = E.make_grid(X0, X0 + NX * dnu, dnu)
    args = (state_numpy(st), grid.numin, grid.dnu, grid.nx, 3)
    K = E.profile(st, grid, 3, remove_plinth=True).cpu().numpy()
    Ko = O.profile_points(*args, remove_plinth=True)
    Kn = O.profile_points(*args)
    assert np.max(np.abs(Kn - Ko)) > 1e-8 * np.max(Kn)
    assert np.max(np.abs(K - Ko) / np.maximum(np.abs(Kn), 1e-12 * np.max(np.abs(Kn)))) <= 1e-12
