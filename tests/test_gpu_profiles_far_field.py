"""Profiles through the tile sum's nodes, constants and compact windows against
the oracle where they can go wrong: grids that end inside a tile or a wave,
windows that end everywhere or cover all, sub-Lorentzian breaks and range ends
inside tiles and on grid points.

Tolerance: that of the profiles' other oracle tests, 1e-12 of the largest
value of max(K, 1e-12 max K) -- a plinth's difference of two sums of n values
carries ~n eps of the larger (n < 2000 here)."""
import numpy as np
import pytest

from helpers import random_lines, rel_err, species_from, state_numpy
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [1, 65, 513, 4500])
@pytest.mark.parametrize("cm, cut", [(0, 2.0), (0, 40.0), (2, 60.0)])
@pytest.mark.parametrize("profile, plinth, chi", [
    (1, True, False), (1, False, True), (1, True, True), (2, False, False), (2, True, True),
    (3, False, False), (3, True, False), (3, True, True), (4, False, False), (4, False, True)])
def test_profile_edges_vs_oracle(nx, cm, cut, profile, plinth, chi):
    from heliosk import engine as E
    dnu = 0.01
    span = nx * dnu
    d = random_lines(1200, seed=nx + profile, numin=2000.0 - 20.0, numax=2020.0 + span,
                     gamma=(0.05, 0.2), delta=-0.002)
    st = E.line_params(species_from(d), 500.0, 0.7, Q=d["iso_Q"], cut_mode=cm, cut=cut)
    grid = E.make_grid(2000.0, 2000.0 + span, dnu)
    # breaks of the factor 0.5 and 5 cm^-1 from a line; the range ends on a
    # grid point and between two
    c = [0.5, 5.0, 20.0, 0.09, 0.05, 0.02, 2000.0 + 0.2 * span, 2000.0 + 0.3 * span + 0.25 * dnu] \
        if chi else None
    K = E.profile(st, grid, profile, remove_plinth=plinth, kmin=1e-30, chi=c).cpu().numpy()
    Ko = O.profile_points(state_numpy(st), grid.numin, grid.dnu, grid.nx, profile,
                          remove_plinth=plinth, chi=c, kmin=1e-30)
    Kn = O.profile_points(state_numpy(st), grid.numin, grid.dnu, grid.nx, profile, chi=c,
                          kmin=1e-30) if plinth else Ko
    assert np.max(np.abs(K - Ko) / np.maximum(np.abs(Kn), 1e-12 * np.max(np.abs(Kn)))) <= 1e-12


@pytest.mark.parametrize("mode", [1, 2])
def test_plinth_alone_after_other_forms(mode):
    """FP32C and compat sums keep their own plinth pass: what it takes off is
    the plinth sum of the oracle."""
    from heliosk import engine as E
    d = random_lines(1500, seed=4, numin=1990.0, numax=2030.0)
    st = E.line_params(species_from(d), 900.0, 0.5, Q=d["iso_Q"], cut_mode=0, cut=6.0)
    grid = E.make_grid(2000.0, 2020.0, 0.003)
    K = E.profile(st, grid, 1, voigt_mode=mode).cpu().numpy()
    Kp = E.profile(st, grid, 1, voigt_mode=mode, remove_plinth=True).cpu().numpy()
    ost = state_numpy(st)
    sub = (O.profile_points(ost, grid.numin, grid.dnu, grid.nx, 1)
           - O.profile_points(ost, grid.numin, grid.dnu, grid.nx, 1, remove_plinth=True))
    assert np.max(np.abs((K - Kp) - sub)) <= 1e-12 * np.max(K)
