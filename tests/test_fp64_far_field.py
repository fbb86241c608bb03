"""The FP64 form's far field: truncation on the kernel's own constants (CPU),
and the sum against the every-pair form and the oracle where tiles, waves and
windows end (GPU).

Tolerance of the GPU comparisons: truncation <= 6e-15 of each far line; a node
sum, its series and the Clenshaw sum carry ~60 FP64 roundings of terms within
a factor (4.25 / 2.25)^2 of each other: 60 * 1.1e-16 * 3.6 = 2.4e-14.  Both
sums are positive, so the relative difference stays below 1e-13."""
import os
import re

import numpy as np
import pytest

from helpers import random_lines, rel_err, species_from, state_numpy
from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _interp_rel_err(d, n):
    """Pointwise relative error of n-node Chebyshev-Gauss interpolation of
    1/(u - d)^2 over [-1, 1], in extended precision."""
    L = np.longdouble
    pi = L("3.14159265358979323846264338327950288")
    th = pi * (np.arange(n).astype(L) + L(0.5)) / n
    f = lambda u: 1 / (u - L(d)) ** 2  # noqa: E731
    c = [(L(2) if m else L(1)) / n * np.sum(f(np.cos(th)) * np.cos(m * th)) for m in range(n)]
    u = np.cos(np.linspace(0, 1, 2001).astype(L) * pi)
    b1, b2 = np.zeros_like(u), np.zeros_like(u)
    for m in range(n - 1, 0, -1):
        b1, b2 = 2 * u * b1 - b2 + c[m], b1
    return float(np.max(np.abs(u * b1 - b2 + c[0] - f(u)) / f(u)))


def test_fp64_node_truncation():
    src = open(os.path.join(ROOT, "helios-k_amd", "csrc", "hk_voigt64.h")).read()
    n = int(re.search(r"constexpr int kFN64 = (\d+);", src).group(1))
    d = float(re.search(r"constexpr double kFarRatio64 = ([\d.]+);", src).group(1))
    assert np.finfo(np.longdouble).eps < 1e-18
    e = _interp_rel_err(d, n)
    print("n=%d d=%g: %.2e" % (n, d, e))
    assert e <= 6e-15
    assert _interp_rel_err(d, n - 2) > 6e-15 and _interp_rel_err(d - 0.5, n) > 6e-15


@pytest.mark.gpu
@pytest.mark.parametrize("nx", [1, 63, 65, 256, 1000, 1025, 4099])
@pytest.mark.parametrize("tile_points", [0, 512, 4096])
@pytest.mark.parametrize("cm, cut, P", [(0, 0.7, 0.5), (0, 0.0, 2.0), (1, 60.0, 1.0),
                                        (2, 40.0, 1e-6)])
def test_fp64_far_field_vs_every_pair(nx, tile_points, cm, cut, P):
    from heliosk import engine as E
    dnu = 0.002
    span = nx * dnu
    d = random_lines(1500, seed=nx + 7 * cm, numin=1000.0 - 3.0 - span, numax=1003.0 + 2.0 * span,
                     delta=-0.003)
    st = E.line_params(species_from(d), 900.0, P, Q=d["iso_Q"], cut_mode=cm, cut=cut)
    grid = E.make_grid(1000.0, 1000.0 + span, dnu)
    K = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64, tile_points=tile_points).cpu().numpy()
    Kx = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64, tile_points=tile_points,
                 exact_pairs=True).cpu().numpy()
    assert K.shape == (nx,)
    np.testing.assert_array_equal(K == 0.0, Kx == 0.0)
    assert rel_err(K, Kx) <= 1e-13
    Ko = O.voigt_points(state_numpy(st), grid.numin, grid.dnu, grid.nx)
    assert rel_err(K, Ko) <= 1e-11


@pytest.mark.gpu
def test_fp64_non_finite_strength_stays_in_its_window():
    """A line of infinite or undefined strength spoils the points of its own
    window only, as it does pair by pair."""
    import torch
    from heliosk import engine as E
    d = random_lines(300, seed=3, numin=1000.0, numax=1060.0)
    sp = species_from(d)
    grid = E.make_grid(1000.0, 1060.0, 0.002)
    st = E.line_params(sp, 900.0, 0.5, Q=d["iso_Q"], cut_mode=0, cut=8.0)
    K = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64)
    x = grid.numin + grid.dnu * torch.arange(grid.nx, dtype=torch.float64, device="cuda")
    for bad in (float("inf"), float("nan")):
        S = sp.S.clone()
        S[150] = bad
        st2 = E.line_params(sp.with_fields(S=S), 900.0, 0.5, Q=d["iso_Q"], cut_mode=0, cut=8.0)
        K2 = E.voigt(st2, grid, 0.0, E.HK_VOIGT_FP64)
        inside = (x - sp.nu[150]).abs() < 8.0
        assert not torch.isfinite(K2[inside]).any()
        a, b = K2[~inside], K[~inside]
        assert torch.isfinite(a).all() and float(((a - b).abs() / b.clamp(min=1e-40)).max()) <= 1e-13


@pytest.mark.gpu
def test_fp64_batch_takes_one_tile_width():
    """A batch of a short and a long grid (one tile width for both) against
    the single sums (each grid's own), and a batch of short grids bit for bit."""
    import torch
    from heliosk import engine as E
    d = random_lines(400, seed=8, numin=1000.0, numax=1060.0)
    st = E.line_params(species_from(d), 900.0, 0.5, Q=d["iso_Q"], cut_mode=0, cut=5.0)
    grids = [E.make_grid(1001.0, 1004.0, 0.001), E.make_grid(1000.0, 1060.0, 1e-4)]
    assert grids[1].nx > 1024 * 512 > grids[0].nx
    K = [torch.empty(g.nx, dtype=torch.float64, device="cuda") for g in grids]
    E.voigt_batched([(st, g, 0.0, k) for g, k in zip(grids, K)], mode=E.HK_VOIGT_FP64)
    for g, k in zip(grids, K):
        assert rel_err(k.cpu().numpy(), E.voigt(st, g, 0.0, E.HK_VOIGT_FP64).cpu().numpy()) <= 1e-13
    short = torch.empty_like(K[0])
    E.voigt_batched([(st, grids[0], 0.0, short)], mode=E.HK_VOIGT_FP64)
    assert torch.equal(short, E.voigt(st, grids[0], 0.0, E.HK_VOIGT_FP64))
    with pytest.raises(Exception, match="tile_points"):
        E.voigt(st, grids[0], 0.0, E.HK_VOIGT_FP64, tile_points=256)
