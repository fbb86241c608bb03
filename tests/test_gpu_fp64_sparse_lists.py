"""Sparse lists (at most two lines per 512 points) have kernels of their own, whose
tiles of up to 32 lines are summed point by point: against the oracle with 0, 1, 31,
32, 33, 64 and more lines in reach of a tile, on the shortest grid that takes them,
the last tile short, for every profile, with plinths and sub-Lorentzian wings, and
in batches.

Tolerance: that of the FP64 form's and the profiles' other oracle tests, 1e-11 and
1e-12 of the sum without plinths."""
import numpy as np
import pytest

from helpers import random_lines, rel_err, species_from, state_numpy
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NX = 511 * 512 + 77              # 512 tiles of 512 points
DNU = 0.01


def _lines(kind):
    span = NX * DNU
    if kind == "spread":
        return random_lines(1000, seed=1, numin=2000.0, numax=2000.0 + span, delta=-0.002)
    if kind == "few":
        return random_lines(3, seed=2, numin=2000.0, numax=2000.0 + span)
    # groups of 1, 31, 32, 33, 64 and 200 lines, each inside one tile's 5 cm^-1
    d = random_lines(361, seed=3, numin=0.0, numax=1.0)
    sizes, at = (1, 31, 32, 33, 64, 200), 0
    rng = np.random.default_rng(4)
    for q, n in enumerate(sizes):
        centre = 2000.0 + 512 * DNU * (40 + 80 * q) + 2.5
        d["nu"][at:at + n] = np.sort(centre + rng.uniform(-1.0, 1.0, n))
        at += n
    return d


@pytest.mark.parametrize("kind", ["spread", "few", "groups"])
@pytest.mark.parametrize("cm, cut, P", [(0, 0.6, 0.3), (0, 40.0, 2.0), (0, 0.0, 0.01),
                                        (1, 50.0, 1.0), (2, 8.0, 1e-4)])
def test_sums_vs_oracle(kind, cm, cut, P):
    import torch
    from heliosk import engine as E
    d = _lines(kind)
    st = E.line_params(species_from(d), 500.0, P, Q=d["iso_Q"], cut_mode=cm, cut=cut)
    grid = E.make_grid(2000.0, 2000.0 + NX * DNU, DNU)
    assert grid.nx == NX and st.nlines <= 1024
    ost = state_numpy(st)
    K = E.voigt(st, grid, 1e-30, E.HK_VOIGT_FP64)
    Ko = O.voigt_points(ost, grid.numin, grid.dnu, grid.nx) + 1e-30
    assert rel_err(K.cpu().numpy(), Ko) <= 1e-11
    # a hand-set width of 512 points is the same kernel, accumulation adds to K
    assert torch.equal(K, E.voigt(st, grid, 1e-30, E.HK_VOIGT_FP64, tile_points=512))
    K2 = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64, K=K.clone(), accumulate=True)
    assert rel_err(K2.cpu().numpy(), 2.0 * Ko - 1e-30) <= 1e-11
    # a batch is sparse or not as a whole: two sparse lists, bit for bit
    B = [torch.empty_like(K) for _ in range(2)]
    E.VoigtBatch([(st, grid, 1e-30, b) for b in B], mode=E.HK_VOIGT_FP64).launch()
    assert torch.equal(B[0], K) and torch.equal(B[1], K)
    # every pair evaluated, in a kernel of its own
    X = E.voigt(st, grid, 1e-30, E.HK_VOIGT_FP64, exact_pairs=True)
    assert rel_err(K.cpu().numpy(), X.cpu().numpy()) <= 1e-13
    c = [0.5, 5.0, 20.0, 0.09, 0.05, 0.02, 2000.0 + 0.2 * NX * DNU,
         2000.0 + 0.55 * NX * DNU + 0.25 * DNU]
    for profile, plinth, chi in ((1, True, None), (1, False, c), (2, False, None), (2, True, None),
                                 (2, True, c), (3, False, None), (3, True, None), (4, False, None)):
        Kp = E.profile(st, grid, profile, remove_plinth=plinth, kmin=1e-30, chi=chi).cpu().numpy()
        args = (ost, grid.numin, grid.dnu, grid.nx, profile)
        Kpo = O.profile_points(*args, remove_plinth=plinth, chi=chi, kmin=1e-30)
        Kn = O.profile_points(*args, chi=chi, kmin=1e-30) if plinth else Kpo
        err = np.abs(Kp - Kpo) / np.maximum(np.abs(Kn), 1e-12 * np.max(np.abs(Kn)))
        assert float(np.max(err)) <= 1e-12, (profile, plinth, chi)


def test_mixed_batch_takes_one_width():
    """A sparse and a dense list in one batch, and an empty list, against the single
    sums."""
    import torch
    from heliosk import engine as E
    grid = E.make_grid(2000.0, 2000.0 + NX * DNU, DNU)
    items, single = [], []
    for n in (500, 5000, 0):
        d = random_lines(max(n, 1), seed=n, numin=2000.0, numax=2000.0 + NX * DNU)
        d["S"] *= n > 0
        st = E.line_params(species_from(d), 500.0, 0.3, Q=d["iso_Q"], cut_mode=0, cut=10.0)
        items.append((st, grid, 1e-30, torch.empty(NX, dtype=torch.float64, device="cuda")))
        single.append(E.voigt(st, grid, 1e-30, E.HK_VOIGT_FP64))
    E.VoigtBatch(items, mode=E.HK_VOIGT_FP64).launch()
    for (_, _, _, K), s in zip(items, single):
        assert rel_err(K.cpu().numpy(), s.cpu().numpy()) <= 1e-13
