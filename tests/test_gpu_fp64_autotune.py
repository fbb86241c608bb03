"""The tuner on FP64 grids shorter than the form's own width needs: the choice
includes that width (tile_points 0), which no caller can ask for by number, and
the tuned call gives the default's bits."""
import pytest

from helpers import random_lines, species_from

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exact", [False, True])
def test_short_grid_tuned_no_slower_than_its_default(exact):
    import torch
    from heliosk import engine as E
    # 30000 points under 1e5 lines that reach all of them: with tiles of 512
    # points the call takes 1.7 times as long as with the form's own 256
    d = random_lines(100000, seed=3, numin=995.0, numax=1035.0)
    st = E.line_params(species_from(d), 900.0, 0.5, Q=d["iso_Q"], cut_mode=0, cut=40.0)
    grid = E.make_grid(1000.0, 1030.0, 0.001)
    E.lib().hk_voigt_autotune_reset()
    tp, stage, ms = E.autotune(st, grid, E.HK_VOIGT_FP64, exact_pairs=exact)
    assert stage in (256, 512) and len(ms) == 8 and all(v > 0.0 for v in ms.values())
    for t in (512, 1024, 2048, 4096):          # timed once
        assert ms[(t, 256)] == ms[(t, 512)]
    if not exact:
        assert tp == 0
    K = E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64, tile_points=tp, stage_lines=stage, exact_pairs=exact)
    if tp == 0:
        assert torch.equal(K, E.voigt(st, grid, 0.0, E.HK_VOIGT_FP64, exact_pairs=exact))
    again = E.autotune(st, grid, E.HK_VOIGT_FP64, exact_pairs=exact)
    assert again[:2] == (tp, stage) and all(v == 0.0 for v in again[2].values())


def test_long_grid_gets_a_width():
    from heliosk import engine as E
    d = random_lines(2000, seed=4, numin=1000.0, numax=1600.0)
    st = E.line_params(species_from(d), 900.0, 0.5, Q=d["iso_Q"], cut_mode=0, cut=5.0)
    grid = E.make_grid(1000.0, 1600.0, 0.001)
    E.lib().hk_voigt_autotune_reset()
    assert E.autotune(st, grid, E.HK_VOIGT_FP64)[0] in (512, 1024, 2048, 4096)
