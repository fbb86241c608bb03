"""The batched sum's queue with one and with several items taken at a time:
the same bits as one call per spectrum, on both sides of the count where
the line-core pass (256 points an item) begins to take two."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

NSPEC = 12


@pytest.fixture(scope="module")
def E():
    from heliosk import engine
    return engine


# 32 chunks for each of 2048 workgroups: 12 x 10922 items are one short of two
# items a chunk, 12 x 10923 are past it; the last chunk is a partial one
@pytest.mark.parametrize("tiles, tail", [(10922, 0), (10923, 0), (10923, -255)])
def test_queue_chunks_do_not_change_a_bit(E, tiles, tail):
    nx, dnu = 256 * tiles + tail, 0.0078125
    grid = E.make_grid(0.0, nx * dnu, dnu)
    assert grid.nx == nx
    items, out = [], torch.full((NSPEC, nx), -1.0, dtype=torch.float64, device="cuda")
    for k in range(NSPEC):
        rng = np.random.default_rng(k)
        n = 50 + 37 * k
        one = np.ones(n)
        sp = E.sort_lines(rng.uniform(0.0, nx * dnu, n), 10.0 ** rng.uniform(-24, -20, n),
                          100.0 * one, 0.05 * one, 0.5 * one, A=0.0 * one, delta=0.0 * one,
                          iso_mass=(18.0 / 6.0221412927e23,))
        st = E.line_params(sp, 300.0 + 100.0 * k, 0.01 * (k + 1), Q=[1.0], cut_mode=0, cut=25.0)
        items.append((st, grid, 0.0, out[k]))
    E.VoigtBatch(items, mode=E.HK_VOIGT_FP32C).launch()
    for k, (st, g, kmin, _) in enumerate(items):
        assert torch.equal(out[k], E.voigt(st, g, kmin, E.HK_VOIGT_FP32C)), k
