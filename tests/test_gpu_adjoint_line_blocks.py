"""The adjoint's ways of sharing lines and points out (64 lines and tiles of 256
or 512 points, 256 lines and 1024 points) at the list lengths where one gives way
to another: the gradient of a line does not depend on the other lines of its
list, so a list of 65536 lines (256) and its halves (64), or one of 3000 (512
points) and its halves (256), give the same entries.

Tolerance: a line's four sums are added in other groups; each carries < 100
roundings of terms whose magnitudes add up to at most ~1e3 times the sum on this
gK > 0: 100 * 1e3 * 1.1e-16 = 1e-11 of the largest entry."""
import numpy as np
import pytest

from helpers import random_lines, species_from

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2999, 3000, 3001, 65535, 65536, 65537])
@pytest.mark.parametrize("nx, cut", [(1025, 2.0), (3000, 0.4)])
def test_whole_list_vs_its_halves(n, nx, cut):
    import torch
    from heliosk import engine as E
    dnu = 0.004
    d = random_lines(n, seed=3, numin=1000.0, numax=1000.0 + nx * dnu)
    grid = E.make_grid(1000.0, 1000.0 + nx * dnu, dnu)
    gK = torch.from_numpy(np.random.default_rng(1).uniform(0.5, 1.0, grid.nx)).cuda()

    def run(part):
        e = {k: v[part] if isinstance(v, np.ndarray) and v.shape[:1] == (n,) else v
             for k, v in d.items()}
        g = E.adjoint(species_from(e), 700.0, 0.1, gK, grid, Q=d["iso_Q"], cut_mode=0, cut=cut)
        return [x.cpu().numpy() for x in g]

    h = n // 2
    tp, gS, gv = run(slice(0, n))
    a, b = run(slice(0, h)), run(slice(h, n))
    for got, want in ((gS, np.concatenate([a[1], b[1]])), (gv, np.concatenate([a[2], b[2]]))):
        assert np.max(np.abs(got - want)) <= 1e-11 * np.max(np.abs(want))
    assert np.all(np.abs(tp - (a[0] + b[0])) <= 1e-11 * (np.abs(a[0]) + np.abs(b[0])) +
                  1e-11 * np.sum(np.abs(gS * d["S"])) / np.array([700.0, 0.1]))
