"""hk_voigt_adjoint takes every workspace it ever took: two numbers a line are
enough (in fewer parts), and the size of a list serves all shorter ones."""
import ctypes
import re

import numpy as np
import pytest

from helpers import random_lines, species_from


def _needed(L, n):
    """Bytes the call asks for, read from its error for a workspace of no bytes,
    which is returned before any device work."""
    from heliosk import _lib
    lines, tp, cut, grid = _lib.Lines(), _lib.TP(), _lib.Cut(0, 25.0), _lib.Grid()
    lines.nlines, lines.niso, lines.form = n, 1, 0
    tp.T, tp.P = 500.0, 1.0
    grid.numin, grid.dnu, grid.nx = 0.0, 0.01, 1000
    rc = L.hk_voigt_adjoint(ctypes.byref(lines), ctypes.byref(tp), ctypes.byref(cut),
                            ctypes.byref(grid), 256, 256, 256, 256, 256, 0, None)
    m = re.search(r"workspace 0 bytes, (\d+) needed", L.hk_last_error().decode())
    assert rc != 0 and m
    return int(m.group(1))


SIZES = sorted({1, 2, 63, 64, 65, 1000, 2999, 3000, 10599, 10600, 65535, 65536, 65537, 333333,
                1356800, 1356801, 10 ** 7} | set(int(v) for v in np.geomspace(1, 3e7, 40)))


def test_two_numbers_a_line_are_enough():
    from heliosk import engine as E
    L = E.lib()
    for n in SIZES:
        need = _needed(L, n)
        assert need <= 16 * n + 16 + 256
        assert need <= L.hk_voigt_adjoint_workspace_bytes(n)


def test_a_longer_lists_workspace_serves_a_shorter_list():
    from heliosk import engine as E
    L = E.lib()
    q = [L.hk_voigt_adjoint_workspace_bytes(n) for n in SIZES]
    assert q == sorted(q)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 300, 5000, 70000])
def test_gradients_do_not_depend_on_the_workspace(n):
    """Query, the former two numbers a line, and room for two parts: the same
    gradients but for the order of the sums (at most 1e4 terms: 1e4 * 1.1e-16
    of the largest, so 2e-12; in dL/dT and dL/dP, a line's area being the same at
    any width, three digits more may cancel: 2e-9)."""
    import torch
    from heliosk import _lib, engine as E
    L = E.lib()
    d = random_lines(n, seed=n, numin=1000.0, numax=1100.0)
    sp = species_from(d)
    grid = E.make_grid(1000.0, 1100.0, 0.01)
    gK = torch.rand(grid.nx, dtype=torch.float64, device="cuda") + 0.5
    lines, tp, cut = sp.lines(), E._tp(700.0, 0.3, d["iso_Q"]), _lib.Cut(0, 25.0)
    out = []
    for nbytes in (L.hk_voigt_adjoint_workspace_bytes(n), 16 * n + 272,
                   8 * (2 * ((n + 63) // 64) + 8 * n + 2) + 256):
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        g = torch.empty(2 * n + 2, dtype=torch.float64, device="cuda")
        E.check(L.hk_voigt_adjoint(ctypes.byref(lines), ctypes.byref(tp), ctypes.byref(cut),
                                   ctypes.byref(grid), gK.data_ptr(), g.data_ptr(),
                                   g[n:].data_ptr(), g[2 * n:].data_ptr(), ws.data_ptr(), nbytes,
                                   None))
        torch.cuda.synchronize()
        out.append(g.cpu().numpy())
    for o in out[1:]:
        for a, b in ((0, n), (n, 2 * n), (2 * n, 2 * n + 1), (2 * n + 1, 2 * n + 2)):
            s = np.abs(out[0][a:b]).max()
            assert np.abs(o[a:b] - out[0][a:b]).max() <= (2e-12 if b <= 2 * n else 2e-9) * s
