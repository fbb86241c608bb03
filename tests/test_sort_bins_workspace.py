"""hk_sort_bins_workspace_bytes covers every list of bins of its spectrum: the
size the call asks for (read from its error for a workspace of no bytes, which
is returned before any device work) is never above the query's."""
import ctypes
import re

import numpy as np
import pytest


def _needed(L, nx, seg):
    seg = np.ascontiguousarray(seg, dtype=np.int64)
    # (addresses never read: the workspace is refused first)
    rc = L.hk_sort_bins(256, nx, seg.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), len(seg) - 1,
                        512, 768, 0, None)
    m = re.search(r"workspace 0 bytes, (\d+) needed", L.hk_last_error().decode())
    assert rc != 0 and m
    return int(m.group(1))


def _segments(nx, nseg, longest, first):
    """nseg bins, one (at place `first`) of `longest` points, the rest spread over
    what is left."""
    rest = np.linspace(0, nx - longest, nseg).astype(np.int64)
    lens = np.insert(np.diff(rest), first, longest)
    return np.concatenate([[0], np.cumsum(lens)])


# lengths where the plan's run length (131072), sample spacing (multiples of
# 16368) and number of runs (multiples of 8192) change, and one point either side
EDGES = [16384, 16385, 32736, 65536, 98304, 114688, 131072, 131073, 147312, 262144, 523776,
         524288, 1048576]


@pytest.mark.parametrize("nseg", [1, 100, 300, 3001])
@pytest.mark.parametrize("extra", [0, 1, 965, 3928, 20000, 300000])
def test_query_covers_every_plan(nseg, extra):
    from heliosk import engine as E
    L = E.lib()
    for edge in EDGES:
        for longest in (edge - 1, edge, edge + 1):
            nx = longest + (extra if nseg > 1 else 0)
            q = L.hk_sort_bins_workspace_bytes(nx, nseg)
            need = _needed(L, nx, _segments(nx, nseg, longest, nseg // 2))
            assert need <= q, (nx, nseg, longest, need, q)


def test_lists_that_were_refused():
    from heliosk import engine as E
    L = E.lib()
    for nx, nseg, longest in ((132037, 100, 131072), (135000, 300, 131072), (524855, 300, 523855)):
        need = _needed(L, nx, _segments(nx, nseg, longest, 0))
        assert need <= L.hk_sort_bins_workspace_bytes(nx, nseg), (nx, nseg, longest)


def test_query_stays_close_to_the_longest_plan():
    """The maximum is no more than a few tables above one plan's size."""
    from heliosk import engine as E
    L = E.lib()
    for nx in (1000, 16385, 131073, 3000000, 30000000):
        one = _needed(L, nx, [0, nx])
        assert one <= L.hk_sort_bins_workspace_bytes(nx, 1) <= one + 8 * nx + 65536


@pytest.mark.gpu
@pytest.mark.parametrize("nx, nseg, longest", [(132037, 100, 131072), (524855, 300, 523855)])
def test_lists_that_were_refused_are_sorted(nx, nseg, longest):
    import torch
    from heliosk import engine as E
    seg = _segments(nx, nseg, longest, 3)
    K = np.random.default_rng(nx).lognormal(0.0, 4.0, nx)
    Ks = E.sort_bins(torch.from_numpy(K).cuda(), seg).cpu().numpy()
    for a, b in zip(seg[:-1], seg[1:]):
        np.testing.assert_array_equal(Ks[a:b], np.sort(K[a:b]))
