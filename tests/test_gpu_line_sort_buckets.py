"""Ordering of raw lists through buckets: the permutation of a stable argsort,
bit for bit, on the sizes and orders where a bucket can be full, empty or
crossed by equal centres, and with the merge passes' smaller workspace."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("S", "EL", "A", "delta", "vy", "n")


@pytest.fixture(scope="module")
def E():
    from heliosk import engine
    return engine


def _centres(order, n):
    rng = np.random.default_rng(n)
    nu = rng.uniform(0.0, 3000.0, n)
    if order == "rising":
        nu.sort()
    elif order == "falling":
        nu = -np.sort(-nu)
    elif order == "equal":
        nu[:] = 7.5
    elif order == "spike":              # most of the list at two centres, zeros of both signs
        nu[rng.uniform(size=n) < 0.9] = 1234.5
        nu[::7] = 0.0
        nu[1::7] = -0.0
    elif order == "ends":
        nu[::3] = np.inf
        nu[1::3] = -np.inf
    elif order == "clusters":           # log-uniform distances from one centre
        nu = 1000.0 + 10.0 ** rng.uniform(-12, 2, n) * rng.choice([-1, 1], n)
    return nu


@pytest.mark.parametrize("order, n", [("random", 65535), ("random", 65536), ("random", 65537),
                                      ("rising", 100003), ("falling", 200000), ("equal", 150001),
                                      ("spike", 262145), ("ends", 99999), ("clusters", 1000003)])
@pytest.mark.parametrize("iso", [True, False])
def test_bucket_order_is_the_stable_argsort(E, order, n, iso):
    nu = _centres(order, n)
    rng = np.random.default_rng(5)
    f = {k: rng.uniform(0.0, 1.0, n) for k in FIELDS}
    iv = rng.integers(0, 4, n).astype(np.int32) if iso else None
    sp = E.sort_lines(nu, f["S"], f["EL"], f["vy"], f["n"], A=f["A"], delta=f["delta"], iso=iv,
                      iso_mass=(1.0, 2.0, 3.0, 4.0), iso_ab=(1.0,) * 4, iso_sscale=(1.0,) * 4)
    o = np.argsort(nu, kind="stable")
    assert np.array_equal(sp.nu.cpu().numpy().view(np.int64), nu[o].view(np.int64))
    for k in FIELDS:
        assert np.array_equal(getattr(sp, k).cpu().numpy(), f[k][o]), k
    if iso:
        assert np.array_equal(sp.iso.cpu().numpy(), iv[o])


def test_merge_passes_with_the_smaller_workspace(E):
    """Two ping-pong (centre, index) pairs are enough workspace at any size."""
    import torch
    n = 90001
    nu = _centres("spike", n)
    rng = np.random.default_rng(6)
    raw = {k: torch.as_tensor(rng.uniform(0.0, 1.0, n), device="cuda") for k in FIELDS}
    raw["nu"] = torch.as_tensor(nu, device="cuda")
    sp = E.sort_lines(raw["nu"], raw["S"], raw["EL"], raw["vy"], raw["n"], A=raw["A"],
                      delta=raw["delta"])
    out = {k: torch.empty_like(v) for k, v in raw.items()}
    Lin, Lout = sp.lines(), sp.lines()
    for k in raw:
        setattr(Lin, k, raw[k].data_ptr())
        setattr(Lout, k, out[k].data_ptr())
    Lin.iso = Lout.iso = None
    up = lambda b: (b + 255) // 256 * 256
    small = 2 * (up(8 * n) + up(4 * n)) + 256
    L = E.lib()
    assert L.hk_lines_sort_workspace_bytes(n) > small
    ws = torch.empty(small, dtype=torch.uint8, device="cuda")
    E.check(L.hk_lines_sort(ctypes.byref(Lin), ctypes.byref(Lout), ws.data_ptr(), small, None))
    torch.cuda.synchronize()
    for k in raw:
        assert torch.equal(out[k].view(torch.int64), getattr(sp, k).view(torch.int64)), k
