"""Long raw lists: the last and first list of each bucket width (512 and 1024
threads a bucket, the splitter table in LDS full) and of the merge passes beyond,
against the device's stable argsort, bit for bit."""
import pytest

pytestmark = pytest.mark.gpu

MAX_BUCKETS = 8192


@pytest.mark.parametrize("n", [MAX_BUCKETS * 1280, MAX_BUCKETS * 1280 + 1, MAX_BUCKETS * 2560,
                               MAX_BUCKETS * 2560 + 1])
@pytest.mark.parametrize("ties", [False, True])
def test_long_list_is_the_stable_argsort(n, ties):
    import torch
    from heliosk import engine as E
    g = torch.Generator(device="cuda").manual_seed(n)
    nu = torch.rand(n, dtype=torch.float64, device="cuda", generator=g) * 30000.0
    if ties:
        nu = torch.round(nu)                    # ~700 lines of each centre
    place = torch.arange(n, dtype=torch.float64, device="cuda")
    f = {k: place * c for k, c in (("S", 1.0), ("EL", 0.5), ("A", 3.0), ("delta", -1.0),
                                   ("vy", 2.0), ("n", -0.25))}
    iso = (torch.arange(n, device="cuda") % 4).to(torch.int32)
    sp = E.sort_lines(nu, f["S"], f["EL"], f["vy"], f["n"], A=f["A"], delta=f["delta"], iso=iso,
                      iso_mass=(1.0, 2.0, 3.0, 4.0), iso_ab=(1.0,) * 4, iso_sscale=(1.0,) * 4)
    want, o = torch.sort(nu, stable=True)
    assert torch.equal(sp.nu, want)
    assert torch.equal(sp.S, o.to(torch.float64))
    for k, c in (("EL", 0.5), ("A", 3.0), ("delta", -1.0), ("vy", 2.0), ("n", -0.25)):
        assert torch.equal(getattr(sp, k), sp.S * c), k
    assert torch.equal(sp.iso, (o % 4).to(torch.int32))
