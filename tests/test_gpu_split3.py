"""Single-precision products large enough for the 16-bit matrix cores (three bf16 parts of every number)."""
import pytest
import torch

from sten_amd import native

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def product(form, a, x, bias=None, pad=0):
    """Through the entry point, with rows `pad` apart and NaN between them."""
    def padded(v):
        buf = torch.full((v.shape[0], v.shape[1] + pad), float("nan"), device=DEV)
        buf[:, :v.shape[1]] = v
        return buf
    O, K = a.shape if form == "nt" else a.shape[::-1]
    T = x.shape[1] if form == "tn" else x.shape[0]
    ab, xb = padded(a), padded(x)
    y = torch.full((T, O + pad), 7.0, device=DEV)
    native.check(getattr(native.load(), "nmg_gemm_" + form)(native.ptr(ab), a.shape[1] + pad, native.ptr(xb), x.shape[1] + pad, native.ptr(y), O + pad,
                                                            native.ptr(bias) if bias is not None else None, O, K, T, native.NMG_F32, None))
    assert bool((y[:, O:] == 7.0).all())
    return y[:, :O]


def operands(form, O, K, T, seed=0):
    gen = torch.Generator(DEV).manual_seed(seed)
    a = torch.randn(*((O, K) if form == "nt" else (K, O)), device=DEV, generator=gen)
    x = torch.randn(*((K, T) if form == "tn" else (T, K)), device=DEV, generator=gen)
    return a, x


def exact(form, a, x):
    return (x.double().t() if form == "tn" else x.double()) @ (a.double().t() if form == "nt" else a.double())


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
@pytest.mark.parametrize("O,K,T", [(2048, 1024, 2048), (2047, 1025, 2045), (2050, 1055, 2046), (1921, 1056, 2048), (1537, 1057, 2047), (768, 2048, 4094), (2046, 1151, 1923)])
def test_ends_of_tiles_and_steps(form, O, K, T):
    a, x = operands(form, O, K, T)
    bias = torch.randn(O, device=DEV)
    y, want = product(form, a, x, bias, pad=3 if K % 2 else 0), exact(form, a, x) + bias.double()
    # K / 16 roundings of sums that grow with the root of their terms, each of half an ulp (2^-24) at the most and 0.58 of
    # that in the mean: sqrt(K / 32) * 0.58 * 2^-24 is 2.8e-7 at K = 2048; the fp32 instruction's sums are off by twice that and more
    assert float((y.double() - want).norm() / want.norm()) <= 3e-7


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
def test_extents_of_the_tests_below_take_the_parts(form):
    # the bound of above; the fp32 instruction rounds eight times as often, 5e-7 and more at this reduction
    a, x = operands(form, 2048, 1024, 2048)
    y, want = product(form, a, x), exact(form, a, x)
    assert float((y.double() - want).norm() / want.norm()) <= 3e-7


@pytest.mark.parametrize("form", ["nt", "tn"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.402e38])
def test_numbers_that_have_no_parts(form, value):
    O, K, T = 2048, 1024, 2048
    a, x = operands(form, O, K, T)
    (x if form == "nt" else x.t())[5, 7] = value
    (x if form == "nt" else x.t())[2000, K - 1] = value
    (a if form == "nt" else a.t())[3, 7] = 0.0
    y, want = product(form, a, x), exact(form, a, x).float()
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isposinf(y), torch.isposinf(want))
    assert torch.equal(torch.isneginf(y), torch.isneginf(want))
    ok = torch.isfinite(want)
    ok[5] = ok[2000] = False
    # K / 2 roundings, those of the fp32 instruction
    assert float((y - want)[ok].norm() / want[ok].norm()) <= 1e-6


@pytest.mark.parametrize("ea,ex", [(0, -100), (0, -120), (8, -130), (-60, -60), (0, 90)])
def test_small_and_large_numbers(ea, ex):
    a, x = operands("nt", 2048, 1024, 2048)
    a, x = a * 2.0 ** ea, (x.double() * 2.0 ** ex).float()
    y, want = product("nt", a, x), exact("nt", a, x)
    assert float((y.double() - want).norm() / want.norm()) <= 1e-6      # as above


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
def test_zeros(form):
    a, x = operands(form, 2048, 1024, 2048)
    (x if form != "tn" else x.t())[1000:] = 0.0
    y = product(form, a, x)
    assert float(y[1000:].abs().max()) == 0.0 and float(y[:1000].abs().min(1).values.max()) > 0.0


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
@pytest.mark.parametrize("e", [-100, -108, -114, -120, -126, -140])
def test_small_rows_among_ordinary_ones(form, e):
    # a few rows of small numbers on either side, in tiles whose other sums are of ordinary size: every row for itself
    print(f"case {form} 2^{e}", flush=True)
    O, K, T = 2048, 1024, 2048
    a, x = operands(form, O, K, T)
    rows_a, rows_x = (a if form == "nt" else a.t()), (x if form != "tn" else x.t())
    small = torch.tensor([3, 200, 2047], device=DEV)
    rows_a[small] = (rows_a[small].double() * 2.0 ** e).float()
    rows_x[small] = (rows_x[small].double() * 2.0 ** e).float()
    y, want = product(form, a, x).double(), exact(form, a, x)
    # K / 2 roundings at the most as above, and half a unit of the smallest fp32 number (2^-149) for every sum
    unit = 2.0 ** -150
    for got, w in ((y, want), (y.t(), want.t())):
        others = torch.ones(got.shape[1], dtype=torch.bool, device=DEV)
        others[small] = False
        got, w = got[:, others], w[:, others]      # (small times small: below every fp32 number)
        off = ((got - w).norm(dim=1) - unit * w.shape[1] ** 0.5).clamp_min(0) / w.norm(dim=1)
        assert float(off.max()) <= 1e-6
    assert float(y[small][:, small].abs().max()) <= 2.0 ** (2 * e + 10)


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
@pytest.mark.parametrize("ea,ex", [(80, -118), (-118, 80), (90, -120), (100, -126), (104, -126)])
def test_small_numbers_times_large_ones(form, ea, ex):
    print(f"case {form} 2^{ea} 2^{ex}", flush=True)
    a, x = operands(form, 2048, 1024, 2048)
    a, x = (a.double() * 2.0 ** ea).float(), (x.double() * 2.0 ** ex).float()
    y, want = product(form, a, x), exact(form, a, x)
    assert float((y.double() - want).norm() / want.norm()) <= 1e-6      # as above


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 2.0 ** 110, -3.0 * 2.0 ** 122])
def test_numbers_that_have_no_parts_in_single_rows(form, value):
    # one such number in one row of a block of 64, at every place of a row in its 32: whichever sums of a lane they reach
    print(f"case {form} {value}", flush=True)
    O, K, T = 2048, 1024, 2048
    for weights in (True, False):
        a, x = operands(form, O, K, T)
        rows = torch.arange(32, device=DEV) * 65
        ((a if form == "nt" else a.t()) if weights else (x if form != "tn" else x.t()))[rows, 9] = value
        y, want = product(form, a, x), exact(form, a, x)
        assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isinf(y), torch.isinf(want.float()))
        y, want = (y.t(), want.t()) if weights else (y, want)
        for got, w in zip((y[rows], y), (want[rows], want)):
            ok = torch.isfinite(w) & torch.isfinite(w.float())
            if got is y:
                ok[rows] = False
            if bool(ok.any()):      # K / 2 roundings, as above
                assert float((got[ok].double() - w[ok]).norm() / w[ok].norm()) <= 1e-6


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 2.0 ** 110])
def test_equal_rows_have_equal_sums(form, value):
    # equal rows of either operand, some in tiles that hold a number without parts, some in tiles of ordinary numbers only
    print(f"case {form} {value}", flush=True)
    O, K, T = 2048, 1024, 2048
    a, x = operands(form, O, K, T)
    rows_a, rows_x = (a if form == "nt" else a.t()), (x if form != "tn" else x.t())
    same = torch.tensor([1, 100, 130, 700, 1500, 2046], device=DEV)
    rows_a[same], rows_x[same] = rows_a[1].clone(), rows_x[1].clone()
    plain = product(form, a, x)
    rows_x[5, 7] = value
    rows_a[1490, 9] = value
    y = product(form, a, x)
    others = torch.ones(2048, dtype=torch.bool, device=DEV)
    others[1490] = False
    assert torch.equal(y[same][:, others], y[1, others].expand(len(same), -1))
    others[1490], others[5] = True, False
    assert torch.equal(y[others][:, same], y[others][:, 1:2].expand(-1, len(same)))
    others[1490] = False
    assert torch.equal(y[others][:, others], plain[others][:, others])      # (rows 5 and 1490 of either operand left out)
