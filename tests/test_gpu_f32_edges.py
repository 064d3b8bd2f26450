"""Single precision products at extents, pitches and alignments that are no multiples of anything."""
import pytest
import torch

from sten_amd import native
from helpers import rel_l2, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
@pytest.mark.parametrize("O,K,T", [(1, 1, 1), (3, 17, 2), (4, 16, 5), (5, 33, 4), (33, 15, 65), (98, 70, 131), (257, 129, 67), (771, 62, 1025), (2139, 333, 504), (3070, 96, 516),
                                   # the loop without guards and the steps behind it: whole steps, one more and one less position; fewer than four rows
                                   (70, 144, 99), (130, 319, 65), (98, 257, 131), (1024, 321, 257), (5, 256, 3), (3, 300, 200), (200, 300, 3)])
@pytest.mark.parametrize("pad,off", [(0, 0), (1, 1), (3, 2)])
def test_gemm_forms(form, O, K, T, pad, off):
    print(f"case {form} O={O} K={K} T={T} pad={pad} off={off}", flush=True)

    def operand(rows, cols, seed):
        # NaN around what the product may use: a value read from there would show
        buf = torch.full((rows * (cols + pad) + off,), float("nan"), device=DEV)
        v = buf[off:].view(rows, cols + pad)[:, :cols]
        v.copy_(seeded((rows, cols), torch.float32, seed=seed).to(DEV))
        return v, buf[off:]
    a, abuf = operand(*((O, K) if form == "nt" else (K, O)), 1)
    x, xbuf = operand(*((K, T) if form == "tn" else (T, K)), 2)
    y = torch.full((T, O + 2), 7.0, device=DEV)
    native.check(getattr(native.load(), "nmg_gemm_" + form)(native.ptr(abuf), a.shape[1] + pad, native.ptr(xbuf), x.shape[1] + pad, native.ptr(y),
                                                            O + 2, None, O, K, T, native.NMG_F32, None))
    want = (x.double() if form != "tn" else x.double().t()) @ (a.double().t() if form == "nt" else a.double())
    assert bool((y[:, O:] == 7.0).all())
    # fp32 sums of K <= 333 terms: K ulps / 2 at the very most, sqrt(K) of them in earnest
    assert rel_l2(y[:, :O].cpu().numpy(), want.cpu().numpy()) <= 3e-6
