"""Dense product of two operands as rows in memory, on 256 x 256 tiles and beside their limit."""
import pytest
import torch

from sten_amd import native
from sten_amd._host_loader import host
from helpers import rel_l2, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# the one rounding of the result is off by half an ulp, 2^-11 / 2^-8 of a value at most; a fiftieth more for the fp32 sums
TOL = {torch.float16: 5e-4, torch.bfloat16: 4e-3}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("O,K,T,pad", [(4096, 64, 4096, 0), (4000, 192, 4090, 8), (8192, 128, 1801, 0), (1, 64, 65537, 0)])
def test_gemm_nt_square_tiles(O, K, T, pad, dtype):
    A, X = seeded((O, K + pad), dtype, seed=1).to(DEV), seeded((T, K + pad), dtype, seed=2).to(DEV)
    bias = seeded((O,), dtype, seed=3).to(DEV)
    Y = torch.full((T, O + 8), 7.0, dtype=dtype, device=DEV)
    native.check(native.load().nmg_gemm_nt(native.ptr(A), K + pad, native.ptr(X), K + pad, native.ptr(Y), O + 8, native.ptr(bias), O, K, T,
                                           native.dtype_code(dtype), None))
    want = X[:, :K].float() @ A[:, :K].float().t() + bias.float()
    assert bool((Y[:, O:] == 7.0).all())
    assert rel_l2(Y[:, :O].float().cpu().numpy(), want.cpu().numpy()) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tn,shape,pitch", [
    (False, (512, 72), 2 ** 21),      # 2 GiB of rows
    (True, (9, 40), 2 ** 24),         # rows of 2^24
    (False, (512, 72), 2 ** 21 - 8),  # the last ones that the 16-bit kernels take
    (True, (9, 40), 2 ** 24 - 8),
])
def test_dense_product_beyond_the_16_bit_kernels_offsets(tn, shape, pitch, dtype):
    """Widened for the fp32 kernel, the result rounded once: no library product."""
    print(f"case tn={tn} {shape} pitch={pitch} {dtype}", flush=True)
    A = torch.empty(shape[0] * pitch, dtype=dtype, device=DEV).as_strided(shape, (pitch, 1))
    A.copy_(seeded(shape, dtype, seed=4))
    X = seeded((shape[0], 24) if tn else (33, shape[1]), dtype, seed=5).to(DEV)
    for x, a in ((X, A), (A, X)):
        got = host.dense_product(tn, x, a)
        want = x.double().t() @ a.double() if tn else x.double() @ a.double().t()
        assert got is not None and got.dtype == dtype and got.shape == want.shape
        assert rel_l2(got.double().cpu().numpy(), want.cpu().numpy()) <= TOL[dtype]
