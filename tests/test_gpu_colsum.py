"""The column sum (bias gradient) and the dense copy of a weight."""
import pytest
import torch

import sten_amd as sten
from sten_amd import native
from helpers import seeded

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,cols,pitch", [(1, 1, 1), (31, 33, 35), (512, 768, 768), (513, 65, 66), (4096, 100, 100)])
def test_colsum(rows, cols, pitch, dtype):
    x = torch.full((rows, pitch), float("nan"), dtype=dtype, device=DEV)
    x[:, :cols] = seeded((rows, cols), dtype, seed=5).to(DEV)
    y = torch.empty(cols, dtype=dtype, device=DEV)
    native.check(native.load().nmg_colsum(native.ptr(x), rows, cols, pitch, native.ptr(y), native.dtype_code(dtype), None))
    want = x[:, :cols].double().sum(0)
    # against the sum of magnitudes: one rounding of the result, fp32 sums
    bound = {torch.float32: 1e-6, torch.float16: 2 ** -10, torch.bfloat16: 2 ** -7}[dtype]
    assert bool(((y.double() - want).abs() <= bound * x[:, :cols].double().abs().sum(0)).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,row_bytes,extra", [
    (255, 64, 0), (257, 68, 0), (1025, 7164, 2), (1023, 7168, 0), (129, 7172, 6), (2, 8192, 10),      # lanes of 64 and of 128 bytes, either side
])
def test_colsum_at_the_edges_of_its_tiles(rows, row_bytes, extra, dtype):
    # a pitch and a first element that are no multiple of 16 bytes; whole numbers: the sums are exact, one rounding at the end
    cols = row_bytes // dtype.itemsize
    pitch = cols + extra + 1
    x = torch.full((rows * pitch + 1,), float("nan"), dtype=dtype, device=DEV)[1:].view(rows, pitch)
    x[:, :cols] = torch.randint(-8, 9, (rows, cols), generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    y = torch.empty(cols, dtype=dtype, device=DEV)
    native.check(native.load().nmg_colsum(native.ptr(x), rows, cols, pitch, native.ptr(y), native.dtype_code(dtype), None))
    assert torch.equal(y, x[:, :cols].double().sum(0).to(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("n,m,g", [(2, 4, 16), (3, 6, 12), (4, 8, 32)])
@pytest.mark.parametrize("R,C", [(100, 203), (768, 520)])
@pytest.mark.parametrize("along", [0, 1])
def test_dense_copy(dtype, n, m, g, R, C, along):
    w = sten.GroupedNMTensor.from_dense(seeded((R, C), dtype, seed=6).to(DEV), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
    d = w.to_dense()
    for rd, want in ((1, d), (0, d.t())):
        for pad in (1, 64):
            a = w.dense_operand(rd, pad_k=pad)
            assert torch.equal(a[:, :want.shape[1]], want) and not bool(a[:, want.shape[1]:].any())
