"""Products of few tokens on the dense matrix cores without slices: every tile of the kernel, ragged in every extent."""
import pytest
import torch

import sten_amd as sten
from sten_amd import native
from helpers import rel_l2, to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = {torch.float16: 1e-3, torch.bfloat16: 8e-3}      # fp32 sums, rounded once


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 5, 16, 17, 33, 64])
@pytest.mark.parametrize("O,K", [(16, 8), (30, 72), (129, 1016), (513, 1408), (2050, 2040), (4096, 256), (10640, 520), (8192, 4104)])
def test_few_tokens(O, K, T, dtype):
    print(f"case {O}x{K} T={T} {dtype}", flush=True)
    gen = torch.Generator(DEV).manual_seed(O + K + T)
    w = sten.GroupedNMTensor.from_dense(torch.randn(O, K, device=DEV, generator=gen).to(dtype), 4, 8, sparse_dim=0, group_size=2, group_dim=1)
    dense = w.to_dense().double()
    buf = torch.full((T, K + 8), float("nan"), device=DEV, dtype=dtype)      # a value read behind a row would show
    x = buf[:, :K]
    x.copy_(torch.randn(T, K, device=DEV, generator=gen))
    b = torch.randn(O, device=DEV, generator=gen).to(dtype)
    want = x.double() @ dense.t() + b.double()
    y = sten.spmm(w, x, b, reduce_dim=1)
    assert rel_l2(to_np(y), to_np(want)) <= TOL[dtype]
    # the kernel itself, whatever the rule says, into rows that go on
    lib = native.load()
    df = w.densefrag(1)
    out = torch.full((T, O + 3), 7.0, device=DEV, dtype=dtype)
    native.check(lib.nmg_spmm_densefrag_few(native.ptr(df), O, K, native.ptr(buf), K + 8, native.ptr(out), O + 3, native.ptr(b), T,
                                            native.dtype_code(dtype), None))
    assert rel_l2(to_np(out[:, :O]), to_np(want)) <= TOL[dtype]
    assert bool((out[:, O:] == 7.0).all())


def test_what_it_does_not_take():
    lib = native.load()
    x = torch.zeros(65, 64, device=DEV, dtype=torch.float16)
    args = lambda K, T, ldx: (native.ptr(x), 16, K, native.ptr(x), ldx, native.ptr(x), 16, None, T, native.NMG_F16, None)
    for K, T, ldx in ((12, 1, 64), (64, 65, 64), (64, 1, 60), (0, 1, 64)):
        with pytest.raises(native.NmgError):
            native.check(lib.nmg_spmm_densefrag_few(*args(K, T, ldx)))


@pytest.mark.parametrize("O,K,N", [(1024, 4096, 17), (1024, 4096, 32), (1000, 3000, 64), (2048, 2048, 40), (4096, 4096, 32), (520, 4096, 64)])
@pytest.mark.parametrize("rd", [0, 1])
def test_few_columns_take_it(O, K, N, rd):
    # op(W) @ B with few columns: the kernel for few tokens on the transposed operands, so the same sums bit for bit.  (A walk over
    # the whole reduction adds in another order: of 32 columns x 1024 outputs some dozens then round to the other side.)
    print(f"case {O}x{K} N={N} rd={rd}", flush=True)
    assert native.load().nmg_densefrag_few(O, -(-K // 64) * 64, N) == 1
    gen = torch.Generator(DEV).manual_seed(O + K + N)
    shape = (O, K) if rd == 1 else (K, O)
    w = sten.GroupedNMTensor.from_dense(torch.randn(*shape, device=DEV, generator=gen).half(), 4, 8, sparse_dim=1, group_size=2, group_dim=0)
    b = torch.randn(K, N, device=DEV, generator=gen).half()
    c = sten.spmm_tt_dense(w, b, reduce_dim=rd)
    assert torch.equal(c, sten.spmm(w, b.t().contiguous(), reduce_dim=rd).t())
    dense = w.to_dense().double()
    assert rel_l2(to_np(c), to_np((dense if rd == 1 else dense.t()) @ b.double())) <= TOL[torch.float16]
