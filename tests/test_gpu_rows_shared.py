"""Activations whose rows share memory: one row expanded over the tokens, windows that overlap, of any reduction."""
import pytest
import torch

import sten_amd as sten
from helpers import rel_l2, to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = {torch.float16: 1e-3, torch.bfloat16: 8e-3, torch.float32: 1e-5}      # fp32 sums, rounded once


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,m,g,along", [(2, 4, 16, 1), (4, 8, 2, 1), (2, 4, 16, 0), (3, 6, 2, 1)])
@pytest.mark.parametrize("K", [72, 2216, 1000, 999, 256])
@pytest.mark.parametrize("T", [1, 2, 16, 17, 64, 300, 600])
def test_expanded_and_overlapping_rows(T, K, n, m, g, along, dtype):
    print(f"case {K} T={T} {n}:{m}:{g} sparse_dim={along} {dtype}", flush=True)
    O = 520
    gen = torch.Generator(DEV).manual_seed(K + T)
    w = sten.GroupedNMTensor.from_dense(torch.randn(O, K, device=DEV, generator=gen).to(dtype), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
    dense = w.to_dense().double()
    flat = torch.randn(T * 8 + K, device=DEV, generator=gen).to(dtype)
    for x in (flat[:K].expand(T, K), flat.unfold(0, K, 8)[:T], flat.unfold(0, K, 3)[:T]):
        y = sten.spmm(w, x, reduce_dim=1)
        assert rel_l2(to_np(y), to_np(x.double() @ dense.t())) <= TOL[dtype]
        if x.stride(0) == 0:
            assert torch.equal(y, y[:1].expand(T, O))
