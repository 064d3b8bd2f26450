"""torch.mm with a sparse weight: B transposed beforehand, products that store their result transposed, reductions cut
into slices."""
import numpy as np
import pytest
import torch

import sten_amd as sten
from sten_amd import native
from helpers import rel_l2, seeded, to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# one rounding of the result: half an ulp of 2^-10 / 2^-7 relative, twice that with the order of the fp32 sums
TOL = {torch.float16: 1e-3, torch.bfloat16: 8e-3}


@pytest.mark.parametrize("rows,cols,pitch,dcols", [(1, 1, 1, 8), (64, 128, 128, 64), (65, 129, 131, 72), (7, 1000, 1000, 64), (200, 3, 5, 200), (0, 4, 4, 8)])
def test_transpose(rows, cols, pitch, dcols):
    src = torch.zeros(max(rows, 1), pitch, dtype=torch.float16, device=DEV)
    src[:rows, :cols] = seeded((rows, cols), torch.float16, seed=3).to(DEV)
    dst = torch.full((cols, dcols + 8), 7.0, dtype=torch.float16, device=DEV)
    native.check(native.load().nmg_transpose16(native.ptr(src), rows, cols, pitch, native.ptr(dst), dcols, dcols + 8, None))
    want = torch.full((cols, dcols + 8), 7.0, dtype=torch.float16)
    want[:, :dcols] = 0
    want[:, :rows] = src[:rows, :cols].t().cpu()
    assert torch.equal(dst.cpu(), want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R,C,N", [(256, 768, 128), (257, 832, 129), (300, 1001, 40), (128, 4096, 24), (130, 4104, 31), (1024, 4096, 17), (4104, 72, 4097)])
@pytest.mark.parametrize("n,m,g,along", [(2, 4, 4, 1), (2, 4, 4, 0), (4, 8, 1, 1), (3, 6, 2, 0)])
def test_mm_forms_of_b(R, C, N, n, m, g, along, dtype):
    w = sten.GroupedNMTensor.from_dense(seeded((R, C), dtype, seed=1, std=0.5).to(DEV), n, m, sparse_dim=along, group_size=g,
                                        group_dim=1 - along)
    Wd = to_np(w.to_dense()).astype(np.float64)
    for K, entry in ((C, sten.spmm_tt), (R, lambda w, b: sten.spmm_tt_dense(w, b, reduce_dim=0))):
        b = seeded((K, N), dtype, seed=2).to(DEV)
        want = (Wd if K == C and entry is sten.spmm_tt else Wd.T) @ to_np(b).astype(np.float64)
        wide = torch.zeros(K, N + 3, dtype=dtype, device=DEV)
        wide[:, 1:N + 1] = b
        print(f"case {R}x{C} N={N} {n}:{m}:{g} along={along} {dtype} K={K}", flush=True)
        for form in (b, wide[:, 1:N + 1], b.t().contiguous().t()):      # rows, rows off 16 bytes, columns
            c = entry(w, form)
            assert c.shape == want.shape and rel_l2(to_np(c), want) <= TOL[dtype]
    b = seeded((1, N), dtype, seed=4).to(DEV).expand(C, N)              # rows that share their memory
    assert rel_l2(to_np(sten.spmm_tt(w, b)), Wd @ to_np(b).astype(np.float64)) <= TOL[dtype]
