"""The matching form of the compressor (csrc/nmg_match.h) at the edges of its tiles, against the CPU oracle: values and
indices must be identical."""
import math

import numpy as np
import pytest
import torch

import sten_amd as sten
from helpers import oracle_sparsify, same_bits, to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,m,g", [(2, 4, 16), (1, 8, 32), (2, 8, 32), (3, 6, 12), (4, 8, 32), (2, 6, 5), (3, 8, 24)])
@pytest.mark.parametrize("along", [0, 1])
def test_tiles_at_their_edges(n, m, g, dtype, along):
    # two chunks of the group dim, the second of one column, half of the columns or all but one; blocks that reach
    # beyond the end by every number of positions; continuous values, few magnitudes, zeros
    cols = math.comb(m, n) * g
    gen = torch.Generator().manual_seed(n * 100 + m * 10 + along)
    extras = (1,) if cols > 1000 else (1, cols // 2, cols - 1)
    for k, extra in enumerate(extras):
        for rest in range(m) if cols <= 1000 else (0, 2, m - 1):
            w = torch.randn(cols + extra, 2 * m + rest, generator=gen) * 0.02
            if (rest + k) % 3 == 1:
                w = torch.randint(-3, 4, w.shape, generator=gen).float() * 0.25
            if (rest + k) % 3 == 2:
                w[torch.rand(w.shape, generator=gen) < 0.5] = 0
            w = w.to(dtype)
            w = w if along == 1 else w.t().contiguous()
            print(f"case {n}:{m}:{g} {dtype} shape={tuple(w.shape)} along={along}", flush=True)
            val, idx, _ = oracle_sparsify(w, n, m, along, g, 1 - along)
            t = sten.GroupedNMTensor.from_dense(w.to(DEV), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
            assert np.array_equal(to_np(t.idx), idx)
            assert same_bits(t.val, val)


# every kind of tile: lists of 2 to 64 keys in 16, 32 and 64 lanes, lists that are too long or too short for them, odd
# numbers of columns, a quarter of a wavefront up to sixteen wavefronts per tile, patterns compiled in and any
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n,m,g", [
    (1, 2, 8), (1, 2, 16), (1, 2, 17), (1, 2, 33), (1, 2, 64), (1, 2, 65),
    (1, 3, 7), (2, 3, 21), (1, 4, 4), (1, 4, 8), (3, 4, 16), (1, 5, 4), (4, 5, 12),
    (2, 4, 3), (2, 4, 5), (2, 4, 6), (2, 4, 10), (2, 4, 11), (2, 4, 21), (2, 4, 22), (2, 4, 32), (2, 4, 33), (2, 4, 43), (2, 4, 64), (2, 4, 85),
    (2, 5, 3), (2, 5, 6), (2, 5, 7), (3, 5, 33), (1, 6, 4), (5, 6, 10), (2, 6, 1), (2, 6, 2), (3, 6, 1), (3, 6, 3), (3, 6, 25),
    (1, 7, 9), (3, 7, 2), (3, 7, 29), (1, 8, 2), (1, 8, 8), (7, 8, 5), (2, 8, 1), (2, 8, 2), (2, 8, 3), (2, 8, 4), (2, 8, 17),
    (2, 8, 64), (3, 8, 1), (3, 8, 50), (4, 8, 1), (4, 8, 7), (4, 8, 15),
])
def test_any_group_size(n, m, g, dtype):
    cols = math.comb(m, n) * g
    gen = torch.Generator().manual_seed(n * 1000 + m * 100 + g)
    for along in (0, 1):
        for k, (extra, blocks, rest) in enumerate(((cols - 1, 17, 0), (cols // 2, 3, m - 1), (1, 2, 1))):
            w = torch.randn(cols + extra, blocks * m + rest, generator=gen) * 0.02
            if (k + along) % 3 == 1:
                w = torch.randint(-3, 4, w.shape, generator=gen).float() * 0.25
            if (k + along) % 3 == 2:
                w[torch.rand(w.shape, generator=gen) < 0.5] = 0
            w = w.to(dtype)
            w = w if along == 1 else w.t().contiguous()
            print(f"case {n}:{m}:{g} {dtype} shape={tuple(w.shape)} along={along}", flush=True)
            val, idx, _ = oracle_sparsify(w, n, m, along, g, 1 - along)
            t = sten.GroupedNMTensor.from_dense(w.to(DEV), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
            assert np.array_equal(to_np(t.idx), idx)
            assert same_bits(t.val, val)


@pytest.mark.parametrize("n,m,g,dtype", [(2, 4, 43, torch.float16), (2, 4, 85, torch.float32), (1, 8, 33, torch.float32),
                                         (2, 8, 18, torch.float16), (3, 6, 20, torch.bfloat16), (1, 4, 66, torch.float16)])
def test_two_wavefronts_per_tile(n, m, g, dtype):
    """Tiles of 257 to 512 columns, enough of them to fill the chip; the last chunk and the last block are partial."""
    cols = math.comb(m, n) * g
    gen = torch.Generator().manual_seed(g)
    w = (torch.randn(cols + cols // 3, 1030 * m + 1, generator=gen) * 0.02).to(dtype)
    w[torch.rand(w.shape, generator=gen) < 0.1] = 0
    for along in (0, 1):
        x = w if along == 1 else w.t().contiguous()
        print(f"case {n}:{m}:{g} {dtype} shape={tuple(x.shape)} along={along}", flush=True)
        val, idx, _ = oracle_sparsify(x, n, m, along, g, 1 - along)
        t = sten.GroupedNMTensor.from_dense(x.to(DEV), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
        assert np.array_equal(to_np(t.idx), idx)
        assert same_bits(t.val, val)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n,m,g", [(2, 4, 16), (1, 8, 32), (2, 8, 32), (3, 6, 12), (4, 8, 32), (2, 4, 8), (2, 4, 32), (2, 8, 8), (3, 8, 8),
                                   (2, 4, 129), (1, 4, 257), (2, 4, 320)])
def test_columns_that_want_the_same_patterns(n, m, g, dtype):
    # magnitudes that fall along the block: most columns propose to one pattern, lists and buckets run over, and the
    # refusals come in long chains; mild, so that the later rounds see them, and steep
    cols = math.comb(m, n) * g
    gen = torch.Generator().manual_seed(n * 100 + m * 10 + g)
    for along in (0, 1):
        for fall in (0.9, 0.6):
            w = (torch.randn(2 * cols - 3, 3 * m, generator=gen) * 0.1 + 1) * fall ** (torch.arange(3 * m) % m)
            w = w.to(dtype)
            w = w if along == 1 else w.t().contiguous()
            print(f"case {n}:{m}:{g} {dtype} along={along} fall={fall}", flush=True)
            val, idx, _ = oracle_sparsify(w, n, m, along, g, 1 - along)
            t = sten.GroupedNMTensor.from_dense(w.to(DEV), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
            assert np.array_equal(to_np(t.idx), idx)
            assert same_bits(t.val, val)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n,m,g", [(2, 8, 32), (3, 6, 12), (4, 8, 4), (3, 8, 8), (5, 8, 2), (2, 6, 1), (3, 7, 1), (6, 8, 1), (1, 8, 32), (2, 4, 16)])
def test_partial_blocks_whose_classes_tie(n, m, g, dtype):
    # every number of real positions; equal magnitudes make a column's best score one of several classes', zeros leave classes
    # without a score, and one chunk is short: the order inside a class and the second choice at the same score decide
    cols = math.comb(m, n) * g
    gen = torch.Generator().manual_seed(n * 100 + m * 10 + g)
    for rest in range(1, m):
        for kind in range(3):
            w = torch.randint(0, (2, 3, 9)[kind], (cols + cols // 3 + 1, m + rest), generator=gen).float() * 0.5
            w = (w * torch.where(torch.rand(w.shape, generator=gen) < 0.5, -1.0, 1.0)).to(dtype)
            print(f"case {n}:{m}:{g} {dtype} rest={rest} kind={kind}", flush=True)
            val, idx, _ = oracle_sparsify(w, n, m, 1, g, 0)
            t = sten.GroupedNMTensor.from_dense(w.to(DEV), n, m, sparse_dim=1, group_size=g, group_dim=0)
            assert np.array_equal(to_np(t.idx), idx)
            assert same_bits(t.val, val)


# The keys of a partial block are sorted in registers, 1, 4 or 8 to a thread of 256 or 512: runs that end at, before and
# behind the extents of a thread, a wavefront and the workgroup.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,m,g,columns", [
    (3, 6, 12, (1, 2, 63, 64, 65, 128, 129)), (2, 8, 32, (3, 4, 5, 255, 257, 511, 513, 769)), (4, 8, 32, (7, 8, 9, 511, 513, 1025)),
    (2, 4, 60, (129, 257)), (3, 8, 20, (512, 1023)),
])
def test_partial_blocks_of_any_number_of_columns(n, m, g, columns, dtype):
    gen = torch.Generator().manual_seed(n * 100 + m * 10 + g)
    for k, cols in enumerate(columns):
        rest = 1 + k % (m - 1)
        w = torch.randn(cols, m + rest, generator=gen) * 0.02
        if k % 3 == 2:
            w = torch.randint(-3, 4, w.shape, generator=gen).float() * 0.25
        w = w.to(dtype)
        print(f"case {n}:{m}:{g} {dtype} shape={tuple(w.shape)}", flush=True)
        val, idx, _ = oracle_sparsify(w, n, m, 1, g, 0)
        t = sten.GroupedNMTensor.from_dense(w.to(DEV), n, m, sparse_dim=1, group_size=g, group_dim=0)
        assert np.array_equal(to_np(t.idx), idx)
        assert same_bits(t.val, val)


@pytest.mark.parametrize("n,m,g", [(4, 8, 45), (4, 8, 46), (4, 8, 47), (3, 8, 58), (3, 8, 59), (3, 6, 100)])
@pytest.mark.parametrize("along", [0, 1])
def test_largest_tiles_with_a_partial_block(n, m, g, along):
    # single precision: 4:8:46 and more leave no room in LDS for a list of a partial block's refused columns, and no other
    # compressor takes a tile of this size; at 3:6:100 it would cost the second workgroup of a CU
    cols = math.comb(m, n) * g
    gen = torch.Generator().manual_seed(g)
    w = torch.randn(cols, 2 * m + 5, generator=gen) * 0.02
    w = w if along == 1 else w.t().contiguous()
    print(f"case {n}:{m}:{g} along={along}", flush=True)
    val, idx, _ = oracle_sparsify(w, n, m, along, g, 1 - along)
    t = sten.GroupedNMTensor.from_dense(w.to(DEV), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
    assert np.array_equal(to_np(t.idx), idx)
    assert same_bits(t.val, val)


# The first round sorts by pattern and by bins of the score, four to an octave (two where a tile has many patterns): scores in one bin, at the bins'
# bounds, many octaves below the largest, subnormal, infinite.  Lists of up to 128 keys, two or four to a lane; tiles of 23 and 24 columns.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,m,g", [(2, 4, 16), (1, 8, 32), (3, 6, 12), (2, 8, 32), (4, 8, 32), (2, 4, 4), (1, 4, 6), (1, 4, 5), (2, 4, 65),
                                   (1, 4, 128), (1, 4, 129), (3, 8, 8), (4, 8, 6)])
def test_scores_of_any_size(n, m, g, dtype):
    cols = math.comb(m, n) * g
    gen = torch.Generator().manual_seed(n * 100 + m * 10 + g)
    for kind in ("equal", "powers", "tails", "subnormal", "infinite"):
        w = torch.randn(cols + cols // 2, 2 * m, generator=gen)
        if kind == "equal":
            w = torch.full_like(w, 0.5)
        elif kind == "powers":
            w = 2.0 ** torch.randint(-9, 1, w.shape, generator=gen) * (1 + 0.25 * torch.randint(0, 4, w.shape, generator=gen))
        elif kind == "tails":
            w = w * torch.exp(2 * torch.randn(w.shape, generator=gen))
        elif kind == "subnormal":
            w = w * 8 * torch.finfo(dtype).smallest_normal / 64
        else:
            w[torch.rand(w.shape, generator=gen) < 0.05] = math.inf
        w = w.to(dtype)
        for along in (0, 1):
            x = w if along == 1 else w.t().contiguous()
            print(f"case {n}:{m}:{g} {dtype} {kind} along={along}", flush=True)
            val, idx, _ = oracle_sparsify(x, n, m, along, g, 1 - along)
            t = sten.GroupedNMTensor.from_dense(x.to(DEV), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
            assert np.array_equal(to_np(t.idx), idx)
            assert same_bits(t.val, val)


# A sum over a weight that is no number is larger than every other one, whatever number its bits stand for (those of 0x7FFF in 16 bits and 0x7FFFFFFF
# lie where the high word of a double is no number either): equal ones take the places of infinities, in whole blocks and partial ones.
@pytest.mark.parametrize("dtype,bits", [(torch.float16, 0x7E00), (torch.float16, 0x7FFF), (torch.float16, 0xFFFF), (torch.bfloat16, 0x7FC0), (torch.bfloat16, 0x7FFF),
                                        (torch.float32, 0x7FC00000), (torch.float32, 0x7FF00001), (torch.float32, 0x7FFFFFFF)])
@pytest.mark.parametrize("n,m,g", [(2, 4, 16), (1, 8, 32), (3, 6, 12), (2, 8, 32), (4, 8, 32), (2, 4, 4), (1, 4, 129), (3, 8, 8), (4, 8, 6)])
@pytest.mark.parametrize("rest", [0, 1])
def test_weights_that_are_no_numbers(n, m, g, dtype, bits, rest):
    cols = math.comb(m, n) * g
    gen = torch.Generator().manual_seed(n * 100 + m * 10 + g)
    w = torch.randn(cols + cols // 2, 4 * m + rest, generator=gen).to(dtype)
    odd = torch.rand(w.shape, generator=gen) < 0.03
    whole = {2: torch.int16, 4: torch.int32}[w.element_size()]
    value = bits - (1 << 8 * w.element_size()) if bits >> (8 * w.element_size() - 1) else bits
    as_none, as_inf = w.view(whole).masked_fill(odd, value).view(dtype), w.masked_fill(odd, math.inf)
    for along in (0, 1):
        x, y = (t if along == 1 else t.t().contiguous() for t in (as_none, as_inf))
        print(f"case {n}:{m}:{g} {dtype} {bits:x} rest={rest} along={along}", flush=True)
        val, idx, _ = oracle_sparsify(y, n, m, along, g, 1 - along)
        t = sten.GroupedNMTensor.from_dense(x.to(DEV), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
        assert np.array_equal(to_np(t.idx), idx)
        none = np.isinf(val.astype(np.float32))
        assert np.array_equal(torch.isnan(t.val).cpu().numpy(), none)
        assert bool((t.val.cpu().view(whole)[torch.from_numpy(none)] == value).all())
        assert same_bits(t.val.masked_fill(torch.isnan(t.val), math.inf), val)


# Which later rounds a tile takes: lists of one key, of up to 128 and 256 (two and four to a lane), of more, which stay in LDS, as all of more than 64 keys
# do in a partial block of more than 256 columns; tiles of 16, 18 and 20 columns; tiles of 48 and more columns on a quarter and on half of a wavefront.  Whole blocks and a partial one.
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n,m,g", [(1, 8, 2), (1, 2, 9), (2, 5, 2), (1, 4, 4), (1, 8, 4), (1, 6, 8), (1, 8, 8), (2, 6, 4), (3, 6, 3), (2, 8, 2), (2, 8, 1), (3, 6, 1),
                                   (4, 8, 1), (1, 2, 128), (1, 2, 129), (2, 4, 160), (1, 8, 256), (1, 2, 257), (1, 4, 257),
                                   (1, 2, 1), (2, 5, 3), (1, 6, 3), (1, 4, 64), (1, 4, 65), (2, 5, 65), (3, 6, 100), (1, 2, 320), (1, 3, 700), (2, 4, 400)])
@pytest.mark.parametrize("rest", [0, 1])
def test_later_rounds_of_any_tile(n, m, g, dtype, rest):
    cols = math.comb(m, n) * g
    gen = torch.Generator().manual_seed(n * 100 + m * 10 + g + rest)
    for along in (0, 1):
        w = torch.randn(2 * cols + cols // 2, 4 * m + rest, generator=gen).to(dtype)
        x = w if along == 1 else w.t().contiguous()
        print(f"case {n}:{m}:{g} {dtype} rest={rest} along={along}", flush=True)
        val, idx, _ = oracle_sparsify(x, n, m, along, g, 1 - along)
        t = sten.GroupedNMTensor.from_dense(x.to(DEV), n, m, sparse_dim=along, group_size=g, group_dim=1 - along)
        assert np.array_equal(to_np(t.idx), idx)
        assert same_bits(t.val, val)


# Lists of more than 128 keys in tiles of two wavefronts, which take tensors of at least 2048 tiles.
@pytest.mark.parametrize("n,m,g", [(1, 2, 128), (1, 2, 129), (1, 2, 256), (1, 3, 160)])
def test_long_lists_in_tiles_of_two_wavefronts(n, m, g):
    cols = math.comb(m, n) * g
    w = torch.randn(8 * cols, 256 * m, generator=torch.Generator().manual_seed(g)).to(torch.float16)
    print(f"case {n}:{m}:{g}", flush=True)
    val, idx, _ = oracle_sparsify(w, n, m, 1, g, 0)
    t = sten.GroupedNMTensor.from_dense(w.to(DEV), n, m, sparse_dim=1, group_size=g, group_dim=0)
    assert np.array_equal(to_np(t.idx), idx)
    assert same_bits(t.val, val)
