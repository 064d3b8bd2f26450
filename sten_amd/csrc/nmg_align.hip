// 16-bit matrices into the shape the matrix-core kernels read: rows that start on 16 bytes, a row length and a row
// count rounded up, zeros in between -- in one pass.
//
// The products want whole K steps and 16-byte rows; an extent such as 1001 has neither.  A padded copy of the activations
// costs their size twice in HBM traffic (a few us), against 3 to 8 times the time of the product in the kernels that take
// any shape.  Bound by memory; a source row may start on any 2-byte boundary (global loads of 16 bytes need no
// alignment, they only touch one more line).  1857 x 10385 and its like: 3 us for 512 rows against 14 us for a fill
// and a strided copy.
#include "nmg_common.h"
#include "nmg_tile.h"

namespace nmg {

struct CopyRows {
    const uint16_t *src;
    uint16_t *dst;
    int64_t rows, cols, ld_src, dst_rows, dst_cols, ld_dst;
    uint32_t per_row;      // pieces of 8 elements per destination row
};

__global__ __launch_bounds__(256) void copy_rows16_kernel(CopyRows P)
{
    const int64_t total = P.dst_rows * P.per_row;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t r = i / P.per_row;
        const int64_t c = (i - r * P.per_row) * 8;
        uint16_t v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        const uint16_t *s = P.src + r * P.ld_src + c;
        if (r < P.rows) {
            if (c + 8 <= P.cols) __builtin_memcpy(v, s, 16);
            else
                for (int e = 0; e < 8; e++) v[e] = c + e < P.cols ? s[e] : (uint16_t)0;
        }
        uint16_t *d = P.dst + r * P.ld_dst + c;
        if (c + 8 <= P.dst_cols) __builtin_memcpy(d, v, 16);
        else
            for (int e = 0; e < 8; e++)
                if (c + e < P.dst_cols) d[e] = v[e];
    }
}

// dst [cols, dst_cols] = src [rows, cols] transposed, zeros for dst_cols > rows.  A workgroup moves 64 source rows x
// 128 columns through LDS: 16 bytes per lane from memory, eight 2-byte reads of a column (rows 260 bytes apart: the 8
// pieces x 8 columns of a wavefront meet every bank once) and 16 bytes per lane back, 128 contiguous bytes per
// destination row.  Bound by memory: 4096 x 2048 (33.6 MB moved) 7.3 us, 4.6 TB/s, launch included.
struct Transpose16 {
    const uint16_t *src;
    uint16_t *dst;
    int64_t rows, cols, ld_src, dst_cols, ld_dst;
    int64_t tiles_c;
};
constexpr int TR_ROWS = 64, TR_COLS = 128, TR_PITCH = TR_COLS + 2;

__global__ __launch_bounds__(256) void transpose16_kernel(Transpose16 P)
{
    __shared__ __align__(16) uint16_t tile[TR_ROWS * TR_PITCH];
    const int tid = threadIdx.x;
    const int64_t r0 = blockIdx.x / P.tiles_c * TR_ROWS, c0 = blockIdx.x % P.tiles_c * TR_COLS;
#pragma unroll
    for (int it = 0; it < TR_ROWS * TR_COLS / 8 / 256; it++) {
        const int i = it * 256 + tid, r = i / (TR_COLS / 8), c = i % (TR_COLS / 8) * 8;
        uint32_t v[4] = {0, 0, 0, 0};
        if (r0 + r < P.rows) {
            const uint16_t *s = P.src + (r0 + r) * P.ld_src + c0 + c;
            if (c0 + c + 8 <= P.cols) __builtin_memcpy(v, s, 16);
            else
                for (int e = 0; e < 8; e++)
                    if (c0 + c + e < P.cols) v[e / 2] |= (uint32_t)s[e] << (16 * (e & 1));
        }
#pragma unroll
        for (int e = 0; e < 4; e++) *(uint32_t *)(tile + r * TR_PITCH + c + 2 * e) = v[e];
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < TR_ROWS * TR_COLS / 8 / 256; it++) {
        const int i = it * 256 + tid, k = i % (TR_ROWS / 8) * 8, c = i / (TR_ROWS / 8);
        if (c0 + c >= P.cols || r0 + k >= P.dst_cols) continue;
        uint32_t v[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
            v[e] = (uint32_t)tile[(k + 2 * e) * TR_PITCH + c] | ((uint32_t)tile[(k + 2 * e + 1) * TR_PITCH + c] << 16);
        __builtin_memcpy(P.dst + (c0 + c) * P.ld_dst + r0 + k, v, 16);
    }
}

// y[c] = sum over the rows of x[r, c], single-precision sums, rounded once: the bias gradient of a linear layer.  A
// workgroup owns 64 or 128 bytes of every row (lanes of 16 bytes; narrow, so that a few hundred columns still are a few
// dozen workgroups), 256 or 128 rows at a time with four loads per lane in flight, and adds its partial rows through LDS in
// order: one launch, no semaphores to clear.  Bound by the loads that a few dozen workgroups keep in flight.  us, lanes of 4 bytes
// and 32 rows at a time -> this: bf16 1667 x 3840 32.5 -> 5.7, 2184 x 1472 40.0 -> 5.4, 3881 x 1640 70.3 -> 9.6, fp16 4096 x 16384
// 104 -> 28 (4.8 TB/s), fp32 512 x 768 3.3 -> 3.2 (the library's sum and the fill in front of it 11.5), 4096 x 4096 19.3 -> 19.1.
struct ColSum {
    const void *x;
    void *y;
    int64_t rows, cols, ld;
};
constexpr int CS_THREADS = 1024, CS_DEEP = 4;

template <typename T, int CS_LANES> __global__ __launch_bounds__(CS_THREADS) void colsum_kernel(ColSum P)
{
    constexpr int CS_ROWS = CS_THREADS / CS_LANES;
    constexpr int E = 16 / (int)sizeof(T), W = CS_LANES * E, GROUPS = CS_THREADS / W;
    __shared__ float part[CS_ROWS][W + 4], sums[GROUPS][W];
    const int tid = threadIdx.x, cl = tid % CS_LANES, rl = tid / CS_LANES;
    const int64_t c = (int64_t)blockIdx.x * W + cl * E;
    const int valid = (int)min((int64_t)E, P.cols - c);      // columns of the lane that exist
    float acc[E];
#pragma unroll
    for (int e = 0; e < E; e++) acc[e] = 0.f;
    const T *x = (const T *)P.x + c;
    if (valid == E) {
        for (int64_t r0 = rl; r0 < P.rows; r0 += CS_ROWS * CS_DEEP) {
            T v[CS_DEEP][E];
#pragma unroll
            for (int u = 0; u < CS_DEEP; u++)      // (a global load needs the alignment of its elements only)
                __builtin_memcpy(v[u], x + min(r0 + u * CS_ROWS, P.rows - 1) * P.ld, 16);
#pragma unroll
            for (int u = 0; u < CS_DEEP; u++)
#pragma unroll
                for (int e = 0; e < E; e++) acc[e] += r0 + u * CS_ROWS < P.rows ? to_f32(v[u][e]) : 0.f;
        }
    } else {
        for (int64_t r = rl; r < P.rows; r += CS_ROWS)
#pragma unroll
            for (int e = 0; e < E; e++)
                if (e < valid) acc[e] += to_f32(x[r * P.ld + e]);
    }
#pragma unroll
    for (int e = 0; e < E; e++) part[rl][cl * E + e] = acc[e];
    __syncthreads();
    const int col = tid % W, grp = tid / W;
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < CS_ROWS / GROUPS; r++) s += part[grp * (CS_ROWS / GROUPS) + r][col];
    sums[grp][col] = s;
    __syncthreads();
    const int64_t to = (int64_t)blockIdx.x * W + tid;
    if (tid >= W || to >= P.cols) return;
    s = 0.f;
#pragma unroll
    for (int r = 0; r < GROUPS; r++) s += sums[r][tid];
    if constexpr (sizeof(T) == 4) ((float *)P.y)[to] = s;
    else ((uint16_t *)P.y)[to] = f32_to_bits16(s, (T *)nullptr);
}

}  // namespace nmg

using namespace nmg;

extern "C" int nmg_copy_rows16(const void *d_src, int64_t rows, int64_t cols, int64_t ld_src, void *d_dst, int64_t dst_rows,
                               int64_t dst_cols, int64_t ld_dst, void *stream)
{
    NMG_REQUIRE(rows >= 0 && cols >= 0 && dst_rows >= 0 && dst_cols >= 0, NMG_ERR_ARG, "negative extent");
    NMG_REQUIRE((rows <= 1 || ld_src >= cols) && (dst_rows <= 1 || ld_dst >= dst_cols), NMG_ERR_ARG,
                "leading dimension smaller than row length");
    if (dst_rows == 0 || dst_cols == 0) return NMG_OK;
    NMG_REQUIRE(d_dst && (d_src || rows == 0 || cols == 0), NMG_ERR_ARG, "null device pointer");
    NMG_REQUIRE(dst_cols < ((int64_t)1 << 34), NMG_ERR_UNSUPPORTED, "rows too long");
    CopyRows P{(const uint16_t *)d_src, (uint16_t *)d_dst, rows < dst_rows ? rows : dst_rows, cols < dst_cols ? cols : dst_cols,
               ld_src, dst_rows, dst_cols, ld_dst, (uint32_t)((dst_cols + 7) / 8)};
    const int64_t blocks = (dst_rows * P.per_row + 255) / 256;
    hipLaunchKernelGGL(copy_rows16_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, (hipStream_t)stream, P);
    NMG_HIP_TRY(hipGetLastError());
    return NMG_OK;
}

extern "C" int nmg_transpose16(const void *d_src, int64_t rows, int64_t cols, int64_t ld_src, void *d_dst, int64_t dst_cols,
                               int64_t ld_dst, void *stream)
{
    NMG_REQUIRE(rows >= 0 && cols >= 0, NMG_ERR_ARG, "negative extent");
    NMG_REQUIRE(dst_cols >= rows && dst_cols % 8 == 0 && ld_dst >= dst_cols && (rows <= 1 || ld_src >= cols), NMG_ERR_ARG,
                "a destination row holds a column and ends on a multiple of 8; leading dimensions cover their rows");
    if (cols == 0 || dst_cols == 0) return NMG_OK;
    NMG_REQUIRE(d_dst && (d_src || rows == 0), NMG_ERR_ARG, "null device pointer");
    Transpose16 P{(const uint16_t *)d_src, (uint16_t *)d_dst, rows, cols, ld_src, dst_cols, ld_dst, (cols + TR_COLS - 1) / TR_COLS};
    const int64_t tiles = P.tiles_c * ((dst_cols + TR_ROWS - 1) / TR_ROWS);
    NMG_REQUIRE(tiles <= 0x7fffffffLL, NMG_ERR_UNSUPPORTED, "matrix too large for one launch");
    hipLaunchKernelGGL(transpose16_kernel, dim3((unsigned)tiles), dim3(256), 0, (hipStream_t)stream, P);
    NMG_HIP_TRY(hipGetLastError());
    return NMG_OK;
}

extern "C" int nmg_colsum(const void *d_x, int64_t rows, int64_t cols, int64_t ld, void *d_y, int dtype, void *stream)
{
    NMG_REQUIRE(dtype == NMG_F32 || dtype == NMG_F16 || dtype == NMG_BF16, NMG_ERR_UNSUPPORTED, "colsum takes f32/f16/bf16");
    NMG_REQUIRE(rows >= 0 && cols >= 0 && (rows <= 1 || ld >= cols), NMG_ERR_ARG, "invalid extents");
    if (cols == 0) return NMG_OK;
    NMG_REQUIRE(d_y && (d_x || rows == 0), NMG_ERR_ARG, "null device pointer");
    ColSum P{d_x, d_y, rows, cols, ld};
    const int64_t row_bytes = cols * (dtype == NMG_F32 ? 4 : 2);
    // us, 4 / 8 / 16 lanes: 3881 x 1640 bf16 9.6 / 13.1 / 23.1, 1667 x 3840 bf16 6.1 / 5.7 / 8.1, 4096 x 4096 fp32 22.9 / 19.1 / 24.8,
    // 4096 x 16384 fp16 42.6 / 28.1 / 29.1: whole 128-byte lines from the width on that still gives enough workgroups
    const int lanes = row_bytes >= 56 * 128 ? 8 : 4;
    const int64_t blocks = (row_bytes + 16 * lanes - 1) / (16 * lanes);
    NMG_REQUIRE(blocks <= 0x7fffffffLL, NMG_ERR_UNSUPPORTED, "too many columns for one launch");
    hipStream_t s = (hipStream_t)stream;
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(CS_THREADS), 0, s, P); };
    switch (dtype) {
    case NMG_F32: launch(lanes == 4 ? colsum_kernel<float, 4> : colsum_kernel<float, 8>); break;
    case NMG_F16: launch(lanes == 4 ? colsum_kernel<__half, 4> : colsum_kernel<__half, 8>); break;
    default: launch(lanes == 4 ? colsum_kernel<__hip_bfloat16, 4> : colsum_kernel<__hip_bfloat16, 8>); break;
    }
    NMG_HIP_TRY(hipGetLastError());
    return NMG_OK;
}
