// 16-bit matrices into the shape the matrix-core kernels read: rows that start on 16 bytes, a row length and a row
// count rounded up, zeros in between -- in one pass.
//
// The products want whole K steps and 16-byte rows; an extent such as 1001 has neither.  A padded copy of the activations
// costs their size twice in HBM traffic (a few us), against 3 to 8 times the time of the product in the kernels that take
// any shape.  Bound by memory; a source row may start on any 2-byte boundary (global loads of 16 bytes need no
// alignment, they only touch one more line).  1857 x 10385 and its like: 3 us for 512 rows against 14 us for a fill
// and a strided copy.
#include "nmg_common.h"

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
