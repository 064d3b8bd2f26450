// Shared host/device helpers for the nmg HIP library (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#include "../../include/nmg_hip.h"

namespace nmg {

// ---- error reporting (thread-local message, integer status) -------------------------------
void set_error(const char *fmt, ...);
int hip_fail(hipError_t e, const char *what, const char *file, int line);

#define NMG_HIP_TRY(expr)                                                         \
    do {                                                                          \
        hipError_t _e = (expr);                                                   \
        if (_e != hipSuccess) return ::nmg::hip_fail(_e, #expr, __FILE__, __LINE__); \
    } while (0)

#define NMG_REQUIRE(cond, code, ...)     \
    do {                                 \
        if (!(cond)) {                   \
            ::nmg::set_error(__VA_ARGS__); \
            return (code);               \
        }                                \
    } while (0)

// ---- pattern order tables -----------------------------------------------------------------
constexpr int kOrderSlotBytes = 8192;      // largest table: c*n int8 entries of one (n, m) pair
constexpr int kOrderPoolBytes = 64 * 1024;  // all tables of one device, packed 16-byte aligned

int64_t binom(int m, int n);
// Host copy of the table (cached per (n, m)); nullptr when (n, m) is invalid.
const int8_t *host_order(int n, int m);
// Device copy living in this library's file-scope table on the current device; copied there
// with a blocking hipMemcpy the first time an (n, m) pair is used on that device.
int device_order(int n, int m, const int8_t **d_order);
// 256 bytes of zeros on the current device (file-scope array, never written).
int device_zero_page(const void **d_zero);

// Y[T, O] = X[T, K] A[O, K]^T (+ bias[o]) in a 16-bit type, both operands as rows, on 256 x 256 tiles (nmg_densefrag.hip);
// whether that is the faster form for the extents.
bool dense_rows16_pays(int64_t O, int64_t T);
int dense_rows16(const void *d_a, int64_t lda, const void *d_x, int64_t ldx, void *d_y, int64_t ldy, const void *d_bias,
                 int64_t O, int64_t K, int64_t T, int dtype, void *stream);
// Y = X A^T (+ bias) in single precision on the 16-bit matrix cores (nmg_split3.hip; `form` as in gemm_f32_host); false, and nothing
// launched, where it does not take the extents or is not expected to beat `other_us`.
bool split3_gemm(const void *d_a, int64_t lda, const void *d_x, int64_t ldx, void *d_y, int64_t ldy, const void *d_bias, int64_t O,
                 int64_t K, int64_t T, int form, double other_us, hipStream_t st);
// The slices of the reduction with which it is fastest, and its time in us (1e30: extents that it does not take); the product in
// slices, their sums at d_part [slices][T][O up to a multiple of 4].
double split3_plan(int64_t lda, int64_t ldx, int64_t O, int64_t K, int64_t T, int form, int *slices);
int split3_gemm_slices(const void *d_a, int64_t lda, const void *d_x, int64_t ldx, void *d_y, int64_t ldy, const void *d_bias, int64_t O,
                       int64_t K, int64_t T, int form, int slices, float *d_part, hipStream_t st);
// Y[G, S] = L[T, G]^T P[T, S] (+ bias[s]) in a 16-bit type on the matrix cores (nmg_sddmm.hip).
int dense_tn16(const void *d_lines, int64_t ld_lines, const void *d_pos, int64_t ld_pos, int64_t T, int64_t G, int64_t S,
               void *d_y, int64_t ldy, const void *d_bias, int dtype, void *stream);

inline size_t dtype_size(int dtype)
{
    switch (dtype) {
    case NMG_F32: return 4;
    case NMG_F16: return 2;
    case NMG_BF16: return 2;
    case NMG_F64: return 8;
    default: return 0;
    }
}

struct TileGeom {
    int64_t outer;       // number of tiles
    int64_t num_chunks;  // ceil(G / (c*g))
    int64_t num_blocks;  // ceil(S / m)
    int c, cols;         // patterns per tile; columns per tile = c*g
};

inline TileGeom tile_geom(const nmg_view &v, int n, int m, int g)
{
    TileGeom t;
    t.c = (int)binom(m, n);
    t.cols = t.c * g;
    t.num_chunks = (v.G + t.cols - 1) / t.cols;
    t.num_blocks = (v.S + m - 1) / m;
    t.outer = v.batch * t.num_chunks * t.num_blocks;
    return t;
}

// ---- device helpers -------------------------------------------------------------------------
#if defined(__HIPCC__)

// Element <-> fp32 conversions that keep the stored bits exact on the way back.
__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(__half x) { return __half2float(x); }
__device__ __forceinline__ float to_f32(__hip_bfloat16 x) { return __bfloat162float(x); }

// Tile of workgroup `id` of `tiles`: consecutive ids are dealt round-robin to the 8 XCDs, each XCD gets a contiguous run of tiles
// (of tiles / 8, the first tiles % 8 of them one more), which the caller's walk makes a compact block whose operands stay in that
// XCD's L2.  Against leaving counts that are no multiple of 8 in the order of the ids, neighbours on different XCDs, us: 2:4
// 11008 x 4096 x 6000 tokens (2021 tiles) 422 -> 312, 2176 x 4096 x 9000 163 -> 113, 1640 x 1920 x 3500 23.5 -> 18.9; 4:8
// 11008 x 4096 x 6000 484 -> 412; of 242 products of 33 to 1024 tokens the fastest 0.71, the slowest 1.03 of the time (2:4 2304 x 4096
// x 384, four slices of 16 steps, 17.5 -> 18.0).
__device__ __forceinline__ int xcd_run(int id, int tiles)
{
    const int xcd = id & 7;
    return xcd * (tiles >> 3) + min(xcd, tiles & 7) + (id >> 3);
}

template <typename T> struct Zero;
template <> struct Zero<float> { __device__ static float v() { return 0.f; } };
template <> struct Zero<double> { __device__ static double v() { return 0.0; } };
template <> struct Zero<__half> { __device__ static __half v() { return __ushort_as_half((unsigned short)0); } };
template <> struct Zero<__hip_bfloat16> {
    __device__ static __hip_bfloat16 v() { return __float2bfloat16(0.f); }
};

// Compressor for 32-bit scores, m <= 8 and at most 128 patterns (nmg_match.h); *done tells whether it took the shape.
struct ViewDev;
#define NMG_MATCH(name)                                                                                                    \
    int name(const void *dense, void *val, int16_t *idx, const ViewDev &view, int64_t outer, int n, int m, int g, int c, \
             int cols, hipStream_t stream, bool *done)
NMG_MATCH(match_f32);
NMG_MATCH(match_f16);
NMG_MATCH(match_bf16);
#undef NMG_MATCH

// Address of element (group index gi, sparse index si) of batch b in a strided view.
struct ViewDev {
    int64_t G, S, stride_b, stride_g, stride_s;
    int64_t num_chunks, num_blocks;
};

#endif

}  // namespace nmg
