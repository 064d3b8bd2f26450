// Pieces shared by the pipelined matrix-core kernels: vector types, LDS-DMA pointer types and the
// output-tile epilogue.
#pragma once
#include "nmg_common.h"

#include <type_traits>

namespace nmg {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *lds_ptr_t;
typedef const __attribute__((address_space(1))) void *glb_ptr_t;

__device__ __forceinline__ uint16_t f32_to_bits16(float x, __half *) { return __half_as_ushort(__float2half(x)); }
__device__ __forceinline__ uint16_t f32_to_bits16(float x, __hip_bfloat16 *)
{
    __hip_bfloat16 b = __float2bfloat16(x);
    return *reinterpret_cast<uint16_t *>(&b);
}

// Grids of at most one workgroup per CU: all workgroups walk the reduction in step, so that the XCDs that share a weight
// or an activation (2 and 4 of the 8 where the tiles are 16 x 16) ask memory for the same line at the same moment and all
// wait for it.  So every band of output tiles starts b / bands of the reduction further on: of the XCDs that share
// activations the first one to come by brings a line into the memory-side cache and the others find it there.  The start depends
// on the outputs alone, so that an activation row is summed in the same order wherever it stands among the tokens.  Operands
// new in every pass, us, in step -> apart: 4096 x 11008 2:4 fp16 x 2048 tokens 115.4 -> 111.7, x 777 67.5 -> 59.8; its transpose
// on the dense cores x 512 57.5 -> 55.6; 8192 x 4096 x 777 43.8 -> 37.7.  A start for every XCD, an eighth apart, sums equal rows
// differently and is not faster over the range (111.8, 62.4, 55.4, 38.8; the first of them and torch.mm 4096^2 x 2048, timed alone in longer
// runs, 3 and 1.6 % faster: 104.7 against 107.7, 175.8 against 178.6).  Starts of single output tiles 1 to 20 steps apart
// in a band: 111.7 to 129, an XCD's workgroups no longer share lines in its L2; bands of two tiles 112.5, 59.3, 55.1, 37.4.
// Shorter walks put the bands a few steps apart only (21 steps of 64: 39.4 -> 42, 32 steps: 56.8 -> 59);
// operands beyond that cache of 256 MB are gone before the others come by (268 MB, dense cores, 16384 x 4096 transposed x
// 4096: 0.5 to 0.8 % of a training step lost); and with more than one round of workgroups the XCDs drift apart by themselves.
inline bool stagger_bands(unsigned workgroups, int steps, int64_t operand_bytes)
{
    return workgroups <= 256 && steps >= 64 && operand_bytes <= (int64_t)192 << 20;
}

// Where an output tile goes: Y[T, M] row-major with leading dimension ldy.
struct TileOut {
    void *y;
    int64_t M, T, ldy;
};

// A sum starts with its feature's bias (bias[M]; zero without one): single precision, rounded once.  Added behind the
// rounding of the sum, as the epilogues once did, a product is rounded twice (4096^2 4:8 bf16: 2.35e-3 off in 2-norm
// instead of 1.66e-3); added to the sums in the epilogue, in a body with a bias beside one without, the 256 x 256 tiles spill.
// The loads have no branch each, which would make each a round trip to memory; what a feature beyond the last one gets is
// never stored.
template <typename T> __device__ __forceinline__ float bias_of(const void *bias, int64_t f, int64_t M)
{
    return to_f32(((const T *)bias)[f < M ? f : M - 1]);
}

// a lane of the 32 x 32 form holds features 8*(r/4) + 4*(l/32) + r%4 of a block
template <typename T, int FB, int TB>
__device__ __forceinline__ void start_sums(f32x16 (&acc)[FB][TB], const void *bias, int lane, int64_t fw, int64_t M)
{
    float b[FB][16] = {};
    if (bias) {
#pragma unroll
        for (int fb = 0; fb < FB; fb++)
#pragma unroll
            for (int r = 0; r < 16; r++) b[fb][r] = bias_of<T>(bias, fw + fb * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), M);
    }
#pragma unroll
    for (int fb = 0; fb < FB; fb++)
#pragma unroll
        for (int tb = 0; tb < TB; tb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[fb][tb][r] = b[fb][r];
}

// ... and one of the 16 x 16 form features 4*(l/16) + 0..3
template <typename T, int AB, int TB>
__device__ __forceinline__ void start_sums(f32x4 (&acc)[AB][TB], const void *bias, int lane, int64_t fw, int64_t M)
{
    float b[AB][4] = {};
    if (bias) {
#pragma unroll
        for (int ab = 0; ab < AB; ab++)
#pragma unroll
            for (int i = 0; i < 4; i++) b[ab][i] = bias_of<T>(bias, fw + ab * 16 + 4 * (lane >> 4) + i, M);
    }
#pragma unroll
    for (int ab = 0; ab < AB; ab++)
#pragma unroll
        for (int tb = 0; tb < TB; tb++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[ab][tb][i] = b[ab][i];
}

// Epilogue of the pipelined kernels.  D[row = feature][col = token]; a lane holds token
// l%32 and features 8*(r/4) + 4*(l/32) + r%4.  The wavefront's TB*32 tokens x FB*32 features are
// staged through its own LDS region `stg` as [token][feature] so the global stores are 16 B per
// lane and FB*64 B contiguous per token row.  fw / tw = first feature / token of the wavefront.
// The caller guarantees that no load into LDS is pending.
// Second half of the staged epilogues: NROWS token rows of FB*64 B (+16 B pad) lie in `stg`; every
// lane moves 16 B per pass, FB*64 B contiguous per token row.
template <int FB, int NROWS>
__device__ __forceinline__ void store_staged_rows(const unsigned char *stg, int lane, int64_t fw, int64_t tw,
                                                  const TileOut &P)
{
    constexpr int ROW = FB * 64 + 16;       // bytes per staged token row (16 B pad: conflict-free)
    constexpr int CPR = FB * 4;             // 16-byte chunks per row
    constexpr int RPP = 64 / CPR;           // token rows per pass of the wavefront
    uint16_t *Y = (uint16_t *)P.y;
    const bool vec_ok = (P.ldy & 7) == 0 && ((uintptr_t)P.y & 15) == 0;
    const int fc = lane % CPR;                      // 8-feature chunk of the row
    const int64_t f = fw + fc * 8;
#pragma unroll 4
    for (int it = 0; it < NROWS / RPP; it++) {
        const int tl = it * RPP + lane / CPR;
        const int64_t tok = tw + tl;
        const u32x4 v = *(const u32x4 *)(stg + tl * ROW + fc * 16);
        if (tok >= P.T || f >= P.M) continue;
        uint16_t *dst = Y + tok * P.ldy + f;
        if (vec_ok && f + 7 < P.M) {
            *(u32x4 *)dst = v;
        } else {
            uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (f + i < P.M) dst[i] = (uint16_t)(w[i >> 1] >> ((i & 1) * 16));
        }
    }
}

template <typename T, int FB, int TB>
__device__ __forceinline__ void smf_store_tile(const f32x16 (&acc)[FB][TB], unsigned char *stg, int lane,
                                               int64_t fw, int64_t tw, const TileOut &P)
{
    constexpr int ROW = FB * 64 + 16;
    const int j = lane & 31, h = lane >> 5;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int tb = 0; tb < TB; tb++)
#pragma unroll
        for (int fb = 0; fb < FB; fb++)
#pragma unroll
            for (int rq = 0; rq < 4; rq++) {
                uint16_t hh[4];
#pragma unroll
                for (int i = 0; i < 4; i++) hh[i] = f32_to_bits16(acc[fb][tb][rq * 4 + i], (T *)nullptr);
                uint2 pk;
                pk.x = (uint32_t)hh[0] | ((uint32_t)hh[1] << 16);
                pk.y = (uint32_t)hh[2] | ((uint32_t)hh[3] << 16);
                *(uint2 *)(stg + (tb * 32 + j) * ROW + (fb * 32 + rq * 8 + h * 4) * 2) = pk;
            }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    store_staged_rows<FB, TB * 32>(stg, lane, fw, tw, P);
}

// A sum out of its accumulation register, one read where it is used: left to the compiler all of them (256 a lane in
// the 256 x 256 tile) are copied to the other registers at the head of the epilogue, for which some are spilled.
__device__ __forceinline__ float from_acc(float a)
{
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
    return v;
}

// The 16 x 16 form of the instruction: a lane holds token l%16 and outputs 4*(l/16) + 0..3 of every
// 16 x 16 block.  AB blocks of 16 outputs (a multiple of 2) x TB blocks of 16 tokens per wavefront.
template <typename T, int AB, int TB>
__device__ __forceinline__ void store_tile16(const f32x4 (&acc)[AB][TB], unsigned char *stg, int lane,
                                             int64_t fw, int64_t tw, const TileOut &P)
{
    static_assert(AB % 2 == 0, "whole 32-output rows of the staging area");
    constexpr int ROW = AB * 32 + 16;
    const int j = lane & 15, q = lane >> 4;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int tb = 0; tb < TB; tb++) {
#pragma unroll
        for (int ab = 0; ab < AB; ab++) {
            uint16_t hh[4];
#pragma unroll
            for (int i = 0; i < 4; i++) hh[i] = f32_to_bits16(from_acc(acc[ab][tb][i]), (T *)nullptr);
            uint2 pk;
            pk.x = (uint32_t)hh[0] | ((uint32_t)hh[1] << 16);
            pk.y = (uint32_t)hh[2] | ((uint32_t)hh[3] << 16);
            *(uint2 *)(stg + (tb * 16 + j) * ROW + (ab * 16 + q * 4) * 2) = pk;
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    store_staged_rows<AB / 2, TB * 16>(stg, lane, fw, tw, P);
}

// The same epilogue for a transposed output, Y[M, T] row-major (tokens contiguous): the
// wavefront's FB*32 features x TB*32 tokens are staged as [feature][token], so that a lane stores
// 16 bytes = 8 tokens of one feature row and TB*64 bytes per row are contiguous.
// Second half of the transposed epilogues: NROWS output rows of TB*64 B (+16 B pad) lie in `stg`
// as [output][token]; a lane moves 16 bytes = 8 tokens of one output row per pass.
template <int TB, int NROWS>
__device__ __forceinline__ void store_staged_rows_t(const unsigned char *stg, int lane, int64_t fw, int64_t tw,
                                                    const TileOut &P)
{
    constexpr int ROW = TB * 64 + 16;       // bytes per staged feature row
    constexpr int CPR = TB * 4;             // 16-byte chunks per row
    constexpr int RPP = 64 / CPR;           // feature rows per pass of the wavefront
    uint16_t *Y = (uint16_t *)P.y;
    const bool vec_ok = (P.ldy & 7) == 0 && ((uintptr_t)P.y & 15) == 0;
    const int tc = lane % CPR;                      // 8-token chunk of the row
    const int64_t tok = tw + tc * 8;
#pragma unroll 4
    for (int it = 0; it < NROWS / RPP; it++) {
        const int fl = it * RPP + lane / CPR;
        const int64_t f = fw + fl;
        const u32x4 v = *(const u32x4 *)(stg + fl * ROW + tc * 16);
        if (f >= P.M || tok >= P.T) continue;
        uint16_t *dst = Y + f * P.ldy + tok;
        if (vec_ok && tok + 7 < P.T) {
            *(u32x4 *)dst = v;
        } else {
            uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (tok + i < P.T) dst[i] = (uint16_t)(w[i >> 1] >> ((i & 1) * 16));
        }
    }
}

template <typename T, int FB, int TB>
__device__ __forceinline__ void smf_store_tile_t(const f32x16 (&acc)[FB][TB], unsigned char *stg, int lane,
                                                 int64_t fw, int64_t tw, const TileOut &P)
{
    constexpr int ROW = TB * 64 + 16;       // bytes per staged feature row
    const int j = lane & 31, h = lane >> 5;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int tb = 0; tb < TB; tb++)
#pragma unroll
        for (int fb = 0; fb < FB; fb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int f = fb * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                *(uint16_t *)(stg + f * ROW + (tb * 32 + j) * 2) = f32_to_bits16(acc[fb][tb][r], (T *)nullptr);
            }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    store_staged_rows_t<TB, FB * 32>(stg, lane, fw, tw, P);
}

// The 16 x 16 form, transposed output: AB blocks of 16 outputs x TB16 blocks of 16 tokens (an even
// number) per wavefront, staged as [output][token].
template <typename T, int AB, int TB16>
__device__ __forceinline__ void store_tile16_t(const f32x4 (&acc)[AB][TB16], unsigned char *stg, int lane,
                                               int64_t fw, int64_t tw, const TileOut &P)
{
    static_assert(TB16 % 2 == 0, "whole 32-token pieces of a staged row");
    constexpr int ROW = TB16 * 32 + 16;
    const int j = lane & 15, q = lane >> 4;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int tb = 0; tb < TB16; tb++) {
#pragma unroll
        for (int ab = 0; ab < AB; ab++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                *(uint16_t *)(stg + (ab * 16 + q * 4 + r) * ROW + (tb * 16 + j) * 2) =
                    f32_to_bits16(from_acc(acc[ab][tb][r]), (T *)nullptr);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    store_staged_rows_t<TB16 / 2, AB * 16>(stg, lane, fw, tw, P);
}

// ---- reductions cut into slices (products with fewer tiles than the GPU has CUs) ----
// Slice s of a tile stores its sums in single precision at part[s][token][feature] (part_ld
// features per token, a multiple of 256: the padded features of the last tile are stored too);
// splitk_sum_kernel adds the slices in order (+ bias) and rounds once.
struct SplitSum {
    const float *part;
    void *y;
    const void *bias;
    int64_t M, T, ldy, part_ld;
    int slices;
};

// A lane holds token l%32 and features 8*(r/4) + 4*(l/32) + r%4 of every 32 x 32 block: four
// consecutive features are one 16-byte store.  fw / tw = first feature / token of the wavefront.
template <int FB, int TB>
__device__ __forceinline__ void store_partial_tile(const f32x16 (&acc)[FB][TB], float *part, int64_t part_ld,
                                                   int lane, int64_t fw, int64_t tw, int64_t T)
{
    const int j = lane & 31, h = lane >> 5;
#pragma unroll
    for (int tb = 0; tb < TB; tb++) {
        const int64_t tok = tw + tb * 32 + j;
        if (tok >= T) continue;
#pragma unroll
        for (int fb = 0; fb < FB; fb++)
#pragma unroll
            for (int rq = 0; rq < 4; rq++) {
                float4 v;
                v.x = acc[fb][tb][rq * 4 + 0];
                v.y = acc[fb][tb][rq * 4 + 1];
                v.z = acc[fb][tb][rq * 4 + 2];
                v.w = acc[fb][tb][rq * 4 + 3];
                *(float4 *)(part + tok * part_ld + fw + fb * 32 + rq * 8 + h * 4) = v;
            }
    }
}

// The same for the 16 x 16 form: a lane holds token l%16 and outputs 4*(l/16) + 0..3 of every block.
template <int AB, int TB>
__device__ __forceinline__ void store_partial_tile16(const f32x4 (&acc)[AB][TB], float *part, int64_t part_ld,
                                                     int lane, int64_t fw, int64_t tw, int64_t T)
{
    const int j = lane & 15, q = lane >> 4;
#pragma unroll
    for (int tb = 0; tb < TB; tb++) {
        const int64_t tok = tw + tb * 16 + j;
        if (tok >= T) continue;
#pragma unroll
        for (int ab = 0; ab < AB; ab++) {
            float4 v;
            v.x = acc[ab][tb][0];
            v.y = acc[ab][tb][1];
            v.z = acc[ab][tb][2];
            v.w = acc[ab][tb][3];
            *(float4 *)(part + tok * part_ld + fw + ab * 16 + q * 4) = v;
        }
    }
}

// Bound by memory.  A workgroup takes 1024 outputs of one token (no division per thread), a thread four outputs: the
// slices' sums are all requested before the first is added (the kernel is a chain of round trips to memory
// otherwise: the sums were written through other L2s), added in slice order, and stored as one 8-byte word.
// 777 x 4096 in two slices, 32 MB: 10.7 -> 8.0 us against the form
// with a division per thread, sixteen guarded loads whatever the number of slices and 2-byte stores.
template <typename T, int U> __global__ __launch_bounds__(256) void splitk_sum_kernel(SplitSum P)
{
    const uint32_t groups = (uint32_t)((P.M + 1023) / 1024);
    const int64_t tok = blockIdx.x / groups, f = ((int64_t)(blockIdx.x - (uint32_t)tok * groups) * 256 + threadIdx.x) * 4;
    if (f >= P.M) return;
    const float *src = P.part + tok * P.part_ld + f;
    const int64_t step = P.T * P.part_ld;
    float4 sum = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < P.slices; s0 += U) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            v[u] = s0 + u < P.slices ? *(const float4 *)(src + (int64_t)(s0 + u) * step) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; u++) {
            sum.x += v[u].x;
            sum.y += v[u].y;
            sum.z += v[u].z;
            sum.w += v[u].w;
        }
    }
    const float o[4] = {sum.x, sum.y, sum.z, sum.w};
    T *dst = (T *)P.y + tok * P.ldy + f;
    const T *bias = (const T *)P.bias;
    using Bits = std::conditional_t<std::is_same<T, float>::value, float, uint16_t>;
    Bits h[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float total = o[i] + (bias && f + i < P.M ? to_f32(bias[f + i]) : 0.f);
        if constexpr (std::is_same<T, float>::value) h[i] = total;
        else h[i] = f32_to_bits16(total, (T *)nullptr);
    }
    if (f + 4 <= P.M) {
        __builtin_memcpy(dst, h, sizeof(h));
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (f + i < P.M) ((Bits *)dst)[i] = h[i];
    }
}

template <typename T> static inline int launch_splitk_sum(const SplitSum &P, hipStream_t s)
{
    const int64_t blocks = P.T * ((P.M + 1023) / 1024);
    NMG_REQUIRE(blocks <= 0x7fffffffLL, NMG_ERR_UNSUPPORTED, "product too large for one launch");
    const dim3 grid((unsigned)blocks);
    if (P.slices <= 2) hipLaunchKernelGGL((splitk_sum_kernel<T, 2>), grid, dim3(256), 0, s, P);
    else if (P.slices <= 4) hipLaunchKernelGGL((splitk_sum_kernel<T, 4>), grid, dim3(256), 0, s, P);
    else if (P.slices <= 8) hipLaunchKernelGGL((splitk_sum_kernel<T, 8>), grid, dim3(256), 0, s, P);
    else hipLaunchKernelGGL((splitk_sum_kernel<T, 16>), grid, dim3(256), 0, s, P);
    NMG_HIP_TRY(hipGetLastError());
    return NMG_OK;
}

// Largest number of slices <= S that leaves none empty: slices of ceil(KP / S) K steps.
static inline int splitk_fit(int64_t KP, int64_t S)
{
    while (S > 1 && (S - 1) * ((KP + S - 1) / S) >= KP) S--;
    return (int)(S < 1 ? 1 : S);
}

}  // namespace nmg
