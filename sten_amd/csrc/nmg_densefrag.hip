// nmg x dense matmul on the dense matrix cores (V_MFMA_F32_16X16X32_{F16,BF16}) with the weight
// expanded beforehand into the register order of the matrix instructions ("densefrag" operand).
//
// Serves what the sparse matrix cores cannot: patterns that do not fit 2-of-4 groups (4:8,
// 3:4, ...) and the reduction along the *group* dim, i.e. the gradient with respect to the
// activations of a weight that is n:m along its own reduction dim:
//
//   transpose = 0:  Y[tok, q] = sum_s X[tok, s] * W2[q, s]      (q = line, s = sparse position)
//   transpose = 1:  Y[tok, s] = sum_q X[tok, q] * W2[q, s]
//
// Two kernels:
//   densefrag_kernel       rowpack -> densefrag, through an LDS tile (reads and writes contiguous);
//   dense16_direct_kernel  the multiplication, same skeleton as the direct-weights kernel of the
//                          sparse matrix cores: 4 wavefronts stacked on the output dim, weight
//                          fragments global -> registers DD_D K steps ahead, activation tile
//                          global -> LDS by DMA, one barrier per K step of 64.
//
// densefrag [OB][K16][64 lanes][8]: for output block ob (32 outputs) and k-step k16 (16 reduction
// positions), lane l holds the 8 weights of output ob*32 + l%32 at reduction positions
// k16*16 + 8*(l/32) + 0..7 -- the A operand of V_MFMA_F32_32X32X16, which the first form of the
// multiplication used; the 16 x 16 x 32 instruction finds its fragments in it with another lane
// offset (below).  OB is padded to a multiple of 8 (256 outputs), the reduction extent to a
// multiple of 64; padding is zero.
#include "nmg_common.h"
#include "nmg_tile.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace nmg {

typedef _Float16 df_f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 df_bf16x8 __attribute__((ext_vector_type(8)));

// ------------------------------------------------------------------ rowpack -> densefrag
constexpr int DFX_L = 64, DFX_P = 128;   // LDS tile: lines x positions (at most; a tile holds whole blocks)

struct DfExpandParams {
    const void *pk_val;
    const void *pk_pat;
    void *df;
    const int8_t *order;
    int64_t G, S, nb;
    int64_t OB, K16;                      // blocks of the operand
    int n, m, pat_bytes, bpt, transpose;  // bpt = blocks of m positions per tile
    int pt;                               // positions per tile: bpt * m, a multiple of 32, at most 128
    int order_bytes;                      // size of the order table (specialised kernels: it fits 2 KiB)
};

// NV = n where the kernel is specialised for it (1, 2, 4: the n values of a block are one load, 3: three loads; the
// order table sits in LDS, and a thread has the loads of four blocks in flight before it scatters
// the first -- pattern -> order entry -> value is otherwise a chain of round trips per block: 3:6
// 9216 x 4608 fp16 any n -> three 45 -> 36 us, 134 MB),
// 0 = any n.
template <typename T, int NV> __global__ __launch_bounds__(256) void densefrag_kernel(DfExpandParams P)
{
    // transpose = 0: tile[line][position], outputs = lines;  transpose = 1: tile[position][line],
    // outputs = positions.  Rows are outputs, columns the reduction; +8 elements of padding keep
    // rows 16-byte aligned and spread the banks.
    constexpr int PAD = 8;
    __shared__ __align__(16) uint16_t tile[DFX_L * (DFX_P + PAD) > DFX_P * (DFX_L + PAD) ? DFX_L * (DFX_P + PAD)
                                                                                        : DFX_P * (DFX_L + PAD)];
    static_assert(sizeof(T) == 2, "16-bit data");
    const int tid = threadIdx.x;
    const int64_t q0 = (int64_t)blockIdx.y * DFX_L, b0 = (int64_t)blockIdx.x * P.bpt;
    const int rows = P.transpose ? P.pt : DFX_L, cols = P.transpose ? DFX_L : P.pt;
    const int pitch = cols + PAD;
    {
        uint4 z = {0, 0, 0, 0};
        for (int i = tid; i < rows * pitch / 8; i += 256) ((uint4 *)tile)[i] = z;
    }
    __syncthreads();
    const uint16_t *pv = (const uint16_t *)P.pk_val;
    if constexpr (NV > 0) {
        __shared__ int8_t s_ord[2048];
        for (int i = tid; i < P.order_bytes; i += 256) s_ord[i] = P.order[i];
        __syncthreads();
        const int items = DFX_L * P.bpt;
        for (int base = tid; base < items; base += 4 * 256) {
            int pat[4];
            uint16_t v[4][NV];
            bool live[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int i = base + u * 256;
                const int ql = i / P.bpt, bl = i - ql * P.bpt;
                const int64_t q = q0 + ql, b = b0 + bl;
                live[u] = i < items && q < P.G && b < P.nb;
                const int64_t blk = live[u] ? q * P.nb + b : 0;
                pat[u] = P.pat_bytes == 1 ? (int)((const uint8_t *)P.pk_pat)[blk]
                                          : (int)((const uint16_t *)P.pk_pat)[blk];
                if constexpr (NV == 1) {
                    v[u][0] = pv[blk];
                } else if constexpr (NV == 2) {
                    const uint32_t w = ((const uint32_t *)pv)[blk];
                    v[u][0] = (uint16_t)w;
                    v[u][1] = (uint16_t)(w >> 16);
                } else if constexpr (NV == 3) {
#pragma unroll
                    for (int j = 0; j < 3; j++) v[u][j] = pv[blk * 3 + j];
                } else {
                    const uint2 w = ((const uint2 *)pv)[blk];
                    v[u][0] = (uint16_t)w.x;
                    v[u][1] = (uint16_t)(w.x >> 16);
                    v[u][2] = (uint16_t)w.y;
                    v[u][3] = (uint16_t)(w.y >> 16);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (!live[u]) continue;
                const int i = base + u * 256;
                const int ql = i / P.bpt, bl = i - ql * P.bpt;
                const int8_t *ord = s_ord + pat[u] * NV;
#pragma unroll
                for (int j = 0; j < NV; j++) {
                    const int pos = bl * P.m + ord[j];
                    if (P.transpose)
                        tile[pos * pitch + ql] = v[u][j];
                    else
                        tile[ql * pitch + pos] = v[u][j];
                }
            }
        }
    } else {
        for (int i = tid; i < DFX_L * P.bpt; i += 256) {
            const int ql = i / P.bpt, bl = i - ql * P.bpt;
            const int64_t q = q0 + ql, b = b0 + bl;
            if (q >= P.G || b >= P.nb) continue;
            const int64_t blk = q * P.nb + b;
            const int pat = P.pat_bytes == 1 ? (int)((const uint8_t *)P.pk_pat)[blk]
                                             : (int)((const uint16_t *)P.pk_pat)[blk];
            const int8_t *ord = P.order + pat * P.n;
            for (int j = 0; j < P.n; j++) {
                const int pos = bl * P.m + ord[j];
                const uint16_t v = pv[blk * P.n + j];
                if (P.transpose)
                    tile[pos * pitch + ql] = v;
                else
                    tile[ql * pitch + pos] = v;
            }
        }
    }
    __syncthreads();
    // tile -> fragments: (rows/32) x (cols/16) fragments of 64 lanes x 16 B
    const int64_t ob0 = (P.transpose ? b0 * P.m : q0) / 32, k0 = (P.transpose ? q0 : b0 * P.m) / 16;
    const int nfk = cols / 16, nfrag = (rows / 32) * nfk;
    uint4 *df = (uint4 *)P.df;
    for (int i = tid; i < nfrag * 64; i += 256) {
        const int f = i >> 6, l = i & 63;
        const int fo = f / nfk, fk = f - fo * nfk;
        const int64_t ob = ob0 + fo, k16 = k0 + fk;
        if (ob >= P.OB || k16 >= P.K16) continue;
        const uint4 v = *(const uint4 *)(tile + (fo * 32 + (l & 31)) * pitch + fk * 16 + 8 * (l >> 5));
        df[(ob * P.K16 + k16) * 64 + l] = v;
    }
}

// ----------------------------------------------------------------------------- the matmul
struct DfParams {
    const void *df;
    const void *x;
    void *y;
    const void *bias;
    int64_t O, K, T, ldx, ldy;
    int64_t lda;         // ROWA: row pitch of the weight, in elements
    int KP;              // K steps of 64
    int tiles_m, tiles_n;
    int turn;            // band b of the tiles starts its walk of the reduction b / bands of the way in
    bool in_order;       // a tile asked for by number: sums in the order of the reduction, alike for every tile
    // reduction cut into slices (0 / 1: whole): slice s of a tile stores its sums in single
    // precision at part[s][token][output], part_ld outputs per token
    int ksplit;
    float *part;
    int64_t part_ld;
    int tail;            // reduction positions of the last K step where they are fewer than 64 (multiple of 8), else 0
};

// K steps in flight and activation stages in LDS (>= steps + 1), by the blocks of 16 outputs of a wavefront: a step of four blocks takes
// twice the MFMA time of one of two, and that of a sparse step
constexpr int dd_steps(int ab) { return ab == 4 ? 2 : 4; }
constexpr int dd_stages(int ab) { return ab == 4 ? 4 : 8; }

// V_MFMA_F32_16X16X32: of the two dense forms of the instruction the one that draws less power
// per flop (from registers, random operands: 1.76-1.97 against 1.61-1.71 PFLOP/s for 32 x 32 x 16),
// and with this skeleton around it the difference stays: the first form of this kernel, on
// 32 x 32 x 16, reached matrix-pipe utilisation 0.90 and was 9-15 % slower.
//   A fragment (16 outputs x 32 k): lane (r = l%16, kq = l/16) wants the 8 weights of output
//     16*ab + r at k = 32*k32 + 8*kq + 0..7, which the densefrag operand stores in fragment
//     (ob = ab/2, k16 = 2*k32 + kq/2) at lane 32*(kq%2) + 16*(ab%2) + r: a load still covers four
//     runs of 256 contiguous bytes.
//   B fragment (16 tokens x 32 k): lane (j = l%16, kq) reads the 16-byte chunk 4*k32 + kq of token
//     row 16*tb + j; with the chunks XOR-swizzled by (row/2)%8 sixteen consecutive rows cover all
//     banks.
//   D: lane holds token l%16, outputs 4*(l/16) + 0..3 of the 16 x 16 block.
// A wavefront owns 64 outputs x TB*16 tokens: 4 x TB accumulator blocks of 4 registers, all of
// them in the accumulation registers.  A K step of 64 is two k-steps of 32; a phase is one
// (k-step, token part) pair of 4 * TB / NH MFMAs: they run while the activation fragments of the
// next phase are read from LDS, and the loads of K step kp+DD_D are dealt out over the phases.
// XT = true is the product with both dense operands transposed, C[O, T] = A * B for B [K, T] (the
// gradient with respect to B of torch.mm(W, B): W^T * grad_out as they lie in memory): the
// activation tile of a K step is then 64 reduction rows x TT tokens, fetched as it lies, an
// activation fragment is two LDS transpose reads (DS_READ_B64_TR_B16), and the epilogue stages
// [output][token] and stores token-contiguous rows.
template <typename T> struct DfMma16;
template <> struct DfMma16<__half> {
    using F = df_f16x8;
    __device__ static f32x4 run(F a, F b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <> struct DfMma16<__hip_bfloat16> {
    using F = df_bf16x8;
    __device__ static f32x4 run(F a, F b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};

// ROWA = true takes the weight as rows in memory, A [O, K] with pitch lda, in place of the fragment order: a
// lane's 16 bytes are those of its output row at the lane's reduction positions, a load touches 64 bytes of 16 rows
// (the two loads of a K step the two halves of a 128-byte line).  Both operands of Y = X A^T as they lie.
// CT = true stores the result transposed, C [O, T].
// TAIL = true takes a last K step of fewer than 64 positions (in the other form it cost a product of one round 1 %).
template <typename T, int TB, int NH, bool XT = false, bool CT = XT, bool ROWA = false, int AB = 4, bool TAIL = false>
__global__ __launch_bounds__(256, 1) void dense16_direct_kernel(DfParams P)
{
    using Mm = DfMma16<T>;
    constexpr int DD_D = dd_steps(AB), DD_NS = dd_stages(AB);
    constexpr int TF = 64 * AB, TT = TB * 16;                 // workgroup tile: outputs x tokens
    constexpr int STAGE = TT * 128;                       // activation bytes per K step
    constexpr int XL = TT / 32;                           // DMA loads per wavefront per K step
    constexpr int OPS = XL + 2 * AB;                      // memory operations per wavefront per K step
    constexpr int BT = TB / NH;                           // token blocks per phase
    constexpr int NP = 2 * NH;                            // phases per K step
    constexpr int NM = AB * BT;                           // MFMAs per phase
    static_assert(TB % NH == 0, "token blocks split evenly into phases");
    static_assert(OPS * DD_D < 64, "vmcnt is a 6-bit counter");
    static_assert(NP >= 2 && NP % 2 == 0, "fragment sets alternate by phase across K steps");
    extern __shared__ __align__(16) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // Workgroup -> tile: consecutive ids are dealt round-robin to the 8 XCDs; give each XCD a
    // contiguous run of ids and walk the grid in bands of 4 output tiles, so that a run covers
    // a compact block of tiles whose weights and activations stay in that XCD's L2.
    int id = blockIdx.x;
    const int ntiles = P.tiles_m * P.tiles_n;
    // Slices of the reduction: an XCD's run goes over slices and tiles, so that few XCDs fetch the same operands (us, weights from memory,
    // against runs of tiles within every slice: 2:4 4096 x 11008 x 200 tokens 34.3 -> 33.2, 1024 x 16384 x 777 38.7 -> 35.4; 4:8 x 300 30.4 -> 27.8);
    // but in short slices an XCD's workgroups wait for the same lines (2:4 2048 x 8192 x 128, 16 steps a slice, 17.3 -> 19.3).
    const int kp_per = P.ksplit > 1 ? (P.KP + P.ksplit - 1) / P.ksplit : P.KP;
    int slice = 0;
    if (kp_per >= 20) {
        id = xcd_run(id, gridDim.x);
        if (P.ksplit > 1) slice = id / ntiles;
        id -= slice * ntiles;
    } else {
        if (P.ksplit > 1) slice = id / ntiles;
        id = xcd_run(id - slice * ntiles, ntiles);
    }
    constexpr int GH = 4;
    const int band = id / (GH * P.tiles_n);
    const int band_h = min(P.tiles_m - band * GH, GH);
    const int in_band = id - band * GH * P.tiles_n;
    const int tile_m = band * GH + in_band % band_h, tile_n = in_band / band_h;
    const int64_t f0 = (int64_t)tile_m * TF, t0 = (int64_t)tile_n * TT;
    // K steps kp_lo .. kp_lo + KP - 1 of the operand's KPT (the host leaves no slice empty)
    const int KPT = P.KP;
    const int kp_lo = slice * kp_per;
    const int KP = min(KPT, kp_lo + kp_per) - kp_lo;
    // A last step of fewer than 64 positions (P.tail) is the walk's first, where the pieces behind the row's end, fetched from its
    // start instead, are overwritten with zeros before anybody reads them; the walk then goes round the KW whole steps.
    const int tail = TAIL && kp_lo + KP == KPT ? P.tail : 0, KW = KP - (tail != 0 ? 1 : 0);
    const int first = P.turn ? band * KW / ((P.tiles_m + GH - 1) / GH) : 0;
    const int ob0 = (int)(f0 / 32) + wave * (AB / 2);

    const unsigned char *av_base[AB / 2];
#pragma unroll
    for (int o = 0; o < AB / 2; o++)
        av_base[o] = (const unsigned char *)P.df +
                     (ROWA ? (int64_t)kp_lo * 128 : (((int64_t)(ob0 + o) * KPT + kp_lo) * 4) * 1024);
    const int r16 = lane & 15, kq = lane >> 4;
    const uint32_t lane_a = (uint32_t)((kq >> 1) * 1024 + ((kq & 1) * 32 + r16) * 16);
    uint32_t row_a[ROWA ? AB : 1];
    if constexpr (ROWA) {
#pragma unroll
        for (int ab = 0; ab < AB; ab++) {
            int64_t row = f0 + wave * (16 * AB) + ab * 16 + r16;
            if (row >= P.O) row = P.O - 1;            // clamped rows are computed, never stored
            row_a[ab] = (uint32_t)(row * P.lda * 2 + kq * 16);
        }
    }
    // K step kp of the activations starts kp * XSTEP bytes into the operand
    const int64_t XSTEP = XT ? 64 * P.ldx * 2 : 128;
    const unsigned char *x_base = (const unsigned char *)P.x + (int64_t)kp_lo * XSTEP;
    uint32_t x_off[XL];
    int x_piece[XL];
#pragma unroll
    for (int i = 0; i < XL; i++) {
        if constexpr (XT) {
            // a DMA load fills 1 KiB = 1024 / (TT * 2) reduction rows of the tile; piece p (8 tokens)
            // of row k holds the logical chunk p ^ (4*(k%4) + 2*((k/8)%2)): the 32 lanes of a
            // transpose read that are served together take rows k .. k+3 and k+8 .. k+11 of one
            // 16-token block, which then fall into 16 different pieces = every bank once
            constexpr int PPR = TT / 8;                       // 16-byte pieces per row
            const int row = (wave * XL + i) * (64 / PPR) + lane / PPR;
            const int chunk = (lane % PPR) ^ (((row & 3) << 2) | (((row >> 3) & 1) << 1));
            int64_t tok = t0 + chunk * 8;
            if (tok > P.T - 8) tok = (P.T - 1) / 8 * 8;       // clamped columns are computed, never stored
            x_off[i] = (uint32_t)((row * P.ldx + tok) * 2);
        } else {
            const int row = (wave * XL + i) * 8 + (lane >> 3);
            const int piece = lane & 7;
            const int q = piece ^ ((row >> 1) & 7);   // logical 16-byte chunk stored at this piece
            int64_t tok = t0 + row;
            if (tok >= P.T) tok = P.T - 1;            // clamped rows are computed, never stored
            x_piece[i] = q;
            x_off[i] = (uint32_t)((tok * P.ldx + (tail != 0 && q * 8 >= tail ? 0 : q * 8)) * 2);
        }
    }

    struct WSet {
        u32x4 a[AB][2];   // [block of 16 outputs][k-step of 32]
    };
    WSet ws[DD_D + 1];
    // load number i (0 .. OPS-1) of the walk's K step kp, step `at` of the operands: first the XL activation DMA loads, then
    // the 2 * AB weight fragments.  Steps beyond the last fetch the last one again: the operation count stays uniform, the
    // data is unused.
    int at = tail != 0 ? KP - 1 : first;
    auto advance = [&](int kp) {      // after the loads of step kp
        const int after = at + 1 == KW ? 0 : at + 1;      // (selects: no branch between the hand-tracked loads)
        at = kp + 1 < KP ? after : at;
    };
    auto issue_one = [&](int kp, WSet &w, int i) {
        if (i < XL) {
            unsigned char *base = smem + (kp & (DD_NS - 1)) * STAGE;
            const unsigned char *xb = x_base + (int64_t)at * XSTEP;
#pragma unroll
            for (int q = 0; q < XL; q++)
                if (q == i) {
                    // (XT: left visible, the compiler makes the transposing reads of every step wait for all loads in flight)
                    if constexpr (XT)
                        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                                     :: "v"(x_off[q]), "s"(xb), "s"((uint32_t)(uintptr_t)(lds_ptr_t)(base + (wave * XL + q) * 1024)) : "memory", "m0");
                    else
                        __builtin_amdgcn_global_load_lds((glb_ptr_t)(xb + x_off[q]),
                                                         (lds_ptr_t)(base + (wave * XL + q) * 1024), 16, 0, 0);
                }
        } else {
            // Written as instructions so that their completion is tracked by the explicit vmcnt
            // waits below and by nothing else.
#pragma unroll
            for (int ab = 0; ab < AB; ab++)
#pragma unroll
                for (int k32 = 0; k32 < 2; k32++)
                    if (XL + ab * 2 + k32 == i) {
                        const unsigned char *av = av_base[ab >> 1] + (int64_t)at * (ROWA ? 128 : 4096);
                        asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3"
                                     : "=v"(w.a[ab][k32])
                                     : "v"(ROWA ? row_a[ROWA ? ab : 0] : lane_a), "s"(av),
                                       "n"(ROWA ? k32 * 64 : k32 * 2048 + (ab & 1) * 256)
                                     : "memory");
                    }
        }
    };

    f32x4 acc[AB][TB];
    start_sums<T>(acc, P.ksplit > 1 ? nullptr : P.bias, lane, f0 + wave * (16 * AB), P.O);   // (slices: the sum adds it)
    auto pin_acc = [&]() {
#pragma unroll
        for (int i = 0; i < AB; i++)
#pragma unroll
            for (int t = 0; t < TB; t++) asm volatile("" : "+a"(acc[i][t]));
    };
    pin_acc();

    const int sw = (r16 >> 1) & 7;
    int b_off[2];
#pragma unroll
    for (int k32 = 0; k32 < 2; k32++) b_off[k32] = r16 * 128 + (((k32 * 4 + kq) ^ sw) << 4);

    struct BFrags {
        u32x4 b[BT];
    };
    BFrags fr[2];
    // XT: lane (kq, i) of a transpose read supplies the 8 bytes at reduction row 8 kq + i/4 (+ 32 k32
    // + 4 r), tokens 4 (i%4) .. +3 of the 16-token block, and receives token i at rows
    // 8 kq + 4 r + 0..3: reads r = 0, 1 are the lane's 8 reduction positions.
    int t_off[XT ? TB : 1];
    if constexpr (XT) {
        const int a = r16 >> 2;
#pragma unroll
        for (int tb = 0; tb < TB; tb++) {
            const int chunk = tb * 2 + ((r16 & 3) >> 1);   // 8-token chunk of the row
            t_off[tb] = (8 * kq + a) * (TT * 2) + ((chunk ^ ((a << 2) | ((kq & 1) << 1))) << 4) + (r16 & 1) * 8;
        }
    }
    auto read_one = [&](BFrags &f, const unsigned char *base, int ph, int t) {
        const int k32 = ph / NH, hh = ph % NH;
        if constexpr (XT) {
            typedef short i16x4 __attribute__((ext_vector_type(4)));
            typedef __attribute__((address_space(3))) i16x4 *lds_i16x4;
            union {
                i16x4 h[2];
                u32x4 u;
            } c;
#pragma unroll
            for (int r = 0; r < 2; r++)
                c.h[r] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_i16x4)(base + t_off[hh * BT + t] + (32 * k32 + 4 * r) * (TT * 2)));
            f.b[t] = c.u;
        } else {
            f.b[t] = *(const u32x4 *)(base + b_off[k32] + (hh * BT + t) * 16 * 128);
        }
    };
    // MFMA number i of phase PH (i = ab * BT + t)
    auto mma = [&](const WSet &w, const BFrags &f, auto ph_tag, int i) {
        constexpr int PH = decltype(ph_tag)::value, K32 = PH / NH, HH = PH % NH;
        const int ab = i / BT, t = i % BT;
        union {
            u32x4 u;
            typename Mm::F v;
        } ca, cb;
        ca.u = w.a[ab][K32];
        cb.u = f.b[t];
        acc[ab][HH * BT + t] = Mm::run(ca.v, cb.v, acc[ab][HH * BT + t]);
    };

    // The counted wait.  Invariants it rests on:
    //  (1) a wavefront's vector memory operations complete in issue order, and it issues exactly
    //      OPS of them per K step (XL DMA loads, then 2 * AB weight fragments), all of step
    //      kp+DD_D before the wait in the last phase of step kp; so at that wait the newest
    //      (DD_D-1) * OPS operations are the steps kp+2 .. kp+DD_D and everything older -- step
    //      kp+1 -- has landed once the counter is down to (DD_D-1) * OPS.  The barrier after it
    //      makes that true for the DMA loads of the other wavefronts too.
    //  (2) the weight set of step kp+1 is passed through the wait as in/out operands: whatever
    //      uses those registers afterwards is ordered after the wait by the compiler as well.
    //      (What it does with them *before* the wait is checked on the compiled code: no
    //      instruction may touch a register with a load in flight, `python -m sten_amd.isa_check`.)
    //  (3) LDS stage (kp+DD_D) % DD_NS is refilled during step kp; its last readers were the
    //      fragment reads of step kp+DD_D-DD_NS <= kp-2, complete (lgkmcnt(0), same wait) before
    //      the barrier that ended that step.  The two fragment sets alternate by phase; NP is
    //      even, so the set read after the barrier (for phase 0 of the next step) is set 0.
    static_assert(DD_NS > DD_D, "a stage must not be refilled while the step that reads it is in flight");
    static_assert(AB == 2 || AB == 4, "the waits list the registers of two or four blocks");
    auto landed = [&](WSet &w) {
        if constexpr (AB == 4)
            asm volatile("s_waitcnt vmcnt(%8) lgkmcnt(0)"
                         : "+v"(w.a[0][0]), "+v"(w.a[0][1]), "+v"(w.a[1][0]), "+v"(w.a[1][1]),
                           "+v"(w.a[AB - 2][0]), "+v"(w.a[AB - 2][1]), "+v"(w.a[AB - 1][0]), "+v"(w.a[AB - 1][1])
                         : "n"((DD_D - 1) * OPS)
                         : "memory");
        else
            asm volatile("s_waitcnt vmcnt(%4) lgkmcnt(0)"
                         : "+v"(w.a[0][0]), "+v"(w.a[0][1]), "+v"(w.a[1][0]), "+v"(w.a[1][1])
                         : "n"((DD_D - 1) * OPS)
                         : "memory");
    };

    // prologue: steps 0 .. DD_D-1 in flight, then wait for step 0
#pragma unroll
    for (int st = 0; st < DD_D; st++) {
#pragma unroll
        for (int i = 0; i < OPS; i++) issue_one(st, ws[st], i);
        advance(st);
        if (TAIL && st == 0) {
            at = tail != 0 && KP > 1 ? first : at;
#pragma unroll
            for (int i = 0; i < XL; i++) x_off[i] += tail != 0 && KP > 1 && x_piece[i] * 8 >= tail ? x_piece[i] * 16 : 0;
        }
    }
    landed(ws[0]);
    if (TAIL && tail != 0) {
#pragma unroll
        for (int i = 0; i < XL; i++)
            if (x_piece[i] * 8 >= tail) *(u32x4 *)(smem + (wave * XL + i) * 1024 + lane * 16) = u32x4{0, 0, 0, 0};
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int t = 0; t < BT; t++) read_one(fr[0], smem, 0, t);

    // The transposed form on narrow tiles has whole turns of the ring in a loop of their own: with the exits inside, the compiler lays its
    // steps out in an order that the check of the loads in flight does not follow.
    int kp0 = 0;
#pragma unroll
    for (int part = XT && AB == 2 ? 0 : 1; part < 2; part++)
    for (; part != 0 ? kp0 < KP : kp0 + DD_D < KP; kp0 += DD_D + 1) {
#pragma unroll
        for (int u = 0; u <= DD_D; u++) {
            const int kp = kp0 + u;
            if (part != 0 && kp >= KP) goto walked;      // (past the loop: a break would be tested again there)
            const unsigned char *base = smem + (kp & (DD_NS - 1)) * STAGE;
            const unsigned char *next = smem + ((kp + 1) & (DD_NS - 1)) * STAGE;
            // A phase: its MFMAs, and behind one MFMA each the fragment reads of the next phase and
            // this phase's share of the loads of step kp+DD_D (dealt out over all phases but the
            // last).  The last phase waits for step kp+1 after two MFMAs, meets the other
            // wavefronts and reads the first fragments of the next stage behind the rest.
            auto phase = [&](auto ph_tag) {
                constexpr int PH = decltype(ph_tag)::value;
                if constexpr (PH == NP - 1) {
                    advance(kp + DD_D);
                    mma(ws[u], fr[PH % 2], ph_tag, 0);
                    mma(ws[u], fr[PH % 2], ph_tag, 1);
                    __builtin_amdgcn_sched_barrier(0);
                    landed(ws[(u + 1) % (DD_D + 1)]);
                    asm volatile("s_barrier" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                    constexpr int SP = (NM - 2) / BT;
#pragma unroll
                    for (int i = 2; i < NM; i++) {
                        mma(ws[u], fr[PH % 2], ph_tag, i);
                        __builtin_amdgcn_sched_barrier(0);
                        if ((i - 2) % SP == 0 && (i - 2) / SP < BT) read_one(fr[(PH + 1) % 2], next, 0, (i - 2) / SP);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
                    constexpr int L0 = PH * OPS / (NP - 1), L1 = (PH + 1) * OPS / (NP - 1);
                    constexpr int NOPS = BT + L1 - L0;
                    constexpr int SP = NM / NOPS > 0 ? NM / NOPS : 1;
                    static_assert(NOPS <= NM, "one memory instruction behind one MFMA");
#pragma unroll
                    for (int i = 0; i < NM; i++) {
                        mma(ws[u], fr[PH % 2], ph_tag, i);
                        __builtin_amdgcn_sched_barrier(0);
                        if (i % SP == 0 && i / SP < NOPS) {
                            const int op = i / SP;
                            if (op < BT)
                                read_one(fr[(PH + 1) % 2], base, PH + 1, op);
                            else
                                issue_one(kp + DD_D, ws[(u + DD_D) % (DD_D + 1)], L0 + op - BT);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            };
            phase(std::integral_constant<int, 0>{});
            phase(std::integral_constant<int, 1>{});
            if constexpr (NP >= 4) {
                phase(std::integral_constant<int, 2>{});
                phase(std::integral_constant<int, 3>{});
            }
            if constexpr (NP >= 8) {
                phase(std::integral_constant<int, 4>{});
                phase(std::integral_constant<int, 5>{});
                phase(std::integral_constant<int, 6>{});
                phase(std::integral_constant<int, 7>{});
            }
            static_assert(NP == 2 || NP == 4 || NP == 8, "one, two or four token parts");
        }
    }
walked:
    pin_acc();
    // The loads of the steps beyond the last are still in flight and nothing reads what they bring:
    // every register of the ring passes through the final wait.
    if constexpr (AB == 4) {
        static_assert(AB != 4 || DD_D == 2, "the final wait lists three weight sets");
        asm volatile("s_waitcnt vmcnt(0)"
                     : "+v"(ws[0].a[0][0]), "+v"(ws[0].a[0][1]), "+v"(ws[0].a[1][0]), "+v"(ws[0].a[1][1]),
                       "+v"(ws[0].a[AB - 2][0]), "+v"(ws[0].a[AB - 2][1]), "+v"(ws[0].a[AB - 1][0]), "+v"(ws[0].a[AB - 1][1]),
                       "+v"(ws[1].a[0][0]), "+v"(ws[1].a[0][1]), "+v"(ws[1].a[1][0]), "+v"(ws[1].a[1][1]),
                       "+v"(ws[1].a[AB - 2][0]), "+v"(ws[1].a[AB - 2][1]), "+v"(ws[1].a[AB - 1][0]), "+v"(ws[1].a[AB - 1][1]),
                       "+v"(ws[2].a[0][0]), "+v"(ws[2].a[0][1]), "+v"(ws[2].a[1][0]), "+v"(ws[2].a[1][1]),
                       "+v"(ws[2].a[AB - 2][0]), "+v"(ws[2].a[AB - 2][1]), "+v"(ws[2].a[AB - 1][0]), "+v"(ws[2].a[AB - 1][1])
                     :
                     : "memory");
    } else {
#pragma unroll
        for (int st = 0; st <= DD_D; st++) {
            WSet &w = ws[st];
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(w.a[0][0]), "+v"(w.a[0][1]), "+v"(w.a[1][0]), "+v"(w.a[1][1]) : : "memory");
        }
    }
    // (no-ops: the compiler does not see that `from_acc` reads what a product may just have written)
    asm volatile("s_barrier\n\ts_nop 15" ::: "memory");
    if (P.ksplit > 1) {
        store_partial_tile16<AB, TB>(acc, P.part + (int64_t)slice * P.T * P.part_ld, P.part_ld, lane,
                                     f0 + wave * (16 * AB), t0, P.T);
        return;
    }
    const TileOut out{P.y, P.O, P.T, P.ldy};
    if constexpr (CT)
        store_tile16_t<T, AB, TB>(acc, smem + wave * (AB * 16 * (TT * 2 + 16)), lane, f0 + wave * (16 * AB), t0, out);
    else
        store_tile16<T, AB, TB>(acc, smem + wave * (TT * (AB * 32 + 16)), lane, f0 + wave * (16 * AB), t0, out);
}

template <typename T, int TB, int NH, bool XT = false, bool CT = XT, bool ROWA = false, int AB = 4> static int launch_dense16(DfParams &P, hipStream_t s)
{
    constexpr int TT = TB * 16;
    P.tiles_m = (int)((P.O + 64 * AB - 1) / (64 * AB));
    P.tiles_n = (int)((P.T + TT - 1) / TT);
    const int slices = P.ksplit > 1 ? P.ksplit : 1;
    dim3 grid((unsigned)(P.tiles_m * P.tiles_n * slices));
    P.turn = !P.in_order && stagger_bands(grid.x, P.KP / slices, P.KP * (P.O + P.T) * 128) ? 1 : 0;
    constexpr size_t ring = (size_t)dd_stages(AB) * TT * 128;
    constexpr size_t stg = CT ? (size_t)4 * 16 * AB * (TT * 2 + 16) : (size_t)4 * TT * (AB * 32 + 16);
    constexpr size_t lds = ring > stg ? ring : stg;
    static_assert(lds <= 160 * 1024, "LDS");
    auto k = dense16_direct_kernel<T, TB, NH, XT, CT, ROWA, AB>;
    if constexpr (!CT && !ROWA)
        if (P.tail != 0) k = dense16_direct_kernel<T, TB, NH, XT, CT, ROWA, AB, true>;
    NMG_HIP_TRY(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k, grid, dim3(256), lds, s, P);
    NMG_HIP_TRY(hipGetLastError());
    if (slices > 1) {
        const SplitSum Q{P.part, P.y, P.bias, P.O, P.T, P.ldy, P.part_ld, slices};
        return launch_splitk_sum<T>(Q, s);
    }
    return NMG_OK;
}

// Few tokens: 16 AB outputs x 16 TB tokens a workgroup, the K steps dealt out to its 16 wavefronts, operands from memory into
// registers, sums added through LDS, rounded once.  One kernel without partial sums in memory, and a reduction that is any
// multiple of 8: the operand holds zeros behind it, the activations' pieces there are not read.
template <typename T, int AB, int TB> __global__ __launch_bounds__(1024) void dense16_few_kernel(DfParams P)
{
    using Mm = DfMma16<T>;
    constexpr int W = 16, AHEAD = AB * TB > 2 ? 2 : AB + TB > 2 ? 3 : 4;      // wavefronts; K steps on their way
    __shared__ __align__(16) f32x4 red[W][AB * TB][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int64_t ob = (int64_t)blockIdx.x * AB, t0 = (int64_t)blockIdx.y * 16 * TB;
    const unsigned char *a[AB], *x[TB];
#pragma unroll
    for (int i = 0; i < AB; i++)
        a[i] = (const unsigned char *)P.df + ((ob + i) >> 1) * P.KP * 4096 + ((ob + i) & 1) * 256 + (kq >> 1) * 1024 + ((kq & 1) * 32 + r16) * 16;
#pragma unroll
    for (int i = 0; i < TB; i++)      // clamped rows are computed, never stored
        x[i] = (const unsigned char *)P.x + (min(t0 + i * 16 + r16, P.T - 1) * P.ldx + kq * 8) * 2;
    struct Step { u32x4 a[AB][2], x[TB][2]; };
    auto fetch = [&](Step &S, int s) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
#pragma unroll
            for (int i = 0; i < AB; i++) S.a[i][k] = *(const u32x4 *)(a[i] + (int64_t)s * 4096 + k * 2048);
            const bool in = (int64_t)s * 64 + k * 32 + kq * 8 < P.K;
#pragma unroll
            for (int i = 0; i < TB; i++) {
                S.x[i][k] = u32x4{0, 0, 0, 0};
                if (in) S.x[i][k] = *(const u32x4 *)(x[i] + (int64_t)s * 128 + k * 64);
            }
        }
    };
    f32x4 acc[AB][TB];
#pragma unroll
    for (int i = 0; i < AB; i++)
#pragma unroll
        for (int t = 0; t < TB; t++) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = wave; s0 < P.KP; s0 += W * AHEAD) {
        Step S[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; u++)
            if (s0 + u * W < P.KP) fetch(S[u], s0 + u * W);
#pragma unroll
        for (int u = 0; u < AHEAD; u++)
            if (s0 + u * W < P.KP)
#pragma unroll
                for (int k = 0; k < 2; k++)
#pragma unroll
                    for (int i = 0; i < AB; i++)
#pragma unroll
                        for (int t = 0; t < TB; t++)
                            acc[i][t] = Mm::run(__builtin_bit_cast(typename Mm::F, S[u].a[i][k]), __builtin_bit_cast(typename Mm::F, S[u].x[t][k]), acc[i][t]);
    }
#pragma unroll
    for (int i = 0; i < AB; i++)
#pragma unroll
        for (int t = 0; t < TB; t++) red[wave][i * TB + t][lane] = acc[i][t];
    __syncthreads();
    if (wave >= AB * TB) return;
    f32x4 sum = red[0][wave][lane];
#pragma unroll
    for (int w = 1; w < W; w++) sum += red[w][wave][lane];
    // a lane holds token r16, outputs 4 kq .. 4 kq + 3 of a block
    const int64_t o = (ob + wave / TB) * 16 + kq * 4, t = t0 + (wave % TB) * 16 + r16;
    if (t >= P.T) return;
    uint16_t *const y = (uint16_t *)P.y + t * P.ldy + o;
    uint16_t h[4];
#pragma unroll
    for (int e = 0; e < 4; e++) h[e] = f32_to_bits16(sum[e] + (P.bias ? bias_of<T>(P.bias, o + e, P.O) : 0.f), (T *)nullptr);
    if (o + 4 <= P.O && ((uintptr_t)y & 7) == 0) {
        *(uint2 *)y = uint2{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (o + e < P.O) y[e] = h[e];
    }
}

// Tiles of the kernel for few tokens, {blocks of 16 outputs, of 16 tokens}: a larger one reads less of the activations, a smaller one
// leaves fewer CUs idle.
static const struct { int ab, tb; } kFewTiles[] = {{1, 1}, {2, 1}, {4, 1}, {2, 2}};

// Its time in us: a CU takes 46 KB of operands a microsecond, the weight comes from memory at 5.1 TB/s.  Fitted to 13 weights of 512 x
// 1024 to 8192^2 with 1 to 48 tokens; the tile that it chooses is 0.5 % behind the best one in the mean.
static double few_cost(int c, int64_t O, int64_t K, int64_t T)
{
    const int ab = kFewTiles[c].ab, tb = kFewTiles[c].tb;
    const int64_t steps = (K + 63) / 64, groups = ((O + 16 * ab - 1) / (16 * ab)) * ((T + 16 * tb - 1) / (16 * tb));
    const double rows = T < 16 * tb ? (double)T / (16 * tb) : 1.0;      // (a lane beyond the last token reads what the last one reads)
    const double walk = (double)((groups + 255) / 256) * (double)steps * 2.048 * (ab + tb * (0.06 + 0.94 * rows)) / 46.0;
    const double mem = (double)((O + 15) / 16 * 16) * (double)steps * 128e-6 / 5.1;
    return 1.7 + std::sqrt(std::sqrt(walk * walk * walk * walk + mem * mem * mem * mem));
}
static int few_tile(int64_t O, int64_t K, int64_t T)
{
    int best = 0;
    for (int c = 1; c < (int)(sizeof(kFewTiles) / sizeof(kFewTiles[0])); c++)
        if (few_cost(c, O, K, T) < few_cost(best, O, K, T)) best = c;
    return best;
}

template <typename T, int AB, int TB> static int launch_few_tile(const DfParams &P, hipStream_t s)
{
    hipLaunchKernelGGL((dense16_few_kernel<T, AB, TB>), dim3((unsigned)((P.O + 16 * AB - 1) / (16 * AB)), (unsigned)((P.T + 16 * TB - 1) / (16 * TB))),
                       dim3(1024), 0, s, P);
    NMG_HIP_TRY(hipGetLastError());
    return NMG_OK;
}
template <typename T> static int launch_few(const DfParams &P, hipStream_t s)
{
    switch (few_tile(P.O, P.K, P.T)) {
    case 0: return launch_few_tile<T, 1, 1>(P, s);
    case 1: return launch_few_tile<T, 2, 1>(P, s);
    case 2: return launch_few_tile<T, 4, 1>(P, s);
    default: return launch_few_tile<T, 2, 2>(P, s);
    }
}

static bool dense16_square(int64_t O, int64_t T)
{
    const int64_t tm = (O + 255) / 256, t256 = tm * ((T + 255) / 256), t128 = tm * ((T + 127) / 128);
    const double fill256 = (double)t256 / (double)((t256 + 255) / 256 * 256);
    const double fill128 = (double)t128 / (double)((t128 + 255) / 256 * 256);
    return t256 >= 256 && fill256 * 1.055 >= fill128;
}

// The tiles of the direct kernel: 256 outputs x 128 tokens, 256 x 256 and, narrow, 128 x 128.
enum { DENSE_WIDE, DENSE_SQUARE, DENSE_NARROW };

static inline int64_t dense16_tiles(int tile, int64_t O, int64_t T)
{
    return (tile == DENSE_NARROW ? (O + 127) / 128 : (O + 255) / 256) * (tile == DENSE_SQUARE ? (T + 255) / 256 : (T + 127) / 128);
}

// Time in us of a product whose reduction of `steps` K steps is cut into `slices`, one workgroup per CU: whole rounds of 256
// workgroups and a last one that is the faster the fewer it has, a step and a fixed part per round; with slices the second kernel and
// the partial sums, written and read once; and the weight comes from memory in any case (fitted without
// the term of smfmac_cost for the narrow tile's fetches).  The constants are those of 17 weights
// of 512^2 to 16384 x 2048 and 1024 x 16384 with 17 to 6000 tokens in 1 to 16 slices (fp16 4:8, weights new in every pass), fitted before the
// slices' workgroups were dealt out by XCD.  Against the best of every tile and slice as the kernels are now, 16 weights x 33 to 4096 tokens:
// 1.6 % behind in the mean, 3 % and more in 47 of 224 (8192 x 1024 x 4096 72.0, 57.7; 512 x 16384 x 450 25.3, 21.9), and 2.1 % for 8 weights
// that no fit has seen (profiles/tile_slice_sweep.txt).  Row operands keep a rule of their own (dense16_square): the product of
// rows has the square tile only, against another kernel.
static double dense16_cost(int tile, int slices, int64_t O, int64_t steps, int64_t T)
{
    static const struct { double step, fixed, crowd; } of[] = {{0.54, 4.3, 0.44}, {0.89, 11.0, 0.49}, {0.30, 3.8, 0.63}};
    const auto c = of[tile];
    const int64_t groups = dense16_tiles(tile, O, T) * slices, rest = groups % 256;
    const double walk = (double)((steps + slices - 1) / slices) * c.step;
    double t = (double)(groups / 256) * (walk * (1 + c.crowd) + c.fixed);
    if (rest) t += walk * (1 + c.crowd * (double)rest / 256) + c.fixed;
    if (slices > 1) t += 2.6 + (double)slices * (double)T * (double)O * 8 * 0.21e-6;
    const double mem = (double)O * (double)steps * 128 * 0.15e-6 + c.fixed;
    return std::sqrt(std::sqrt(t * t * t * t + mem * mem * mem * mem));
}

// The tile of a product.  Where 128 x 128 needs more than one round it is behind (4096 x 4096 x 2048 tokens: 256 wide tiles 52.8 us, 512
// narrow 65.7).  Below, it leaves fewer CUs idle: x 777 in two slices of wide tiles and their sum 36.7, 224 narrow tiles 30.0;
// 1024 x 1024 x 777 16.6 -> 9.7; 768 x 3072 x 4096 31.5 -> 22.1.  256 x 256 moves the fewest bytes per flop and is for what wide
// tiles do not take in one round: 4096 x 11008 x 2500, 320 wide tiles 265, 160 square 195; but 752 against 384 412 and 428.
static int dense16_tile(int slices, int64_t O, int64_t steps, int64_t T)
{
    const double wide = dense16_cost(DENSE_WIDE, slices, O, steps, T);
    if (dense16_tiles(DENSE_NARROW, O, T) * slices <= 256) return dense16_cost(DENSE_NARROW, slices, O, steps, T) < wide ? DENSE_NARROW : DENSE_WIDE;
    // (4 % between the two is within the error of the model)
    if (slices == 1 && dense16_tiles(DENSE_WIDE, O, T) > 256 && dense16_cost(DENSE_SQUARE, 1, O, steps, T) * 1.04 < wide) return DENSE_SQUARE;
    return DENSE_WIDE;
}

// The slices of a product on the direct kernel and its time.
static double dense16_best(int64_t O, int64_t steps, int64_t T, int *slices)
{
    *slices = 1;
    double least = dense16_cost(dense16_tile(1, O, steps, T), 1, O, steps, T);
    // at most a workgroup per CU and eight slices (sixteen for a handful of tiles), at least four steps each
    const int64_t wide = dense16_tiles(DENSE_WIDE, O, T);
    for (int64_t s = 2; s <= std::min<int64_t>(wide <= 8 ? 16 : 8, steps / 4) && wide * s <= 256; s++) {
        if (splitk_fit(steps, s) != s) continue;
        const double t = dense16_cost(dense16_tile((int)s, O, steps, T), (int)s, O, steps, T);
        if (t < least) {
            least = t;
            *slices = (int)s;
        }
    }
    return least;
}

// Whether the kernel for few tokens takes a product: it is not behind the direct kernel, from 17 tokens on 15 % ahead
// by both models.  us, direct kernel in slices and their sum -> this, weights from memory: 512 x 1024, 16 tokens 7.1 -> 3.6, 640 x 1408, 1
// 7.2 -> 3.2, 2048^2, 8 7.9 -> 4.2, 32 8.6 -> 4.8, 4096^2, 16 14.6 -> 10.1, 10624 x 1664, 8 14.5 -> 9.0, 8192^2, 16 30.2 -> 25.2;
// long reductions of few outputs stay: 888 x 8128, 16 11.0, 15.3.
static bool few_takes(int64_t O, int64_t K, int64_t T) { return T <= 64 && O > 0 && K > 0 && T > 0 && O <= ((int64_t)1 << 24); }
static bool few_ahead(int64_t O, int64_t K, int64_t T, double direct_us)
{
    return few_cost(few_tile(O, K, T), O, K, T) * (T > 16 ? 1.15 : 1.0) < direct_us;
}
static bool few_pays(int64_t O, int64_t K, int64_t T)
{
    int slices;
    return few_takes(O, K, T) && few_ahead(O, K, T, dense16_best(O, (K + 63) / 64, T, &slices));
}

template <typename T, bool CT = false> static int launch_dense(DfParams &P, int variant, hipStream_t s)
{
    // Variant 0: 256 outputs x 128 tokens per workgroup, 1: 256 x 256, -1: the faster one of all tiles.
    // (A sixteen-phase form of the 256 x 256 tile on the 32 x 32 x 16 instruction once gave wrong
    // values now and then; the forms here pass the static check of their hand-tracked loads and
    // the repeated full-chip test.)
    P.in_order = variant >= 0;
    const int tile = variant < 0 ? dense16_tile(P.ksplit > 1 ? P.ksplit : 1, P.O, P.KP, P.T) : variant;
    if (tile == DENSE_NARROW) return launch_dense16<T, 8, 2, false, CT, false, 2>(P, s);
    if (tile == DENSE_SQUARE) return launch_dense16<T, 16, 4, false, CT>(P, s);
    return launch_dense16<T, 8, 2, false, CT>(P, s);
}

// C = A B from B as it lies, on the tile of the plain product.  us, with every step waiting for the loads that it had just issued (256 x 128
// tiles only) -> now: 4096 x 4096 x 2048 columns 80.5 -> 62, 1024^3 20 -> 11, 512 x 4096 x 4096 78 -> 39, 768 x 768 x 512 16.3 -> 9.1,
// 8192 x 4096 x 4096 (256 x 256 tiles) 340 -> 216.
template <typename T> static int launch_dense_tt(DfParams &P, hipStream_t s)
{
    const int tile = dense16_tile(1, P.O, P.KP, P.T);
    if (tile == DENSE_NARROW) return launch_dense16<T, 8, 2, true, true, false, 2>(P, s);
    if (tile == DENSE_SQUARE) return launch_dense16<T, 16, 4, true>(P, s);
    return launch_dense16<T, 8, 2, true>(P, s);
}

// Y[T, O] = X[T, K] A[O, K]^T (+ bias), both operands rows in memory, on 256 x 256 tiles.  The caller has checked
// extents, pitches and alignment (nmg_gemm_nt).  Bound by the vector memory path: a weight load touches 16 rows.  us,
// 256 x 128 kernel of nmg_gemm_nt -> this one: 4096 x 4096, K = 2048 (the weight gradient of torch.mm) 77 -> 68;
// 16384 x 4096, K = 512 112 -> 94.  On 256 x 128 tiles this form is behind (8192 x 512, K = 4096: 60 -> 83), so it
// takes the results that fill the chip with 256 x 256 tiles.
bool dense_rows16_pays(int64_t O, int64_t T) { return dense16_square(O, T); }

int dense_rows16(const void *d_a, int64_t lda, const void *d_x, int64_t ldx, void *d_y, int64_t ldy, const void *d_bias,
                 int64_t O, int64_t K, int64_t T, int dtype, void *stream)
{
    DfParams P{};
    P.df = d_a;
    P.lda = lda;
    P.x = d_x;
    P.y = d_y;
    P.bias = d_bias;
    P.O = O;
    P.K = K;
    P.T = T;
    P.ldx = ldx;
    P.ldy = ldy;
    P.KP = (int)(K / 64);
    hipStream_t s = (hipStream_t)stream;
    return dtype == NMG_F16 ? launch_dense16<__half, 16, 4, false, false, true>(P, s)
                            : launch_dense16<__hip_bfloat16, 16, 4, false, false, true>(P, s);
}

}  // namespace nmg

using namespace nmg;

// positions per expansion tile: the largest multiple of lcm(m, 32) that fits 128 (0: none)
static int densefrag_tile_positions(int m)
{
    if (m < 1 || m > 64) return 0;
    int l = m;
    while (l % 32 != 0) l += m;   // lcm(m, 32)
    return l <= DFX_P ? DFX_P / l * l : 0;
}

extern "C" int nmg_densefrag_supported(int n, int m)
{
    // m a power of two, or three times one (3, 6, 12, 24, 48): a tile of whole blocks that is also
    // a whole number of 32-output blocks and 16-position k-steps
    return (n >= 0 && n <= m && densefrag_tile_positions(m) > 0) ? 1 : 0;
}

extern "C" int nmg_densefrag_elems(int64_t O, int64_t K, int64_t *elems)
{
    NMG_REQUIRE(O >= 0 && K >= 0 && elems, NMG_ERR_ARG, "invalid extents");
    *elems = ((O + 255) / 256) * 256 * ((K + 63) / 64 * 64);
    return NMG_OK;
}

extern "C" int nmg_densefrag(const void *d_pk_val, const void *d_pk_pat, int64_t G, int64_t S, int transpose,
                             void *d_df, int n, int m, int dtype, void *stream)
{
    NMG_REQUIRE(nmg_densefrag_supported(n, m), NMG_ERR_UNSUPPORTED,
                "densefrag needs m to be a power of two or three times one (at most 64), got %d:%d", n, m);
    NMG_REQUIRE(dtype == NMG_F16 || dtype == NMG_BF16, NMG_ERR_UNSUPPORTED, "densefrag takes f16/bf16");
    NMG_REQUIRE(G >= 0 && S >= 0, NMG_ERR_ARG, "negative extent");
    const int64_t O = transpose ? S : G, K = transpose ? G : S, Kp = (K + 63) / 64 * 64;
    if (O == 0 || K == 0) return NMG_OK;
    NMG_REQUIRE(d_pk_val && d_pk_pat && d_df, NMG_ERR_ARG, "null device pointer");
    DfExpandParams P{};
    if (int rc = device_order(n, m, &P.order)) return rc;
    P.pk_val = d_pk_val;
    P.pk_pat = d_pk_pat;
    P.df = d_df;
    P.G = G;
    P.S = S;
    P.nb = (S + m - 1) / m;
    P.OB = (O + 255) / 256 * 8;
    P.K16 = Kp / 16;
    P.n = n;
    P.m = m;
    P.pat_bytes = binom(m, n) <= 256 ? 1 : 2;
    P.pt = densefrag_tile_positions(m);
    P.bpt = P.pt / m;
    P.transpose = transpose ? 1 : 0;
    // the grid covers the padded operand: outputs up to a multiple of 256, the reduction to one of 64
    const int64_t Gp = transpose ? Kp : P.OB * 32, Sp = transpose ? P.OB * 32 : Kp;
    const int64_t gx = (Sp + P.pt - 1) / P.pt, gy = (Gp + DFX_L - 1) / DFX_L;
    NMG_REQUIRE(gx <= 0x7fffffffLL && gy <= 65535, NMG_ERR_UNSUPPORTED, "weight too large for one launch");
    dim3 grid((unsigned)gx, (unsigned)gy);
    hipStream_t s = (hipStream_t)stream;
    // the specialised forms load the n values of a block as one word: n * 2 bytes, aligned
    const int64_t table = binom(m, n) * n;
    P.order_bytes = (int)(table <= 2048 ? table : 0);
    const int nv = (n == 3 || ((n == 1 || n == 2 || n == 4) && (uintptr_t)d_pk_val % (2 * n) == 0)) && table <= 2048 ? n : 0;
    auto launch = [&](auto tag) {
        using T = decltype(tag);
        switch (nv) {
        case 1: hipLaunchKernelGGL((densefrag_kernel<T, 1>), grid, dim3(256), 0, s, P); break;
        case 2: hipLaunchKernelGGL((densefrag_kernel<T, 2>), grid, dim3(256), 0, s, P); break;
        case 3: hipLaunchKernelGGL((densefrag_kernel<T, 3>), grid, dim3(256), 0, s, P); break;
        case 4: hipLaunchKernelGGL((densefrag_kernel<T, 4>), grid, dim3(256), 0, s, P); break;
        default: hipLaunchKernelGGL((densefrag_kernel<T, 0>), grid, dim3(256), 0, s, P); break;
        }
    };
    if (dtype == NMG_F16)
        launch(__half{});
    else
        launch(__hip_bfloat16{});
    NMG_HIP_TRY(hipGetLastError());
    return NMG_OK;
}

extern "C" int nmg_densefrag_few(int64_t O, int64_t K, int64_t T) { return K % 8 == 0 && few_pays(O, K, T) ? 1 : 0; }

extern "C" int nmg_spmm_densefrag_few(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx, void *d_y, int64_t ldy,
                                      const void *d_bias, int64_t T, int dtype, void *stream)
{
    NMG_REQUIRE(dtype == NMG_F16 || dtype == NMG_BF16, NMG_ERR_UNSUPPORTED, "densefrag takes f16/bf16");
    NMG_REQUIRE(O >= 0 && K >= 0 && T >= 0, NMG_ERR_ARG, "negative extent");
    NMG_REQUIRE(ldx >= K && ldy >= O, NMG_ERR_ARG, "leading dimension smaller than row length");
    NMG_REQUIRE(K % 8 == 0 && K > 0 && ldx % 8 == 0 && ((uintptr_t)d_x % 16) == 0, NMG_ERR_UNSUPPORTED,
                "needs K %% 8 == 0 and 16-byte aligned activation rows");
    NMG_REQUIRE(T <= 64 && O <= ((int64_t)1 << 24) && K <= ((int64_t)1 << 30), NMG_ERR_UNSUPPORTED, "at most 64 tokens, 2^24 outputs and a reduction of 2^30");
    if (O == 0 || T == 0) return NMG_OK;
    NMG_REQUIRE(d_df && d_x && d_y, NMG_ERR_ARG, "null device pointer");
    DfParams P{};
    P.df = d_df;
    P.x = d_x;
    P.y = d_y;
    P.bias = d_bias;
    P.O = O;
    P.K = K;
    P.T = T;
    P.ldx = ldx;
    P.ldy = ldy;
    P.KP = (int)((K + 63) / 64);
    hipStream_t s = (hipStream_t)stream;
    return dtype == NMG_F16 ? launch_few<__half>(P, s) : launch_few<__hip_bfloat16>(P, s);
}

extern "C" int nmg_spmm_densefrag(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx,
                                  void *d_y, int64_t ldy, const void *d_bias, int64_t T, int dtype,
                                  int variant, void *stream)
{
    NMG_REQUIRE(dtype == NMG_F16 || dtype == NMG_BF16, NMG_ERR_UNSUPPORTED, "densefrag takes f16/bf16");
    NMG_REQUIRE(O >= 0 && K >= 0 && T >= 0, NMG_ERR_ARG, "negative extent");
    NMG_REQUIRE(variant >= -1 && variant <= 1, NMG_ERR_ARG, "unknown tile variant %d", variant);
    NMG_REQUIRE(ldx >= K && ldy >= O, NMG_ERR_ARG, "leading dimension smaller than row length");
    NMG_REQUIRE(K % 64 == 0 && K > 0 && ldx % 8 == 0 && ((uintptr_t)d_x % 16) == 0, NMG_ERR_UNSUPPORTED,
                "needs K %% 64 == 0 and 16-byte aligned activation rows");
    NMG_REQUIRE(T * ldx * 2 < ((int64_t)1 << 31), NMG_ERR_UNSUPPORTED, "activations must be smaller than 2 GiB");
    if (O == 0 || T == 0) return NMG_OK;
    NMG_REQUIRE(d_df && d_x && d_y, NMG_ERR_ARG, "null device pointer");
    DfParams P{};
    P.df = d_df;
    P.x = d_x;
    P.y = d_y;
    P.bias = d_bias;
    P.O = O;
    P.K = K;
    P.T = T;
    P.ldx = ldx;
    P.ldy = ldy;
    P.KP = (int)(K / 64);
    hipStream_t s = (hipStream_t)stream;
    if (variant < 0 && few_pays(O, K, T)) return dtype == NMG_F16 ? launch_few<__half>(P, s) : launch_few<__hip_bfloat16>(P, s);
    return dtype == NMG_F16 ? launch_dense<__half>(P, variant, s) : launch_dense<__hip_bfloat16>(P, variant, s);
}

extern "C" int nmg_spmm_densefrag_tt(const void *d_df, int64_t O, int64_t K, const void *d_b, int64_t ldb, void *d_c,
                                     int64_t ldc, const void *d_bias, int64_t T, int dtype, void *stream)
{
    NMG_REQUIRE(dtype == NMG_F16 || dtype == NMG_BF16, NMG_ERR_UNSUPPORTED, "densefrag takes f16/bf16");
    NMG_REQUIRE(O >= 0 && K >= 0 && T >= 0, NMG_ERR_ARG, "negative extent");
    NMG_REQUIRE(ldb >= T && ldc >= T, NMG_ERR_ARG, "leading dimension smaller than row length");
    NMG_REQUIRE(K % 64 == 0 && K > 0 && ldb % 8 == 0 && ((uintptr_t)d_b % 16) == 0, NMG_ERR_UNSUPPORTED,
                "the transposed product needs K %% 64 == 0, ldb %% 8 == 0 and a 16-byte aligned B");
    NMG_REQUIRE(ldb < ((int64_t)1 << 24), NMG_ERR_UNSUPPORTED, "leading dimension too large");
    if (O == 0 || T == 0) return NMG_OK;
    NMG_REQUIRE(d_df && d_b && d_c, NMG_ERR_ARG, "null device pointer");
    DfParams P{};
    P.df = d_df;
    P.x = d_b;
    P.y = d_c;
    P.bias = d_bias;
    P.O = O;
    P.K = K;
    P.T = T;
    P.ldx = ldb;
    P.ldy = ldc;
    P.KP = (int)(K / 64);
    hipStream_t s = (hipStream_t)stream;
    return dtype == NMG_F16 ? launch_dense_tt<__half>(P, s) : launch_dense_tt<__hip_bfloat16>(P, s);
}

// C[O, T] = A X^T for X [T, K]: the product above with a transposed result.
extern "C" int nmg_spmm_densefrag_ct(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx, void *d_c,
                                     int64_t ldc, const void *d_bias, int64_t T, int dtype, void *stream)
{
    NMG_REQUIRE(dtype == NMG_F16 || dtype == NMG_BF16, NMG_ERR_UNSUPPORTED, "densefrag takes f16/bf16");
    NMG_REQUIRE(O >= 0 && K >= 0 && T >= 0, NMG_ERR_ARG, "negative extent");
    NMG_REQUIRE(ldx >= K && ldc >= T, NMG_ERR_ARG, "leading dimension smaller than row length");
    NMG_REQUIRE(K % 64 == 0 && K > 0 && ldx % 8 == 0 && ((uintptr_t)d_x % 16) == 0, NMG_ERR_UNSUPPORTED,
                "needs K %% 64 == 0 and 16-byte aligned activation rows");
    NMG_REQUIRE(T * ldx * 2 < ((int64_t)1 << 31), NMG_ERR_UNSUPPORTED, "activations must be smaller than 2 GiB");
    if (O == 0 || T == 0) return NMG_OK;
    NMG_REQUIRE(d_df && d_x && d_c, NMG_ERR_ARG, "null device pointer");
    DfParams P{};
    P.df = d_df;
    P.x = d_x;
    P.y = d_c;
    P.bias = d_bias;
    P.O = O;
    P.K = K;
    P.T = T;
    P.ldx = ldx;
    P.ldy = ldc;
    P.KP = (int)(K / 64);
    hipStream_t s = (hipStream_t)stream;
    return dtype == NMG_F16 ? launch_dense<__half, true>(P, -1, s) : launch_dense<__hip_bfloat16, true>(P, -1, s);
}

extern "C" int nmg_densefrag_plan(int64_t O, int64_t K, int64_t T, int *slices, int64_t *workspace_bytes)
{
    NMG_REQUIRE(O >= 0 && K >= 0 && T >= 0, NMG_ERR_ARG, "negative extent");
    NMG_REQUIRE(slices && workspace_bytes, NMG_ERR_ARG, "null output pointer");
    int best = 1;
    if (O > 0 && T > 0 && K / 64 > 0) {
        const double us = dense16_best(O, K / 64, T, &best);
        if (few_takes(O, K, T) && few_ahead(O, K, T, us)) best = 1;
    }
    *slices = best;
    *workspace_bytes = best > 1 ? (int64_t)best * T * ((O + 255) / 256) * 256 * 4 : 0;
    return NMG_OK;
}

extern "C" int nmg_spmm_densefrag_splitk(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx,
                                         void *d_y, int64_t ldy, const void *d_bias, int64_t T, int dtype,
                                         int slices, void *d_workspace, int64_t workspace_bytes, void *stream)
{
    if (slices <= 1) return nmg_spmm_densefrag(d_df, O, K, d_x, ldx, d_y, ldy, d_bias, T, dtype, -1, stream);
    NMG_REQUIRE(dtype == NMG_F16 || dtype == NMG_BF16, NMG_ERR_UNSUPPORTED, "densefrag takes f16/bf16");
    NMG_REQUIRE(O >= 0 && K >= 0 && T >= 0, NMG_ERR_ARG, "negative extent");
    NMG_REQUIRE(ldx >= K && ldy >= O, NMG_ERR_ARG, "leading dimension smaller than row length");
    NMG_REQUIRE(K % 64 == 0 && K > 0 && ldx % 8 == 0 && ((uintptr_t)d_x % 16) == 0, NMG_ERR_UNSUPPORTED,
                "needs K %% 64 == 0 and 16-byte aligned activation rows");
    NMG_REQUIRE(T * ldx * 2 < ((int64_t)1 << 31), NMG_ERR_UNSUPPORTED, "activations must be smaller than 2 GiB");
    if (O == 0 || T == 0) return NMG_OK;
    const int64_t KP = K / 64, tiles_m = (O + 255) / 256;
    NMG_REQUIRE(slices <= 256 && splitk_fit(KP, slices) == slices, NMG_ERR_ARG,
                "%d slices leave one empty (%lld K steps)", slices, (long long)KP);
    const int64_t need = (int64_t)slices * T * tiles_m * 256 * 4;
    NMG_REQUIRE(d_workspace && workspace_bytes >= need && ((uintptr_t)d_workspace % 16) == 0, NMG_ERR_ARG,
                "workspace of %lld bytes (16-byte aligned) needed, %lld given", (long long)need,
                (long long)workspace_bytes);
    NMG_REQUIRE(d_df && d_x && d_y, NMG_ERR_ARG, "null device pointer");
    DfParams P{};
    P.df = d_df;
    P.x = d_x;
    P.y = d_y;
    P.bias = d_bias;
    P.O = O;
    P.K = K;
    P.T = T;
    P.ldx = ldx;
    P.ldy = ldy;
    P.KP = (int)KP;
    P.ksplit = slices;
    P.part = (float *)d_workspace;
    P.part_ld = tiles_m * 256;
    hipStream_t s = (hipStream_t)stream;
    return dtype == NMG_F16 ? launch_dense<__half>(P, -1, s) : launch_dense<__hip_bfloat16>(P, -1, s);
}

// A reduction that is a multiple of 8 only, activations as they lie (slices and workspace: nmg_densefrag_plan of the extent in whole
// steps).  us, copy of the activations in whole steps and the product -> this: 4:8 1768 x 2216 x 298
// tokens 18.7 -> 15.8, 11256 x 672 x 240 from memory 20.5 -> 18.2.
extern "C" int nmg_spmm_densefrag_ragged(const void *d_df, int64_t O, int64_t K, const void *d_x, int64_t ldx, void *d_y, int64_t ldy,
                                         const void *d_bias, int64_t T, int dtype, int slices, void *d_workspace, int64_t workspace_bytes,
                                         void *stream)
{
    NMG_REQUIRE(dtype == NMG_F16 || dtype == NMG_BF16, NMG_ERR_UNSUPPORTED, "densefrag takes f16/bf16");
    NMG_REQUIRE(O >= 0 && K >= 0 && T >= 0, NMG_ERR_ARG, "negative extent");
    NMG_REQUIRE(ldx >= K && ldy >= O, NMG_ERR_ARG, "leading dimension smaller than row length");
    NMG_REQUIRE(K % 8 == 0 && K > 0 && ldx % 8 == 0 && ((uintptr_t)d_x % 16) == 0, NMG_ERR_UNSUPPORTED,
                "needs K %% 8 == 0 and 16-byte aligned activation rows");
    NMG_REQUIRE(T * ldx * 2 < ((int64_t)1 << 31), NMG_ERR_UNSUPPORTED, "activations must be smaller than 2 GiB");
    if (O == 0 || T == 0) return NMG_OK;
    const int64_t KP = (K + 63) / 64, tiles_m = (O + 255) / 256;
    NMG_REQUIRE(slices >= 1 && slices <= 256 && splitk_fit(KP, slices) == slices, NMG_ERR_ARG, "%d slices leave one empty (%lld K steps)",
                slices, (long long)KP);
    const int64_t need = slices > 1 ? (int64_t)slices * T * tiles_m * 256 * 4 : 0;
    NMG_REQUIRE(need == 0 || (d_workspace && workspace_bytes >= need && ((uintptr_t)d_workspace % 16) == 0), NMG_ERR_ARG,
                "workspace of %lld bytes (16-byte aligned) needed, %lld given", (long long)need, (long long)workspace_bytes);
    NMG_REQUIRE(d_df && d_x && d_y, NMG_ERR_ARG, "null device pointer");
    DfParams P{};
    P.df = d_df;
    P.x = d_x;
    P.y = d_y;
    P.bias = d_bias;
    P.O = O;
    P.K = K;
    P.T = T;
    P.ldx = ldx;
    P.ldy = ldy;
    P.KP = (int)KP;
    P.tail = (int)(K % 64);
    P.ksplit = slices;
    P.part = (float *)d_workspace;
    P.part_ld = tiles_m * 256;
    hipStream_t s = (hipStream_t)stream;
    return dtype == NMG_F16 ? launch_dense<__half>(P, -1, s) : launch_dense<__hip_bfloat16>(P, -1, s);
}
