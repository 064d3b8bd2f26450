// Dense -> grouped n:m compressor (bit-exact with the reference CPU sparsifier), plus the
// element-wise companions: to_dense scatter, same-pattern gather and the rowpack re-ordering.
//
// Reference algorithm (grouped_nm_tensor.py:255-297), per tile of c*g columns x m values:
//   score[o][p] = sum_j |d[o][order[p][j]]|  (left to right, in the input precision)
//   sort all (score, o, p) descending (ties: larger o, then larger p)
//   walk the sorted list; accept (o, p) if column o is free and pattern p has < g members;
//   the k-th column accepted by pattern p lands in slot p*g + k.
//
// GPU formulation (same result, no global sort): the sorted walk always accepts next the
// largest key among {(o, p): o free, p not full}.  Every free column keeps its "head" = its best
// key over the patterns that still have room; one step = arg-max of the heads over the free
// columns, accept it, and if that filled the pattern, recompute the heads that pointed to it.
// A step is a wavefront (or workgroup) max-reduction; a tile needs c*g steps.  The kernels
// further down batch these steps (lane teams: many small tiles per wavefront); most tiles never come
// here but are solved as a matching (nmg_match.h).
//
// Work split: a "team" of TW wavefronts owns one tile; a workgroup holds NT teams that work on
// NT consecutive tiles, which are adjacent in memory along the sparse dim when that dim is the
// contiguous one, so the cooperative tile load is coalesced across them.
#include "nmg_common.h"

#include <algorithm>

namespace nmg {

template <typename T> struct ScoreOf { using type = float; using bits = uint32_t; };
template <> struct ScoreOf<double> { using type = double; using bits = uint64_t; };

__device__ __forceinline__ uint32_t score_bits(float s) { return __float_as_uint(s); }
__device__ __forceinline__ uint64_t score_bits(double s) { return (uint64_t)__double_as_longlong(s); }

__device__ __forceinline__ float score_of(float x) { return fabsf(x); }
__device__ __forceinline__ double score_of(double x) { return fabs(x); }
__device__ __forceinline__ float score_of(__half x) { return fabsf(__half2float(x)); }
__device__ __forceinline__ float score_of(__hip_bfloat16 x) { return fabsf(__bfloat162float(x)); }

// Key = (score bits, (o << 16 | p) + 1); the all-zero key means "nothing".
template <typename SB> struct Key {
    SB s;
    uint32_t op;
};
template <typename SB> __device__ __forceinline__ bool key_gt(const Key<SB> &a, const Key<SB> &b)
{
    return a.s > b.s || (a.s == b.s && a.op > b.op);
}

__device__ __forceinline__ uint32_t shfl_xor_bits(uint32_t v, int mask)
{
    return (uint32_t)__shfl_xor((int)v, mask, 64);
}
__device__ __forceinline__ uint64_t shfl_xor_bits(uint64_t v, int mask)
{
    uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, mask, 64);
    uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), mask, 64);
    return ((uint64_t)hi << 32) | lo;
}

template <typename SB> __device__ __forceinline__ Key<SB> wave_max(Key<SB> k)
{
#pragma unroll
    for (int mask = 32; mask >= 1; mask >>= 1) {
        Key<SB> o;
        o.s = shfl_xor_bits(k.s, mask);
        o.op = shfl_xor_bits(k.op, mask);
        if (key_gt(o, k)) k = o;
    }
    return k;
}

struct SparsifyParams {
    const void *dense;
    void *val;
    int16_t *idx;
    const int8_t *order;  // device table [c][n]
    ViewDev view;
    int64_t outer;
    int n, m, g, c, cols;
    int team_bytes;  // LDS bytes of one team's region
    int off_hs, off_hp, off_cnt, off_oval, off_oidx, off_wbest;  // offsets inside a team region
};

template <int TW> __device__ __forceinline__ void team_sync()
{
    if (TW == 1) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

template <typename T, int TW, int NT>
__global__ __launch_bounds__(64 * TW * NT) void sparsify_kernel(SparsifyParams P)
{
    using CT = typename ScoreOf<T>::type;
    using SB = typename ScoreOf<T>::bits;
    constexpr int TS = 64 * TW;  // threads per team
    extern __shared__ __align__(16) unsigned char smem[];

    const int n = P.n, m = P.m, g = P.g, c = P.c, cols = P.cols;
    const int tid = threadIdx.x;
    const int team = tid / TS, tt = tid % TS;
    const int wave_in_team = tt / 64;

    // LDS: [order table][team 0 region][team 1 region]...
    int8_t *s_order = (int8_t *)smem;
    const int order_bytes = (c * n + 15) & ~15;
    unsigned char *region = smem + order_bytes + (size_t)team * P.team_bytes;
    T *s_d = (T *)region;
    SB *s_hs = (SB *)(region + P.off_hs);
    uint16_t *s_hp = (uint16_t *)(region + P.off_hp);
    int16_t *s_cnt = (int16_t *)(region + P.off_cnt);
    T *s_oval = (T *)(region + P.off_oval);
    int16_t *s_oidx = (int16_t *)(region + P.off_oidx);
    Key<SB> *s_wbest = (Key<SB> *)(region + P.off_wbest);

    for (int i = tid; i < c * n; i += 64 * TW * NT) s_order[i] = P.order[i];

    // ---- cooperative load of the NT tiles of this workgroup (zero beyond G / S) ----
    const int64_t tile0 = (int64_t)blockIdx.x * NT;
    const T *dense = (const T *)P.dense;
    const int per_tile = cols * m;
    for (int e = tid; e < NT * per_tile; e += 64 * TW * NT) {
        int r = e % m;
        int rest = e / m;
        int tm = rest % NT;
        int o = rest / NT;
        int64_t t = tile0 + tm;
        T v = Zero<T>::v();
        if (t < P.outer) {
            int64_t tiles_per_b = P.view.num_chunks * P.view.num_blocks;
            int64_t b = t / tiles_per_b;
            int64_t rem = t - b * tiles_per_b;
            int64_t kc = rem / P.view.num_blocks;
            int64_t mb = rem - kc * P.view.num_blocks;
            int64_t gi = kc * cols + o, si = mb * m + r;
            if (gi < P.view.G && si < P.view.S)
                v = dense[b * P.view.stride_b + gi * P.view.stride_g + si * P.view.stride_s];
        }
        T *dst = (T *)(smem + order_bytes + (size_t)tm * P.team_bytes);
        dst[o * m + r] = v;
    }
    for (int p = tt; p < c; p += TS) s_cnt[p] = 0;
    __syncthreads();

    // Best key of column o over the patterns that still have room (skip_p = pattern that just
    // filled up and whose counter may not be visible yet).
    auto head_of = [&](int o, int skip_p, SB &best_s, int &best_p) {
        best_p = -1;
        best_s = 0;
        const T *col = s_d + o * m;
        for (int p = 0; p < c; p++) {
            if (p == skip_p || s_cnt[p] >= g) continue;
            CT acc = 0;
            for (int j = 0; j < n; j++) acc += score_of(col[s_order[p * n + j]]);
            SB sb = score_bits(acc);
            if (best_p < 0 || sb >= best_s) {  // ties: larger p wins
                best_s = sb;
                best_p = p;
            }
        }
    };
    auto local_best = [&]() {
        Key<SB> lb;
        lb.s = 0;
        lb.op = 0;
        for (int o = tt; o < cols; o += TS) {
            uint16_t hp = s_hp[o];
            if (hp == 0xFFFF) continue;
            Key<SB> k;
            k.s = s_hs[o];
            k.op = (((uint32_t)o << 16) | hp) + 1u;
            if (key_gt(k, lb)) lb = k;
        }
        return lb;
    };

    for (int o = tt; o < cols; o += TS) {
        SB bs;
        int bp;
        head_of(o, -1, bs, bp);
        s_hs[o] = bs;
        s_hp[o] = (uint16_t)bp;
    }
    Key<SB> lb = local_best();

    for (int step = 0; step < cols; step++) {
        Key<SB> b = wave_max(lb);
        if (TW > 1) {
            if ((tt & 63) == 0) s_wbest[wave_in_team] = b;
            __syncthreads();
            b = s_wbest[0];
#pragma unroll
            for (int w = 1; w < TW; w++) {
                Key<SB> o = s_wbest[w];
                if (key_gt(o, b)) b = o;
            }
        }
        const uint32_t op = b.op - 1u;
        const int o_star = (int)(op >> 16), p_star = (int)(op & 0xFFFFu);
        const int oldcnt = s_cnt[p_star];
        team_sync<TW>();
        bool dirty = false;
        if (o_star % TS == tt) {
            const int slot = p_star * g + oldcnt;
            s_cnt[p_star] = (int16_t)(oldcnt + 1);
            s_hp[o_star] = 0xFFFF;
            s_oidx[slot] = (int16_t)o_star;
            for (int j = 0; j < n; j++) s_oval[slot * n + j] = s_d[o_star * m + s_order[p_star * n + j]];
            dirty = true;
        }
        if (oldcnt + 1 == g) {
            for (int o = tt; o < cols; o += TS) {
                if (s_hp[o] != (uint16_t)p_star) continue;
                SB bs;
                int bp;
                head_of(o, p_star, bs, bp);
                s_hs[o] = bs;
                s_hp[o] = (uint16_t)bp;
                dirty = true;
            }
        }
        if (dirty) lb = local_best();
        team_sync<TW>();
    }

    // ---- coalesced store of the team's tile ----
    __syncthreads();
    const int64_t t = tile0 + team;
    if (t < P.outer) {
        T *val = (T *)P.val + t * (int64_t)cols * n;
        int16_t *idx = P.idx + t * (int64_t)cols;
        for (int i = tt; i < cols * n; i += TS) val[i] = s_oval[i];
        for (int i = tt; i < cols; i += TS) idx[i] = s_oidx[i];
    }
}

static inline int align_up(int x, int a) { return (x + a - 1) / a * a; }

template <typename T, int TW, int NT>
static int launch_sparsify(SparsifyParams &P, hipStream_t stream)
{
    using SB = typename ScoreOf<T>::bits;
    const int cols = P.cols, n = P.n, m = P.m, c = P.c;
    int off = align_up(cols * m * (int)sizeof(T), 16);
    P.off_hs = off;
    off = align_up(off + cols * (int)sizeof(SB), 16);
    P.off_hp = off;
    off = align_up(off + cols * 2, 16);
    P.off_cnt = off;
    off = align_up(off + c * 2, 16);
    P.off_oval = off;
    off = align_up(off + cols * (n > 0 ? n : 1) * (int)sizeof(T), 16);
    P.off_oidx = off;
    off = align_up(off + cols * 2, 16);
    P.off_wbest = off;
    off = align_up(off + TW * (int)sizeof(Key<SB>), 16);
    P.team_bytes = off;
    const size_t lds = (size_t)align_up(c * n, 16) + (size_t)NT * P.team_bytes;
    NMG_REQUIRE(lds <= 160 * 1024, NMG_ERR_UNSUPPORTED,
                "sparsify tile (c*g=%d columns, m=%d) needs %zu bytes of LDS, limit 163840", cols,
                m, lds);
    auto kern = sparsify_kernel<T, TW, NT>;
    if (lds > 64 * 1024)
        NMG_HIP_TRY(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)lds));
    const int64_t grid = (P.outer + NT - 1) / NT;
    NMG_REQUIRE(grid <= 0x7fffffffLL, NMG_ERR_UNSUPPORTED, "too many tiles (%lld)", (long long)grid);
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * TW * NT), lds, stream, P);
    NMG_HIP_TRY(hipGetLastError());
    return NMG_OK;
}

// ------------------------------------------------------------- small tiles: lane teams
// For tiles of a few hundred columns a wavefront-wide arg-max per step wastes most of the
// machine on communication.  Here a tile belongs to a *team* of L consecutive lanes (16 tiles
// per wavefront for L = 4); lane j of the team owns the columns o = j (mod L) and keeps the best
// of them in registers, so a step is a short scan of the owner's own columns plus log2(L)
// exchanges inside the team.
//
// Heads are maintained lazily: when a pattern fills up, the heads that point to it are left
// stale.  A stale head is an upper bound of the column's true key (the true head is the best over
// a subset of the patterns), so the largest head over the free columns is either valid -- then it
// is the true maximum and is accepted -- or stale, and then only that one column is recomputed
// over the patterns that still have room and the step is repeated.  Every iteration of a team
// is therefore one "pop": accept or repair, followed by the owner's rescan.
//
// LDS per team: the tile's data, head score (+1, 0 = column taken), head pattern, pattern
// counters and the idx output; a team region is padded to L (mod 64) words so that the teams of
// a wavefront, which all touch the same offsets of their regions, hit distinct banks.
// Exchange inside a team of L consecutive lanes without going through LDS: DPP lane
// permutations.  After the stages for L the value has been combined over the whole team:
// quad_perm [1,0,3,2] and [2,3,0,1] reduce a quad, row_half_mirror (i <-> 7-i) joins the two
// quads of 8 lanes, row_mirror (i <-> 15-i) the two halves of 16.
template <int CTRL> __device__ __forceinline__ uint32_t dpp_u32(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL> __device__ __forceinline__ uint64_t dpp_u64(uint64_t v)
{
    return ((uint64_t)dpp_u32<CTRL>((uint32_t)(v >> 32)) << 32) | dpp_u32<CTRL>((uint32_t)v);
}
template <int CTRL> __device__ __forceinline__ uint32_t dpp_bits(uint32_t v) { return dpp_u32<CTRL>(v); }
template <int CTRL> __device__ __forceinline__ uint64_t dpp_bits(uint64_t v) { return dpp_u64<CTRL>(v); }

template <int CTRL, typename SB> __device__ __forceinline__ void team_stage(Key<SB> &b)
{
    Key<SB> o;
    o.s = dpp_bits<CTRL>(b.s);
    o.op = dpp_u32<CTRL>(b.op);
    if (key_gt(o, b)) b = o;
}
template <int L, typename SB> __device__ __forceinline__ Key<SB> team_max(Key<SB> b)
{
    if (L >= 2) team_stage<0xB1>(b);    // quad_perm [1,0,3,2]
    if (L >= 4) team_stage<0x4E>(b);    // quad_perm [2,3,0,1]
    if (L >= 8) team_stage<0x141>(b);   // row_half_mirror
    if (L >= 16) team_stage<0x140>(b);  // row_mirror
    static_assert(L <= 16, "a team lives inside one DPP row of 16 lanes");
    return b;
}

struct TeamParams {
    SparsifyParams sp;
    int region_bytes;                  // LDS bytes of one team
    int t_hs, t_hp, t_cnt, t_oidx;     // offsets inside a team region
    int teams;                         // teams (= tiles) per workgroup
    uint64_t magic_cols, magic_g;      // ceil(2^32 / cols), ceil(2^32 / g): x / d == (x * magic) >> 32 for x < 2^16
};

template <typename T, int L, bool SMALLC>
__global__ __launch_bounds__(128) void sparsify_teams_kernel(TeamParams Q)
{
    using CT = typename ScoreOf<T>::type;
    using SB = typename ScoreOf<T>::bits;
    const SparsifyParams &P = Q.sp;
    extern __shared__ __align__(16) unsigned char smem[];

    const int n = P.n, m = P.m, g = P.g, c = P.c, cols = P.cols;
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int team = tid / L, tl = tid % L;
    const int teams = Q.teams;

    // LDS: [order table][pattern masks (m <= 8)][team regions]
    int8_t *s_order = (int8_t *)smem;
    uint8_t *s_mask = (uint8_t *)(smem + ((c * n + 15) & ~15));
    const int order_bytes = ((c * n + 15) & ~15) + ((c + 15) & ~15);
    unsigned char *region = smem + order_bytes + (size_t)team * Q.region_bytes;
    T *s_d = (T *)region;
    SB *s_hs = (SB *)(region + Q.t_hs);
    uint16_t *s_hp = (uint16_t *)(region + Q.t_hp);
    int16_t *s_cnt = (int16_t *)(region + Q.t_cnt);
    int16_t *s_oidx = (int16_t *)(region + Q.t_oidx);

    for (int i = tid; i < c * n; i += nthr) s_order[i] = P.order[i];
    if (m <= 8)
        for (int p = tid; p < c; p += nthr) {
            int mk = 0;
            for (int j = 0; j < n; j++) mk |= 1 << P.order[p * n + j];
            s_mask[p] = (uint8_t)mk;
        }

    // ---- cooperative load of the workgroup's tiles (zero beyond G / S); consecutive threads
    //      take the same column of consecutive tiles, which are adjacent along the sparse dim ----
    const int64_t tile0 = (int64_t)blockIdx.x * teams;
    const T *dense = (const T *)P.dense;
    const int64_t tiles_per_b = P.view.num_chunks * P.view.num_blocks;
    // A thread keeps one (tile, position r) pair and walks the tile's columns, so the 64-bit
    // index arithmetic is done once per pair and the loads of the walk are independent.
    for (int pair = tid; pair < teams * m; pair += nthr) {
        const int tm = pair / m, r = pair - tm * m;
        const int64_t t = tile0 + tm;
        T *dst = (T *)(smem + order_bytes + (size_t)tm * Q.region_bytes) + r;
        const T *src = nullptr;
        int valid_cols = 0;
        if (t < P.outer) {
            const int64_t b = t / tiles_per_b;
            const int64_t rem = t - b * tiles_per_b;
            const int64_t kc = rem / P.view.num_blocks;
            const int64_t mb = rem - kc * P.view.num_blocks;
            const int64_t si = mb * m + r;
            if (si < P.view.S) {
                src = dense + b * P.view.stride_b + kc * cols * P.view.stride_g + si * P.view.stride_s;
                const int64_t left = P.view.G - kc * cols;
                valid_cols = left < cols ? (int)left : cols;
            }
        }
        const int64_t sg = P.view.stride_g;
#pragma unroll 8
        for (int o = 0; o < cols; o++) dst[o * m] = o < valid_cols ? src[o * sg] : Zero<T>::v();
    }
    if (team < teams)
        for (int p = tl; p < c; p += L) s_cnt[p] = 0;
    __syncthreads();

    const bool live = team < teams && tile0 + team < P.outer;

    // SMALLC (at most 8 patterns, m <= 8, g <= 255): the pattern masks and the pattern counters
    // (8 bits each, packed) stay in registers of every lane of the team -- all lanes see every
    // accepted (column, pattern) -- so neither the staleness test nor a repair waits for LDS
    // beyond the read of the column itself.
    int mk_r[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    uint64_t cnt64 = 0;
    if (SMALLC) {
#pragma unroll
        for (int p = 0; p < 8; p++) mk_r[p] = p < c ? (int)s_mask[p] : 0;
    }
    auto cnt_of = [&](int p) { return (int)((cnt64 >> (8 * p)) & 0xFF); };

    // Best key of column o over the patterns that still have room: score bits + 1 and pattern.
    // LDS reads are issued in batches of independent loads (the column first, then 8 patterns'
    // masks and counters at a time): the loop is latency-bound, not throughput-bound.
    auto head_of = [&](int o, SB &best_s, int &best_p) {
        best_p = 0;
        best_s = 0;
        const T *col = s_d + o * m;
        if (SMALLC) {
            CT a[8];
#pragma unroll
            for (int r = 0; r < 8; r++) a[r] = score_of(col[r < m ? r : 0]);
#pragma unroll
            for (int p = 0; p < 8; p++) {
                if (p >= c || cnt_of(p) >= g) continue;
                CT acc = 0;
#pragma unroll
                for (int r = 0; r < 8; r++) {
                    if (r >= m) break;
                    if ((mk_r[p] >> r) & 1) acc += a[r];
                }
                const SB sb = score_bits(acc) + 1;
                if (sb >= best_s) {
                    best_s = sb;
                    best_p = p;
                }
            }
            return;
        }
        if (m <= 8) {
            CT a[8];
#pragma unroll
            for (int r = 0; r < 8; r++) a[r] = score_of(col[r < m ? r : 0]);
            for (int p0 = 0; p0 < c; p0 += 8) {
                int mk[8], cn[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int p = p0 + i < c ? p0 + i : c - 1;
                    mk[i] = s_mask[p];
                    cn[i] = s_cnt[p];
                }
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if (p0 + i >= c || cn[i] >= g) continue;
                    // left-to-right sum over the pattern's positions (ascending), as the reference
                    CT acc = 0;
#pragma unroll
                    for (int r = 0; r < 8; r++) {
                        if (r >= m) break;
                        if ((mk[i] >> r) & 1) acc += a[r];
                    }
                    const SB sb = score_bits(acc) + 1;
                    if (sb >= best_s) {  // ties: larger p wins
                        best_s = sb;
                        best_p = p0 + i;
                    }
                }
            }
            return;
        }
        for (int p = 0; p < c; p++) {
            if (s_cnt[p] >= g) continue;
            CT acc = 0;
            for (int j = 0; j < n; j++) acc += score_of(col[s_order[p * n + j]]);
            const SB sb = score_bits(acc) + 1;
            if (sb >= best_s) {
                best_s = sb;
                best_p = p;
            }
        }
    };
    // Largest head among this lane's free columns (ties: larger o wins); s == 0 when none is left.
    // A lane owns at most 32 columns (the launcher picks L accordingly), kept as 4 groups of 8
    // whose maxima live in registers: a change rescans one group only.
    SB gs[4] = {0, 0, 0, 0};
    int go[4] = {0, 0, 0, 0};   // column << 16 | pattern of the group's best head
    auto scan_group = [&](int k) {
        SB v[8];
        int hp[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int o = tl + L * (k * 8 + i);
            v[i] = s_hs[o < cols ? o : tl];
            hp[i] = s_hp[o < cols ? o : tl];
        }
        // pairwise (tree) reduction; on equal scores the larger column, i.e. the later entry, wins
        SB bs[8];
        int bo[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int o = tl + L * (k * 8 + i);
            bs[i] = o < cols ? v[i] : 0;
            bo[i] = (o << 16) | hp[i];
        }
#pragma unroll
        for (int w = 1; w < 8; w <<= 1)
#pragma unroll
            for (int i = 0; i < 8; i += 2 * w)
                if (bs[i + w] >= bs[i] && bs[i + w] != 0) {
                    bs[i] = bs[i + w];
                    bo[i] = bo[i + w];
                }
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (q == k) {
                gs[q] = bs[0];
                go[q] = bo[0];
            }
    };
    auto local_best = [&]() {
        Key<SB> lb;
        lb.s = 0;
        lb.op = 0;
        SB best_s = 0;
        int best_op = 0;
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (gs[q] != 0 && gs[q] >= best_s) {
                best_s = gs[q];
                best_op = go[q];
            }
        lb.s = best_s;
        lb.op = best_s != 0 ? (uint32_t)best_op : 0u;
        return lb;
    };

    Key<SB> lb;
    lb.s = 0;
    lb.op = 0;
    if (live) {
        for (int o = tl; o < cols; o += L) {
            SB bs;
            int bp;
            head_of(o, bs, bp);
            s_hs[o] = bs;
            s_hp[o] = (uint16_t)bp;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) scan_group(k);
        lb = local_best();
    }

    // Every column is accepted once and repaired at most once per pattern that fills up, which
    // bounds the loop whatever the data.
    int accepted = live ? 0 : cols;
    const int max_iter = cols * (c + 1);
    for (int iter = 0; iter < max_iter && __any(accepted < cols); iter++) {
        if (accepted < cols) {
            // ---- team arg-max ----
            const Key<SB> b = team_max<L>(lb);
            const int o_star = (int)(b.op >> 16), p_star = (int)(b.op & 0xFFFFu);
            const int cntp = SMALLC ? cnt_of(p_star) : (int)s_cnt[p_star];
            const bool stale = cntp >= g;
            if (SMALLC && !stale) cnt64 += (uint64_t)1 << (8 * p_star);
            if (o_star % L == tl) {
                if (stale) {
                    SB bs;
                    int bp;
                    head_of(o_star, bs, bp);
                    s_hs[o_star] = bs;
                    s_hp[o_star] = (uint16_t)bp;
                } else {
                    if (!SMALLC) s_cnt[p_star] = (int16_t)(cntp + 1);
                    s_hs[o_star] = 0;
                    s_oidx[p_star * g + cntp] = (int16_t)o_star;
                }
                scan_group((o_star / L) >> 3);
                lb = local_best();
            }
            if (!stale) accepted++;
        }
        // the team's LDS writes must be visible to its other lanes in the next iteration
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    // ---- coalesced store of the workgroup's tiles: one thread per slot writes its index and
    //      gathers its n values from the tile data (divisions by multiplication: e < 2^16) ----
    __syncthreads();
    T *val = (T *)P.val;
    for (int e = tid; e < teams * cols; e += nthr) {
        const int tm = (int)(((uint64_t)e * Q.magic_cols) >> 32), slot = e - tm * cols;
        const int64_t t = tile0 + tm;
        if (t >= P.outer) break;
        const unsigned char *reg = smem + order_bytes + (size_t)tm * Q.region_bytes;
        const int o = ((const int16_t *)(reg + Q.t_oidx))[slot];
        const int p = (int)(((uint64_t)slot * Q.magic_g) >> 32);
        const T *col = (const T *)reg + o * m;
        const int64_t at = t * (int64_t)cols + slot;
        P.idx[at] = (int16_t)o;
        for (int j = 0; j < n; j++) val[at * n + j] = col[s_order[p * n + j]];
    }
}

template <typename T, int L> static int launch_sparsify_teams(SparsifyParams &P, hipStream_t stream, bool *done)
{
    using SB = typename ScoreOf<T>::bits;
    *done = false;
    TeamParams Q{};
    Q.sp = P;
    const int cols = P.cols, m = P.m, c = P.c, n = P.n;
    int off = align_up(cols * m * (int)sizeof(T), 8);
    Q.t_hs = off;
    off = align_up(off + cols * (int)sizeof(SB), 4);
    Q.t_hp = off;
    off = align_up(off + cols * 2, 4);
    Q.t_cnt = off;
    off = align_up(off + c * 2, 4);
    Q.t_oidx = off;
    off = align_up(off + cols * 2, 4);
    // region size = L (mod 64) words spreads the teams of a wavefront over the banks; regions of
    // 8-byte data stay 8-byte aligned (an even number of words)
    int words = off / 4, target = L % 64;
    if ((sizeof(T) == 8 || sizeof(SB) == 8) && (target & 1)) target++;
    while (words % 64 != target) words++;
    Q.region_bytes = words * 4;
    const size_t order_bytes = (size_t)align_up(c * n, 16) + (size_t)align_up(c, 16);
    // workgroups of 128 threads when two of them fit in a CU's LDS, else 64 threads
    int threads = 128;
    size_t lds = order_bytes + (size_t)(threads / L) * Q.region_bytes;
    if (lds > 80 * 1024) {
        threads = 64;
        lds = order_bytes + (size_t)(threads / L) * Q.region_bytes;
    }
    if (lds > 160 * 1024) return NMG_OK;   // too large for this kernel: the caller falls back
    Q.teams = threads / L;
    Q.magic_cols = (((uint64_t)1 << 32) + cols - 1) / cols;
    Q.magic_g = (((uint64_t)1 << 32) + P.g - 1) / P.g;
    const bool smallc = c <= 8 && m <= 8 && P.g <= 255;
    auto kern = smallc ? sparsify_teams_kernel<T, L, true> : sparsify_teams_kernel<T, L, false>;
    if (lds > 64 * 1024)
        NMG_HIP_TRY(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)lds));
    const int64_t grid = (P.outer + Q.teams - 1) / Q.teams;
    NMG_REQUIRE(grid <= 0x7fffffffLL, NMG_ERR_UNSUPPORTED, "too many tiles (%lld)", (long long)grid);
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(threads), lds, stream, Q);
    NMG_HIP_TRY(hipGetLastError());
    *done = true;
    return NMG_OK;
}

static int match_tiles(const SparsifyParams &P, const float *d, hipStream_t s, bool *done)
{
    return match_f32(d, P.val, P.idx, P.view, P.outer, P.n, P.m, P.g, P.c, P.cols, s, done);
}
static int match_tiles(const SparsifyParams &P, const __half *d, hipStream_t s, bool *done)
{
    return match_f16(d, P.val, P.idx, P.view, P.outer, P.n, P.m, P.g, P.c, P.cols, s, done);
}
static int match_tiles(const SparsifyParams &P, const __hip_bfloat16 *d, hipStream_t s, bool *done)
{
    return match_bf16(d, P.val, P.idx, P.view, P.outer, P.n, P.m, P.g, P.c, P.cols, s, done);
}
static int match_tiles(const SparsifyParams &, const double *, hipStream_t, bool *) { return NMG_OK; }      // 64-bit scores

template <typename T> static int dispatch_sparsify(SparsifyParams &P, hipStream_t stream)
{
    // Tiles of at least 16 columns with at most 128 patterns of at most 8 positions: nmg_match.h.  Most smaller tiles are
    // faster in the lane teams (4096 x 4096 fp16, teams / matching: 1:2:4 201 / 265 us, 1:8:1 163 / 203, 1:4:2 165 / 206, 2:3:5
    // 164 / 186, 2:4:2 188 / 181, 4:5:3 281 / 146; from 16 columns on 1:2:8 179 / 148, 1:4:4 256 / 121, 2:4:4 312 / 116).
    bool matched = false;
    if (int rc = match_tiles(P, (const T *)P.dense, stream, &matched)) return rc;
    if (matched) return NMG_OK;
    // The rest (tiles of fewer than 16 columns, double, m > 8, more than 128
    // patterns) goes step by step: lane teams for tiles of up to 512 columns, else one
    // wavefront per tile (four tiles per workgroup) or four wavefronts per tile -- more of them
    // lose to the two workgroup barriers of every step (measured on 896-column tiles: 1 / 2 / 4 /
    // 8 / 16 wavefronts -> 17.6 / 12.6 / 10.9 / 21.1 / 69 ms for an 8192 x 8192 weight).
    if (P.cols <= 512 && P.n > 0) {
        // lane teams: about 16 to 32 columns per lane
        bool done = false;
        int rc;
        if (P.cols <= 32) rc = launch_sparsify_teams<T, 1>(P, stream, &done);
        else if (P.cols <= 64) rc = launch_sparsify_teams<T, 2>(P, stream, &done);
        else if (P.cols <= 128) rc = launch_sparsify_teams<T, 4>(P, stream, &done);
        else if (P.cols <= 256) rc = launch_sparsify_teams<T, 8>(P, stream, &done);
        else rc = launch_sparsify_teams<T, 16>(P, stream, &done);
        if (rc != NMG_OK || done) return rc;
    }
    if (P.cols <= 128) return launch_sparsify<T, 1, 4>(P, stream);
    return launch_sparsify<T, 4, 1>(P, stream);
}

static int check_common(const nmg_view *view, int n, int m, int g, int dtype, TileGeom *tg)
{
    NMG_REQUIRE(view != nullptr, NMG_ERR_ARG, "null view");
    NMG_REQUIRE(m >= 1 && m <= 64 && n >= 0 && n <= m && g >= 1, NMG_ERR_ARG,
                "invalid n:m:g = %d:%d:%d", n, m, g);
    NMG_REQUIRE(dtype_size(dtype) != 0, NMG_ERR_ARG, "invalid dtype code %d", dtype);
    NMG_REQUIRE(view->batch >= 0 && view->G >= 0 && view->S >= 0, NMG_ERR_ARG, "negative extent");
    int64_t c = binom(m, n);
    NMG_REQUIRE(c * g < 32768, NMG_ERR_ARG,
                "chunk_size * group_size = %lld must be < 2^15 (int16 indices)", (long long)(c * g));
    *tg = tile_geom(*view, n, m, g);
    return NMG_OK;
}

static ViewDev view_dev(const nmg_view &v, const TileGeom &tg)
{
    ViewDev d;
    d.G = v.G;
    d.S = v.S;
    d.stride_b = v.stride_b;
    d.stride_g = v.stride_g;
    d.stride_s = v.stride_s;
    d.num_chunks = tg.num_chunks;
    d.num_blocks = tg.num_blocks;
    return d;
}

// ------------------------------------------------------------------ element-wise companions

struct ScatterParams {
    const void *val;
    const int16_t *idx;
    void *dense;
    const int8_t *order;
    ViewDev view;
    int64_t outer;
    int n, m, g, c, cols;
};

// One thread per slot: writes the m values of its column (kept ones + zeros), so every element
// of the view is written exactly once (idx is a permutation of the tile's columns).
template <typename T> __global__ void to_dense_kernel(ScatterParams P)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= P.outer * P.cols) return;
    const int64_t t = gid / P.cols;
    const int slot = (int)(gid - t * P.cols);
    const int p = slot / P.g;
    const int o = P.idx[gid];
    if (o < 0 || o >= P.cols) return;
    const int64_t tiles_per_b = P.view.num_chunks * P.view.num_blocks;
    const int64_t b = t / tiles_per_b;
    const int64_t rem = t - b * tiles_per_b;
    const int64_t kc = rem / P.view.num_blocks, mb = rem - kc * P.view.num_blocks;
    const int64_t gi = kc * P.cols + o;
    if (gi >= P.view.G) return;
    const T *v = (const T *)P.val + gid * P.n;
    T *base = (T *)P.dense + b * P.view.stride_b + gi * P.view.stride_g;
    int j = 0;
    for (int r = 0; r < P.m; r++) {
        T x = Zero<T>::v();
        if (j < P.n && P.order[p * P.n + j] == r) x = v[j++];
        const int64_t si = mb * P.m + r;
        if (si < P.view.S) base[si * P.view.stride_s] = x;
    }
}

template <typename T> __global__ void gather_kernel(ScatterParams P)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= P.outer * P.cols) return;
    const int64_t t = gid / P.cols;
    const int slot = (int)(gid - t * P.cols);
    const int p = slot / P.g;
    const int o = P.idx[gid];
    const int64_t tiles_per_b = P.view.num_chunks * P.view.num_blocks;
    const int64_t b = t / tiles_per_b;
    const int64_t rem = t - b * tiles_per_b;
    const int64_t kc = rem / P.view.num_blocks, mb = rem - kc * P.view.num_blocks;
    const int64_t gi = kc * P.cols + o;
    T *v = (T *)P.val + gid * P.n;  // here val is the output
    const T *base = (const T *)P.dense + b * P.view.stride_b + gi * P.view.stride_g;
    for (int j = 0; j < P.n; j++) {
        const int64_t si = mb * P.m + P.order[p * P.n + j];
        T x = Zero<T>::v();
        if (o >= 0 && gi < P.view.G && si < P.view.S) x = base[si * P.view.stride_s];
        v[j] = x;
    }
}

struct RowpackParams {
    const void *val;
    const int16_t *idx;
    void *pk_val;
    void *pk_pat;
    int64_t G, nb, num_chunks, outer;
    int n, g, c, cols, pat_bytes;
};

template <typename T> __global__ void rowpack_kernel(RowpackParams P)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= P.outer * P.cols) return;
    const int64_t t = gid / P.cols;
    const int slot = (int)(gid - t * P.cols);
    const int p = slot / P.g;
    const int o = P.idx[gid];
    const int64_t kc = t / P.nb, mb = t - kc * P.nb;
    const int64_t q = kc * P.cols + o;
    if (o < 0 || q >= P.G) return;
    const T *v = (const T *)P.val + gid * P.n;
    T *dst = (T *)P.pk_val + (q * P.nb + mb) * P.n;
    for (int j = 0; j < P.n; j++) dst[j] = v[j];
    if (P.pat_bytes == 1)
        ((uint8_t *)P.pk_pat)[q * P.nb + mb] = (uint8_t)p;
    else
        ((uint16_t *)P.pk_pat)[q * P.nb + mb] = (uint16_t)p;
}

}  // namespace nmg

using namespace nmg;

extern "C" int nmg_sparsify(const void *d_dense, const nmg_view *view, void *d_val, int16_t *d_idx,
                            int n, int m, int g, int dtype, void *stream)
{
    TileGeom tg;
    if (int rc = check_common(view, n, m, g, dtype, &tg)) return rc;
    if (tg.outer == 0) return NMG_OK;
    NMG_REQUIRE(d_dense && d_val && d_idx, NMG_ERR_ARG, "null device pointer");
    SparsifyParams P{};
    P.dense = d_dense;
    P.val = d_val;
    P.idx = d_idx;
    if (int rc = device_order(n, m, &P.order)) return rc;
    P.view = view_dev(*view, tg);
    P.outer = tg.outer;
    P.n = n;
    P.m = m;
    P.g = g;
    P.c = tg.c;
    P.cols = tg.cols;
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
    case NMG_F32: return dispatch_sparsify<float>(P, s);
    case NMG_F16: return dispatch_sparsify<__half>(P, s);
    case NMG_BF16: return dispatch_sparsify<__hip_bfloat16>(P, s);
    case NMG_F64: return dispatch_sparsify<double>(P, s);
    }
    return NMG_ERR_ARG;
}

template <template <typename> class K> struct Launch;

// Tiled forms of the two kernels above for views whose sparse dim is contiguous (the layout of
// a weight with n:m blocks along its rows' direction).  There a tile is c*g lines x m positions:
// one slot's m values are a few bytes of a line, so the slot-per-thread kernels touch every cache
// line of the dense tensor many times.  Here a workgroup takes NT tiles that are neighbours along
// the sparse dim -- a region of c*g lines x NT*m contiguous positions -- and moves it through
// LDS: rows of the region go to / come from global memory as contiguous segments, val / idx are
// contiguous for the NT tiles anyway.
struct TiledParams {
    ScatterParams sp;
    int nt;                      // tiles per workgroup
    int pitch;                   // elements per region row in LDS
    int groups_per_chunk;        // workgroups along the sparse dim
    int runs;                    // an XCD's workgroups are neighbours
    uint64_t magic_cols, magic_g;
};

// GC: the group dim is the contiguous one instead (the reference's default orientation of a Linear
// weight).  The region of NT tiles that are neighbours along the sparse dim is then NT*m rows (one
// per position) of c*g contiguous columns; LDS holds it as [position][column].
template <typename T, bool GATHER, bool GC>
__global__ __launch_bounds__(1024) void scatter_tiled_kernel(TiledParams Q)
{
    const ScatterParams &P = Q.sp;
    extern __shared__ __align__(16) unsigned char smem[];
    T *tile = (T *)smem;
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int n = P.n, m = P.m, cols = P.cols, nt = Q.nt, pitch = Q.pitch;
    // workgroup -> (batch, group-dim chunk, first block)
    const int64_t wg = Q.runs ? xcd_run(blockIdx.x, gridDim.x) : blockIdx.x;
    const int64_t chunk_id = wg / Q.groups_per_chunk;
    const int64_t mb0 = (wg - chunk_id * Q.groups_per_chunk) * nt;
    const int64_t b = chunk_id / P.view.num_chunks, kc = chunk_id - b * P.view.num_chunks;
    const int64_t t0 = (b * P.view.num_chunks + kc) * P.view.num_blocks + mb0;
    const int tiles = (int)min((int64_t)nt, P.view.num_blocks - mb0);
    const int64_t g0 = kc * cols, s0 = mb0 * m;
    // region: `all_rows` rows of `width` contiguous elements; rows / valid_w of them exist
    const int width = GC ? cols : tiles * m;
    const int all_rows = GC ? tiles * m : cols;
    const int rows = GC ? (int)max((int64_t)0, min((int64_t)all_rows, P.view.S - s0))
                        : (int)min((int64_t)cols, P.view.G - g0);
    const int valid_w = GC ? (int)min((int64_t)cols, P.view.G - g0)
                           : (int)max((int64_t)0, min((int64_t)width, P.view.S - s0));
    const int64_t row_stride = GC ? P.view.stride_s : P.view.stride_g;
    T *dense = (T *)P.dense + b * P.view.stride_b + g0 * P.view.stride_g + s0 * P.view.stride_s;
    constexpr int V = 16 / sizeof(T);
    const bool vec = (row_stride % V) == 0 && ((GC ? g0 : s0) % V) == 0 && (P.view.stride_b % V) == 0 &&
                     ((uintptr_t)P.dense % 16) == 0 && (pitch % V) == 0;
    const int wv = (width + V - 1) / V;

    if (GATHER) {
        // region -> LDS (zeros beyond G / S)
        for (int i = tid; i < all_rows * wv; i += nthr) {
            const int r = i / wv, cc = (i - r * wv) * V;
            T *dst = tile + r * pitch + cc;
            const T *src = dense + (int64_t)r * row_stride + cc;
            if (vec && r < rows && cc + V <= valid_w) {
                *(uint4 *)dst = *(const uint4 *)src;
            } else {
                for (int e = 0; e < V && cc + e < pitch; e++)
                    dst[e] = (r < rows && cc + e < valid_w) ? src[e] : Zero<T>::v();
            }
        }
    } else {
        const uint4 z = {0, 0, 0, 0};
        for (int i = tid; i < all_rows * pitch * (int)sizeof(T) / 16; i += nthr) ((uint4 *)tile)[i] = z;
    }
    // the order table in LDS where it fits: a slot's positions are then one LDS read away instead
    // of a round trip to L2 behind the load of its index
    __shared__ int8_t s_ord[1024];
    const bool ord_lds = P.c * n <= 1024;
    if (ord_lds)
        for (int i = tid; i < P.c * n; i += nthr) s_ord[i] = P.order[i];
    const int8_t *order = ord_lds ? s_ord : P.order;
    __syncthreads();
    // slots of the NT tiles: contiguous in val / idx (slot e of the workgroup is element
    // t0 * cols + e).  Four slots per thread are loaded before the first is used: index -> LDS ->
    // store is otherwise one round trip to HBM per slot and thread.
    const int total = tiles * cols;
    const int64_t at0 = t0 * (int64_t)cols;
    // NV > 0: n is the constant NV and a slot's NV values are one aligned word of 4 or 8 bytes -- one
    // load (issued with the index loads) or store per slot instead of NV of 2 or 4 bytes; NV = 0:
    // any n, value by value.
    auto run_slots = [&](auto nv_tag) {
        constexpr int NV = decltype(nv_tag)::value;
        constexpr int WB = NV * (int)sizeof(T);            // bytes of a slot's word
        using Word = typename std::conditional<WB == 8, uint2, uint32_t>::type;
        for (int base = tid; base < total; base += 4 * nthr) {
            int o[4];
            Word vw[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int e = base + u * nthr;
                o[u] = e < total ? (int)P.idx[at0 + e] : -1;
                if (!GATHER && NV > 0) vw[u] = ((const Word *)P.val)[at0 + (e < total ? e : 0)];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int e = base + u * nthr;
                if (e >= total) continue;
                const int tm = (int)(((uint64_t)e * Q.magic_cols) >> 32), slot = e - tm * cols;
                const int p = (int)(((uint64_t)slot * Q.magic_g) >> 32);
                const bool ok = o[u] >= 0 && o[u] < cols;
                T *v = (T *)P.val + (at0 + e) * n;
                // element (column oc, position ps of tile tm) of the region
                const int oc = ok ? o[u] : 0;
                auto at = [&](int ps) { return GC ? (tm * m + ps) * pitch + oc : oc * pitch + tm * m + ps; };
                if constexpr (NV > 0) {
                    T w[NV];
                    if (GATHER) {
#pragma unroll
                        for (int j = 0; j < NV; j++) w[j] = ok ? tile[at(order[p * NV + j])] : Zero<T>::v();
                        Word raw;
                        __builtin_memcpy(&raw, w, WB);
                        ((Word *)P.val)[at0 + e] = raw;
                    } else if (ok) {
                        __builtin_memcpy(w, &vw[u], WB);
#pragma unroll
                        for (int j = 0; j < NV; j++) tile[at(order[p * NV + j])] = w[j];
                    }
                } else {
                    if (GATHER) {
                        for (int j = 0; j < n; j++) v[j] = ok ? tile[at(order[p * n + j])] : Zero<T>::v();
                    } else if (ok) {
                        for (int j = 0; j < n; j++) tile[at(order[p * n + j])] = v[j];
                    }
                }
            }
        }
    };
    const int vbytes = n * (int)sizeof(T);
    const bool aligned = ((uintptr_t)P.val % 8) == 0;
    if (aligned && vbytes == 4 && n == 1) run_slots(std::integral_constant<int, (sizeof(T) == 4 ? 1 : 0)>{});
    else if (aligned && vbytes == 4 && n == 2) run_slots(std::integral_constant<int, (sizeof(T) == 2 ? 2 : 0)>{});
    else if (aligned && vbytes == 8 && n == 2) run_slots(std::integral_constant<int, (sizeof(T) == 4 ? 2 : 0)>{});
    else if (aligned && vbytes == 8 && n == 4) run_slots(std::integral_constant<int, (sizeof(T) == 2 ? 4 : 0)>{});
    else run_slots(std::integral_constant<int, 0>{});
    if (GATHER) return;
    __syncthreads();
    // LDS -> region
    for (int i = tid; i < rows * wv; i += nthr) {
        const int r = i / wv, cc = (i - r * wv) * V;
        if (cc >= valid_w) continue;
        const T *src = tile + r * pitch + cc;
        T *dst = dense + (int64_t)r * row_stride + cc;
        if (vec && cc + V <= valid_w) {
            *(uint4 *)dst = *(const uint4 *)src;
        } else {
            for (int e = 0; e < V && cc + e < valid_w; e++) dst[e] = src[e];
        }
    }
}

// Launches the tiled kernel when it applies; *done tells whether it did.
template <typename T>
static int launch_scatter_tiled(bool gather, ScatterParams &P, hipStream_t s, bool *done)
{
    *done = false;
    const bool gc = P.view.stride_s != 1 && P.view.stride_g == 1;   // group dim contiguous
    if ((P.view.stride_s != 1 && !gc) || P.view.num_blocks < 4) return NMG_OK;
    // Tiles per workgroup: about 8 KiB of LDS (many small workgroups overlap each other's
    // latencies: a 16384 x 4096 2:4:16 gather takes 81 us with 10 tiles, 112 us with 64), but at
    // least 8 tiles so that a row of the region is a decent run of bytes, or 4 where 8 do not fit
    // (2:8:32 with 8 tiles of 896 lines: 139 us against 760 us for the slot-per-thread kernel).
    const int V = 16 / (int)sizeof(T);
    const int64_t per_tile = (int64_t)P.cols * P.m * (int64_t)sizeof(T);
    int nt = (int)std::min<int64_t>(64, (8 * 1024) / per_tile);
    if (nt < 8) nt = 8;
    // whole 128-byte lines of the dense rows where enough workgroups stay (4096^2 2:4:16 fp16 gather / scatter with 10 tiles 21.4 / 16.2
    // us, with 16 15.2 / 14.5; 640 x 512 4.4 / 4.0 against 5.0 / 4.5)
    const int64_t chunks = P.outer / P.view.num_blocks;   // batches x group-dim chunks
    const int line = (int)(128 / (P.m * (int64_t)sizeof(T)));
    if (!gc && 128 % (P.m * (int)sizeof(T)) == 0 && nt < line && nt * 2 > line && chunks * (P.view.num_blocks / line) >= 512) nt = line;
    nt = (int)std::min<int64_t>(nt, P.view.num_blocks);
    auto pitch_of = [&](int tiles, bool pad) { return (((gc ? P.cols : tiles * P.m) + V - 1) / V) * V + (pad ? V : 0); };
    bool pad = true;
    auto lds_of = [&](int tiles, bool pd) {
        return (size_t)(gc ? tiles * P.m : P.cols) * pitch_of(tiles, pd) * sizeof(T);
    };
    // Tiles of many columns.  Small tensors, about what the caches of a few CUs hold, have too few workgroups of them: a slot per thread is ahead
    // (4:8:32 fp32 1001^2, along the blocks, gather / dense 8.4 / 10.3 against 13.5 / 12.5 us; 2048 x 1536 25 / 42 against 15 / 14).
    const double mi = (double)P.view.G * (double)P.view.S * (double)(P.outer / (P.view.num_blocks * P.view.num_chunks)) / (1 << 20);
    if (per_tile > (gc && gather ? 16 : 32) * 1024 && mi <= (gather ? 2.5 : gc ? 0.5 : 1.5)) return NMG_OK;
    // Group dim contiguous: a row of the region is long however few tiles there are, so as many as keep several workgroups on a CU.  Else the
    // rows are runs of the tiles' positions: 4 tiles, or 2 where 4 take nearly all of the LDS (dense: with a row's padding more than it).
    // us, gather / dense, before -> this: 4:8:32 fp32 3712 x 3584 group dim contiguous (a slot per thread) 69 / 102 -> 25 / 31, else
    // 97 / 156 -> 35 / 31; 12160 x 1408 bf16 38 / 20 (4 tiles) -> 18 / 17, 37 / 28 -> 34 / 24; 2:8:32 8192^2 fp16 55 / 51 (4 / 8 tiles)
    // -> 52 / 44, 2048 x 1536 fp32 8.0 / 8.4 -> 6.7 / 6.8.  13 patterns x 9 sizes, two types, both dims: 0.86 of the time with 8 or 4 tiles or a slot
    // per thread, at the most 1.12 of it (2:8:32 fp32 4096 x 1024 dense 9.5 -> 10.6).
    if (gc && per_tile * 8 > 48 * 1024) nt = (int)std::min<int64_t>(nt, std::max<int64_t>(1, 32 * 1024 / per_tile));
    if (!gc && lds_of(nt, pad) > 150 * 1024) nt = (int)std::min<int64_t>(4, P.view.num_blocks);
    // (rows that do not lie on 16 bytes are read and written element by element, and longer runs are then ahead: 4:8:32 fp16 12971 x 2722
    // gather 116, with 2 tiles 124; dense 117, 127)
    const bool odd_rows = !gc && P.view.stride_g * (int64_t)sizeof(T) % 16 != 0, four = odd_rows && lds_of(nt, false) <= 150 * 1024 && nt >= 4;
    if (!gc && !four && lds_of(nt, pad) > (gather ? 128 : 150) * 1024) nt = 2;
    if (lds_of(nt, pad) > 150 * 1024) pad = false;    // rows without the vector of padding
    if (lds_of(nt, pad) > 150 * 1024) return NMG_OK;
    TiledParams Q{};
    Q.sp = P;
    Q.nt = nt;
    Q.pitch = pitch_of(nt, pad);
    Q.groups_per_chunk = (int)((P.view.num_blocks + nt - 1) / nt);
    // Runs that are no whole lines of 128 bytes share their lines with the next workgroup's: one XCD for both.  us, gather, dealt
    // round-robin -> this: 4:8:32 12160 x 1408 bf16 (runs of 32 bytes) 34 -> 23, 3712 x 3584 fp32 (64) 35 -> 32, 3:6:12 9216 x 4608 fp16 (96) 52 -> 45;
    // whole lines lose: 2:4:16 16384 x 4096 58 -> 64.  Dense only the short runs, 4:8:32 4096^2 fp16 22.4 -> 20.5; else it loses, 3:6:50 fp32 1024 x
    // 4096 17.0 -> 20.0, 2:4:64 fp16 2048 x 1536 7.0 -> 7.5.
    Q.runs = !gc && !odd_rows && nt * P.m * (int)sizeof(T) % 128 != 0 && (gather || (nt == 2 && sizeof(T) == 2)) ? 1 : 0;
    Q.magic_cols = (((uint64_t)1 << 32) + P.cols - 1) / P.cols;
    Q.magic_g = (((uint64_t)1 << 32) + P.g - 1) / P.g;
    const size_t lds = lds_of(nt, pad);
    if ((int64_t)nt * P.cols >= 65536) return NMG_OK;
    const int64_t grid = chunks * Q.groups_per_chunk;
    if (grid > 0x7fffffffLL) return NMG_OK;
    auto kern = gc ? (gather ? scatter_tiled_kernel<T, true, true> : scatter_tiled_kernel<T, false, true>)
                   : (gather ? scatter_tiled_kernel<T, true, false> : scatter_tiled_kernel<T, false, false>);
    if (lds > 64 * 1024)
        NMG_HIP_TRY(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    // Large regions leave few workgroups on a CU: as many threads as it can use.  us, gather / scatter, 256 threads -> this, fp16:
    // 2:8:32 8192^2 141 / 81 -> 57 / 44, 14152 x 1192 45 / 29 -> 21 / 18; 4:8:32 4096^2 37 / 24 -> 24 / 19; 3:6:12 4096^2 27 / 23 -> 22 / 20;
    // 1:8:32 2584 x 1472 9.4 / 8.4 -> 6.3 / 6.4.  At 2:4:16 (8 to 12 KB) more threads lose: 4096^2 21 / 16 -> 21 / 22.
    const int threads = lds >= 48 * 1024 ? 1024 : lds >= 16 * 1024 ? 512 : 256;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(threads), lds, s, Q);
    NMG_HIP_TRY(hipGetLastError());
    *done = true;
    return NMG_OK;
}

static int launch_scatter(bool gather, const void *dense, const nmg_view *view, const void *val,
                          const int16_t *idx, int n, int m, int g, int dtype, void *stream)
{
    TileGeom tg;
    if (int rc = check_common(view, n, m, g, dtype, &tg)) return rc;
    if (tg.outer == 0) return NMG_OK;
    NMG_REQUIRE(dense && val && idx, NMG_ERR_ARG, "null device pointer");
    ScatterParams P{};
    P.val = val;
    P.idx = idx;
    P.dense = (void *)dense;
    if (int rc = device_order(n, m, &P.order)) return rc;
    P.view = view_dev(*view, tg);
    P.outer = tg.outer;
    P.n = n;
    P.m = m;
    P.g = g;
    P.c = tg.c;
    P.cols = tg.cols;
    const int64_t total = tg.outer * tg.cols;
    const int bs = 256;
    const int64_t grid = (total + bs - 1) / bs;
    NMG_REQUIRE(grid <= 0x7fffffffLL, NMG_ERR_UNSUPPORTED, "too many slots");
    hipStream_t s = (hipStream_t)stream;
    {
        bool done = false;
        int rc = NMG_OK;
        switch (dtype) {
        case NMG_F32: rc = launch_scatter_tiled<float>(gather, P, s, &done); break;
        case NMG_F16: rc = launch_scatter_tiled<__half>(gather, P, s, &done); break;
        case NMG_BF16: rc = launch_scatter_tiled<__hip_bfloat16>(gather, P, s, &done); break;
        case NMG_F64: rc = launch_scatter_tiled<double>(gather, P, s, &done); break;
        }
        if (rc != NMG_OK || done) return rc;
    }
#define NMG_LAUNCH(T)                                                                         \
    do {                                                                                      \
        if (gather)                                                                           \
            hipLaunchKernelGGL(gather_kernel<T>, dim3((unsigned)grid), dim3(bs), 0, s, P);    \
        else                                                                                  \
            hipLaunchKernelGGL(to_dense_kernel<T>, dim3((unsigned)grid), dim3(bs), 0, s, P);  \
    } while (0)
    switch (dtype) {
    case NMG_F32: NMG_LAUNCH(float); break;
    case NMG_F16: NMG_LAUNCH(__half); break;
    case NMG_BF16: NMG_LAUNCH(__hip_bfloat16); break;
    case NMG_F64: NMG_LAUNCH(double); break;
    }
#undef NMG_LAUNCH
    NMG_HIP_TRY(hipGetLastError());
    return NMG_OK;
}

extern "C" int nmg_to_dense(const void *d_val, const int16_t *d_idx, void *d_dense,
                            const nmg_view *view, int n, int m, int g, int dtype, void *stream)
{
    return launch_scatter(false, d_dense, view, d_val, d_idx, n, m, g, dtype, stream);
}

extern "C" int nmg_gather(const void *d_dense, const nmg_view *view, const int16_t *d_idx,
                          void *d_val, int n, int m, int g, int dtype, void *stream)
{
    return launch_scatter(true, d_dense, view, d_val, d_idx, n, m, g, dtype, stream);
}

extern "C" int64_t nmg_rowpack_pat_bytes(int n, int m) { return binom(m, n) <= 256 ? 1 : 2; }

extern "C" int nmg_rowpack(const void *d_val, const int16_t *d_idx, int64_t G, int64_t S,
                           void *d_pk_val, void *d_pk_pat, int n, int m, int g, int dtype,
                           void *stream)
{
    nmg_view v{1, G, S, 0, S, 1};
    TileGeom tg;
    if (int rc = check_common(&v, n, m, g, dtype, &tg)) return rc;
    NMG_REQUIRE(dtype != NMG_F64, NMG_ERR_UNSUPPORTED, "rowpack supports f32/f16/bf16");
    if (tg.outer == 0) return NMG_OK;
    NMG_REQUIRE(d_val && d_idx && d_pk_val && d_pk_pat, NMG_ERR_ARG, "null device pointer");
    RowpackParams P{};
    P.val = d_val;
    P.idx = d_idx;
    P.pk_val = d_pk_val;
    P.pk_pat = d_pk_pat;
    P.G = G;
    P.nb = tg.num_blocks;
    P.num_chunks = tg.num_chunks;
    P.outer = tg.outer;
    P.n = n;
    P.g = g;
    P.c = tg.c;
    P.cols = tg.cols;
    P.pat_bytes = (int)nmg_rowpack_pat_bytes(n, m);
    const int64_t total = tg.outer * tg.cols;
    const int bs = 256;
    const int64_t grid = (total + bs - 1) / bs;
    NMG_REQUIRE(grid <= 0x7fffffffLL, NMG_ERR_UNSUPPORTED, "too many slots");
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
    case NMG_F32: hipLaunchKernelGGL(rowpack_kernel<float>, dim3((unsigned)grid), dim3(bs), 0, s, P); break;
    case NMG_F16: hipLaunchKernelGGL(rowpack_kernel<__half>, dim3((unsigned)grid), dim3(bs), 0, s, P); break;
    case NMG_BF16: hipLaunchKernelGGL(rowpack_kernel<__hip_bfloat16>, dim3((unsigned)grid), dim3(bs), 0, s, P); break;
    }
    NMG_HIP_TRY(hipGetLastError());
    return NMG_OK;
}
