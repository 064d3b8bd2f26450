// Dense -> grouped n:m for scores of 32 bits and m <= 8, at most 128 patterns: the tile as a matching problem.
// Included by nmg_match_{f32,f16,bf16}.hip, one instantiation each.
//
// The sorted walk of the reference (nmg_sparsify.hip) accepts edges (column o, pattern p) in descending
// order of one key that both ends share.  That is the stable matching of columns (one pattern each) with
// patterns (g columns each) under preferences given by the key, and it is unique: whatever order the
// columns propose in, deferred acceptance ends in it.  So all columns propose at once to their best pattern,
// a pattern keeps its g best and sends the others away, those propose to the best pattern whose last kept
// key is below theirs, and so on.  Inside a pattern the walk hands out slots in descending key order, so the
// patterns' lists are kept sorted and are the result.
//
// The walk batched by "until the next pattern fills", which this replaced, took up to one round per pattern
// over all free columns (6 / 28 / 70 rounds for 2:4, 2:8, 4:8).  Random weights need 3.5 / 6 / 8 rounds here,
// and all but the first concern a few columns: 12 of 96 are proposed again in total (2:4:16), 106 of 896
// (2:8:32), 276 of 2240 (4:8:32).
//
// A round over all columns:
//   1. every pending column computes its proposal (one thread per column; threshold of a pattern = key of its
//      last slot, 0 while it has room);
//   2. counting sort of all columns' proposals, kept and new, by pattern and by bins of the score below the tile's largest;
//   3. every proposal finds its rank: those in larger bins of its pattern plus those of its own bin that are larger (all pairs);
//   4. what ranks below the pattern's capacity is written to its slot, the rest is pending.
// A quarter of the columns and fewer (any n:m:g: half) insert into the lists lane by lane, into long ones key by key (the code says how).
//
// us, 4096 x 4096 fp16 with the blocks along the contiguous / the slow dim (8192 x 8192 for 2:8:32), batched walk -> ranks among all
// proposals of a pattern -> this: 2:4:16 99 -> 59 / 58 -> 51.5 / 51.5, 1:8:32 39 / 41 -> 32 / 34, 3:6:12 77 / 73 -> 63 / 61, 2:8:32 727 -> 195 / 197 -> 146 / 150,
// 4:8:32 390 -> 120 / 114 -> 75 / 74; any n:m:g: 2:4:4 168 / 231 -> 111 / 110 -> 90, 2:4:8 115 / 146 -> 72 -> 59, 2:4:32 118 / 135 -> 104 / 114 ->
// 94 / 104, 2:4:64 130 / 146 -> 115 / 123 -> 98 / 107, 1:2:8 192 / 302 -> 148 / 139 -> 137 / 130, 2:8:8 293 / 326 -> 131 / 133 -> 101 / 104, 1:8:8 86 / 117 -> 76 -> 60,
// 4:8:16 870 / 810 -> 280 / 295 -> 233 / 239, 2:4:100 144 / 162 -> 121 / 135.  What each part gave, 2:8:32: bins 43 -> 20 us of the first round, score and pattern
// compared as one double 17 -> 7 (a select behind a select on the same condition takes 17 to 40 clocks, a 64-bit maximum 4), the sorted keys in the place of the
// lists (six workgroups a CU instead of five) 168 -> 150, the reads of a column's patterns in flight together 150 -> 145.  4:8:32: 125 -> 102, and 73 where the
// later rounds are inlined: in a function their addresses are not known to lie in LDS.  Of the 151 us of 2:8:32 along the slow dim tile data and results
// take 50, first proposals 14, the first round 20, the later ones 67, of the 54 of 2:4:16 (same box) 16, 5, 12 and 21: chains of LDS round trips and the issue
// of vector instructions, 1500 and 1105 a wavefront.
//
// Columns that have no pattern with room and a positive score wait.  In the walk they come last, together
// with the zero columns beyond the end of the group dim, in descending column order, and each takes the
// largest pattern with room: that is written in closed form.
//
// A block that reaches beyond the end of the sparse dim has positions that are zero for every column, so patterns
// that agree in the real positions tie for every column: all columns propose to the largest of such a class, and
// one pattern's worth of them is kept in a round.  `match_partial` does the first rounds of such a tile.
#pragma once
#include "nmg_common.h"

#include <algorithm>

namespace nmg {

constexpr int match_binom(int m, int n)
{
    long r = 1;
    for (int i = 1; i <= n; i++) r = r * (m - n + i) / i;
    return (int)r;
}

// The patterns of n:m as position masks in the library's order (nmg_runtime.hip), at compile time.
template <int N, int M> struct MatchMasks {
    uint8_t mask[match_binom(M, N)] = {};
    constexpr int fill(int at, int n, int m, bool flip, int high)
    {
        if (n == m || n == 0) {
            mask[at] = (uint8_t)(((1 << n) - 1) | high);
            return at + 1;
        }
        const int mid = fill(at, n, m - 1, true, high);
        if (flip)
            for (int i = at, j = mid - 1; i < j; i++, j--) {
                const uint8_t t = mask[i];
                mask[i] = mask[j];
                mask[j] = t;
            }
        return fill(mid, n - 1, m - 1, !flip, high | (1 << (m - 1)));
    }
    constexpr MatchMasks() { fill(0, N, M, false, 0); }
};

struct MatchParams {
    const void *dense;
    void *val;
    int16_t *idx;
    ViewDev view;
    int64_t outer;
    int n, m, g, c, cols;
    int region_bytes, r_mem, r_arr, r_int;     // LDS bytes of one tile, offsets inside
    int unit;                                  // bytes of one load of the tile data (16, 8, 4, or one element)
    int out4;                                  // four slots per thread on the way out
    int lanes_log2;                            // lanes that hold a pattern's list in the later rounds; 0: no such rounds
    int listed;                                // a partial block's refused columns have a list of their own in LDS
    uint32_t masks[32];                        // position mask of every pattern, four per word
    uint64_t magic_cols, magic_g;
};

template <int NT> __device__ __forceinline__ void match_sync()
{
    if (NT <= 64) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

// Inclusive prefix sum over 64, 32 or 16 consecutive lanes: DPP shifts inside the rows of 16 lanes, then lane
// 15 of rows 0 and 2 into rows 1 and 3, then lane 31 into rows 2 and 3.
template <int CTRL, int ROWS> __device__ __forceinline__ int match_dpp(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, CTRL < 0x140);
}
template <int LANES> __device__ __forceinline__ int match_prefix(int v)
{
    v += match_dpp<0x111, 0xF>(v);
    v += match_dpp<0x112, 0xF>(v);
    v += match_dpp<0x114, 0xF>(v);
    v += match_dpp<0x118, 0xF>(v);
    if (LANES >= 32) v += match_dpp<0x142, 0xA>(v);
    if (LANES == 64) v += match_dpp<0x143, 0xC>(v);
    return v;
}

template <int CTRL> __device__ __forceinline__ uint64_t match_swap(uint64_t v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, 0xF, 0xF, true);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ float match_abs(float x) { return fabsf(x); }
__device__ __forceinline__ float match_abs(__half x) { return fabsf(__half2float(x)); }
__device__ __forceinline__ float match_abs(__hip_bfloat16 x) { return fabsf(__bfloat162float(x)); }

// Key of the edge (column o, pattern p): patterns below each other in descending order of the number that they
// put on top, so that a group of proposals is followed by smaller keys.  0: none.
__device__ __forceinline__ uint64_t match_key(uint32_t score, int o, int p)
{
    return ((uint64_t)(((uint32_t)(255 - p) << 16) | (score >> 16)) << 32) | ((score << 16) | (uint32_t)o);
}
__device__ __forceinline__ int match_pattern(uint64_t key) { return 255 - (int)(key >> 48); }
__device__ __forceinline__ int match_column(uint64_t key) { return (int)(key & 0xFFFFu); }

constexpr int kMatchTables = 6;      // c ints each, and four counts (three of them for partial blocks only)
constexpr int kMatchPad = 32;        // bytes behind the proposals: a batch of four keys past the end of the last bin

// Value of lane (this one ^ X), X = 2^k or 2^k - 1.
template <int X> __device__ __forceinline__ uint32_t match_lane_xor(uint32_t v)
{
    auto dpp = [](uint32_t x, auto ctrl) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xF, 0xF, true); };
    if constexpr (X == 1) return dpp(v, std::integral_constant<int, 0xB1>{});
    else if constexpr (X == 2) return dpp(v, std::integral_constant<int, 0x4E>{});
    else if constexpr (X == 3) return dpp(v, std::integral_constant<int, 0x1B>{});
    else if constexpr (X == 4) return dpp(dpp(v, std::integral_constant<int, 0x141>{}), std::integral_constant<int, 0x1B>{});
    else if constexpr (X == 7) return dpp(v, std::integral_constant<int, 0x141>{});
    else if constexpr (X == 8) return dpp(v, std::integral_constant<int, 0x128>{});
    else if constexpr (X == 15) return dpp(v, std::integral_constant<int, 0x140>{});
    else if constexpr (X < 32) return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (X << 10) | 0x1F);
    else return (uint32_t)__shfl_xor((int)v, X);
}

// An edge's score (31 bits) and pattern as a positive double that is no NaN for any score.  (With the score as the high word those from 0x7FF00000
// on, which a weight that is no number may give, would be NaNs, and the maximum below drops them.)
__device__ __forceinline__ uint64_t match_edge(uint32_t score, uint32_t p) { return ((uint64_t)(score >> 1) << 32) | ((score << 31) | p); }
// Whether a pattern's positions are n from a multiple of n on.
constexpr bool match_run(int mask, int n)
{
    for (int at = 0; at + n <= 8; at += n)
        if (mask == ((1 << n) - 1) << at) return true;
    return false;
}
__device__ __forceinline__ uint32_t match_edge_score(uint64_t edge) { return (uint32_t)(edge >> 31); }
__device__ __forceinline__ int match_edge_pattern(uint64_t edge) { return (int)(edge & 0xFFu); }

// Larger one of two edges or keys.  One instruction, where fmax canonicalises its operands first.  The compiler does not
// know it for a vector instruction: `s_nop 1` before a move between lanes reads its result.
__device__ __forceinline__ uint64_t match_larger(uint64_t a, uint64_t b)
{
    uint64_t r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ uint64_t match_smaller(uint64_t a, uint64_t b)
{
    uint64_t r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Largest of LANES consecutive lanes, in all of them.
template <int LANES> __device__ __forceinline__ uint32_t match_top(uint32_t v)
{
    v = max(v, match_lane_xor<1>(v));
    v = max(v, match_lane_xor<2>(v));
    v = max(v, match_lane_xor<7>(v));
    v = max(v, match_lane_xor<15>(v));
    if constexpr (LANES >= 32) v = max(v, match_lane_xor<16>(v));
    if constexpr (LANES >= 64) v = max(v, match_lane_xor<32>(v));
    return v;
}

// Bins of a pattern in the first round, by score: 8 (four to an octave below the tile's largest score, the last one open) where a lane then
// has at most four of the tile's bins to sum up, else 4 (two to an octave).
constexpr int match_bins_log2(int nt, int c) { return 8 * c <= 4 * (nt < 64 ? nt : 64) ? 3 : 2; }
constexpr int match_bin_bytes(int bins) { return (4 + bins + 4) * 4; }      // a multiple of 16: bins come in fours

// Bytes of a tile's s_arr: a round's bins; then the later rounds' two lists of pending columns and the patterns' buckets (a batch is read past the
// last); then the waiting columns, flags and runs of the closed form; a partial block's proposals.  One after the other in the same place: 2:8:32 takes
// 25.8 KB a tile of fp16 instead of 29.5, six workgroups of a CU instead of five.
constexpr int match_few(int sg) { return sg != 0 ? 4 : 2; }
// Keys of a list that a lane holds where g is not compiled in: 64 lanes hold lists of 128, with four keys a lane 256 (us, 4096 x 4096 fp16, tiles of two
// wavefronts, two keys a lane -> four: 2:4:64 108 -> 113, 2:8:16 101 -> 105).
constexpr int match_list_keys(int nt) { return nt >= 256 ? 4 : 2; }
// Longer lists stay in LDS, a wavefront moves their keys (us, 4096 x 4096 fp16, rounds over all columns ->
// this: 1:4:300 297 -> 168, 2:4:400 298 -> 142, 1:8:257 160 -> 80, 1:2:1000 1205 -> 640).  It takes many proposals at a time for what a shift along
// the lanes does with eight, which a partial block gains from with lists of more than 64 keys: its columns want the same few patterns (2000 x 3000 bf16, blocks along the slow dim, 3:6:100 202 -> 125, 3:6:128 293 -> 152).
// Whole blocks of up to 256 keys are faster in the lanes (7:8:160 106, 116; 2:6:100 125, 139), but two or three patterns take eight proposals each
// in many rounds there (512 x 640 fp16 1:2:160 20.4 -> 17.4, 1:2:256 26.2 -> 20.6).
constexpr bool match_long(int nt, int c, int g, bool partial) { return nt >= 128 && g > (partial || c <= 3 ? 64 : 64 * match_list_keys(nt)); }
// Proposals that a pattern takes in a later round: what has room where the closed form, a first round's bins (short lists) or a partial block's
// proposals lie anyway.  With one for lists of up to three keys 1:6:3 was slower than by rounds, 178 against 157; 150 with three, 2:8:2 167 -> 159.
constexpr int match_bucket(bool longs, int g, bool partial)
{
    if (longs) return partial ? (g * 11 / 16 < 64 ? g * 11 / 16 : 64) : (g / 4 < 64 ? g / 4 : 64);
    return g < 3 ? 2 : g == 3 ? 3 : g / 2 < 8 ? g / 2 : 8;
}
static inline int match_scratch(bool longs, int cols, int c, int g, int bins_log2, bool lists, bool partial, int few)
{
    int bytes = std::max(match_bin_bytes(c << bins_log2), 4 * cols + cols / 4 + 16);
    if (lists) bytes = std::max(bytes, ((few + 1) / 2 + c * match_bucket(longs, g, partial) + 2) * 8);
    if (partial) bytes = std::max(bytes, cols * 8);
    return (bytes + 15) & ~15;
}

// Sorts s_arr[0 .. count), count <= NT * KPT, larger keys first, all NT threads at it: thread t has the keys t * KPT .. + KPT - 1 in registers, steps
// up to KPT apart are its own, up to 64 * KPT apart go between lanes, wider ones through s_arr.  Every exchange puts the
// larger key first, so the zeros beyond the end stay there.
template <int NT, int KPT> __device__ __forceinline__ void match_sort(uint64_t *s_arr, int count)
{
    const int t = threadIdx.x % NT, lane = t & 63;
    uint64_t k[KPT];
#pragma unroll
    for (int r = 0; r < KPT; r++) k[r] = t * KPT + r < count ? s_arr[t * KPT + r] : 0;
    auto step = [&](auto x_tag, auto flip_tag) {      // partner: thread t ^ X; with a flip, its registers reversed
        constexpr int X = decltype(x_tag)::value;
        constexpr bool FLIP = decltype(flip_tag)::value;
        uint64_t o[KPT];
        if constexpr (X < 64) {
#pragma unroll
            for (int r = 0; r < KPT; r++) {
                const uint64_t v = k[FLIP ? KPT - 1 - r : r];
                o[r] = ((uint64_t)match_lane_xor<X>((uint32_t)(v >> 32)) << 32) | match_lane_xor<X>((uint32_t)v);
            }
        } else {
            __syncthreads();
#pragma unroll
            for (int r = 0; r < KPT; r++)
                if (t * KPT + r < count) s_arr[t * KPT + r] = k[r];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < KPT; r++) {
                const int from = (t ^ X) * KPT + (FLIP ? KPT - 1 - r : r);
                o[r] = from < count ? s_arr[from] : 0;
            }
        }
        constexpr int TOP = FLIP ? (X + 1) / 2 : X;
        const bool first = ((X < 64 ? lane : t) & TOP) == 0;
#pragma unroll
        for (int r = 0; r < KPT; r++) k[r] = (o[r] > k[r]) == first ? o[r] : k[r];
    };
    auto own = [&](auto d_tag, bool flip) {      // pairs of registers D apart; with a flip, mirrored in blocks of 2 D
        constexpr int D = decltype(d_tag)::value;
#pragma unroll
        for (int r = 0; r < KPT; r++) {
            const int q = flip ? r ^ (2 * D - 1) : r ^ D;
            if (q > r && q < KPT) {
                const uint64_t x = k[r], y = k[q];
                const bool turn = y > x;
                k[r] = turn ? y : x;
                k[q] = turn ? x : y;
            }
        }
    };
    auto own_from = [&](auto d_tag) {      // D, D / 2, .. 1
        constexpr int D = decltype(d_tag)::value;
        if constexpr (D >= 4) own(std::integral_constant<int, 4>{}, false);
        if constexpr (D >= 2) own(std::integral_constant<int, 2>{}, false);
        if constexpr (D >= 1) own(std::integral_constant<int, 1>{}, false);
    };
    static_assert(KPT <= 8 && (KPT & (KPT - 1)) == 0 && NT <= 1024, "the steps below");
    if constexpr (KPT >= 2) own(std::integral_constant<int, 1>{}, true);
    if constexpr (KPT >= 4) {
        own(std::integral_constant<int, 2>{}, true);
        own_from(std::integral_constant<int, 1>{});
    }
    if constexpr (KPT >= 8) {
        own(std::integral_constant<int, 4>{}, true);
        own_from(std::integral_constant<int, 2>{});
    }
    auto merge = [&](auto w_tag) {      // runs of W threads into runs of 2 W
        constexpr int W = decltype(w_tag)::value;
        if constexpr (2 * W <= NT) {
            if (W * KPT >= count) return;
            step(std::integral_constant<int, 2 * W - 1>{}, std::true_type{});
            if constexpr (W >= 512) step(std::integral_constant<int, 256>{}, std::false_type{});
            if constexpr (W >= 256) step(std::integral_constant<int, 128>{}, std::false_type{});
            if constexpr (W >= 128) step(std::integral_constant<int, 64>{}, std::false_type{});
            if constexpr (W >= 64) step(std::integral_constant<int, 32>{}, std::false_type{});
            if constexpr (W >= 32) step(std::integral_constant<int, 16>{}, std::false_type{});
            if constexpr (W >= 16) step(std::integral_constant<int, 8>{}, std::false_type{});
            if constexpr (W >= 8) step(std::integral_constant<int, 4>{}, std::false_type{});
            if constexpr (W >= 4) step(std::integral_constant<int, 2>{}, std::false_type{});
            if constexpr (W >= 2) step(std::integral_constant<int, 1>{}, std::false_type{});
            own_from(std::integral_constant<int, KPT / 2>{});
        }
    };
    merge(std::integral_constant<int, 1>{});
    merge(std::integral_constant<int, 2>{});
    merge(std::integral_constant<int, 4>{});
    merge(std::integral_constant<int, 8>{});
    merge(std::integral_constant<int, 16>{});
    merge(std::integral_constant<int, 32>{});
    merge(std::integral_constant<int, 64>{});
    merge(std::integral_constant<int, 128>{});
    merge(std::integral_constant<int, 256>{});
    merge(std::integral_constant<int, 512>{});
    __syncthreads();
#pragma unroll
    for (int r = 0; r < KPT; r++)
        if (t * KPT + r < count) s_arr[t * KPT + r] = k[r];
    __syncthreads();
}

// First rounds of a tile with `real_rows` < m real positions.  All columns' keys are sorted by pattern and key in
// every round, since most of them are refused and sit in few, long groups.  Patterns that agree in the real positions are a class: where
// there are few, a column sums and compares once for each class.  One such tile is as long as the launch: three to seven rounds, each a
// sort, a pass over the keys and the new proposals.  The sort is a compare-exchange network on keys in registers (10 stages of 55 for
// 896 keys in LDS) and for the patterns of the compiled kernels a column's sums are folded in, as those of the other tiles (18
// instructions a pattern against 36).  us, network in LDS or places counted by all pairs and sums from masks -> now: 3:6:12 512 x 1792 fp32
// 53 -> 40, 1280 x 2176 bf16 57 -> 37, 2:8:32 3054 x 3960 bf16 143 -> 60 (3056 x 3960, without partial blocks, 50), 2001 x 2001 fp32 80 -> 51,
// 4:8:32 512 x 4099 fp16 100 -> 60, 1005 x 3000 bf16 536 -> 279, 7742 x 933 fp32 437 -> 253, 2:4:16 1001 x 1000 fp16 24 -> 21; any pattern,
// 3:8:8 997 x 1003 fp16 163 -> 122.  Of the 2:8:32 one 14 us came from the refused columns proposing one per lane instead of where they lie.  Sorts that lost:
// runs of 64 merged by binary search (gathers at random places of LDS, 1.5 x), keys broadcast from a wavefront's lanes (1.2 x).  A refused
// column skips the patterns of its class that those ahead of it are certain to fill: all of them that have no other
// class with the same score to turn to, which bit 0 of a key says here.  Stops when at most `few` columns are pending;
// leaves s_mem, s_occ, the waiting columns in s_np[1] and the pending ones in s_arr and s_np[0].
// A function of its own: its registers are not those of the other tiles.
template <typename T, int NT, int KPT, int SN, int SM, int SG>
__device__ __noinline__ void match_partial(int region_at, int r_mem, int r_arr, int r_int, int c, int m, int g, int so, int sr,
                                           int real_cols, int real_rows, int few, int listed)
{
    extern __shared__ __align__(16) unsigned char smem[];
    for (int *x : {&region_at, &r_mem, &r_arr, &r_int, &c, &m, &g, &so, &sr, &real_cols, &real_rows, &few, &listed})
        *x = __builtin_amdgcn_readfirstlane(*x);      // (arguments come in vector registers)
    const uint32_t *s_mask = (const uint32_t *)smem + c;
    const T *s_d = (const T *)(smem + region_at);
    uint64_t *s_mem = (uint64_t *)(smem + region_at + r_mem), *s_arr = (uint64_t *)(smem + region_at + r_arr);
    int *s_dem = (int *)(smem + region_at + r_int), *s_start = s_dem + c, *s_occ = s_start + c;
    int *s_list = s_occ + c, *s_at = s_list + c, *s_last = s_at + c, *s_np = s_last + c;      // the classes, largest patterns first
    if (SG != 0) g = SG;
    if (SM != 0) m = SM;
    const bool lists = KPT > 1 && (SG != 0 || listed);      // (at the compiled group sizes the list costs nothing)
    if (SM != 0 && SN != 0) c = match_binom(SM ? SM : 1, SN);
    const int tt = threadIdx.x % NT, real_mask = (1 << real_rows) - 1;
    auto column = [](uint64_t key) { return (int)((key >> 1) & 0x7FFFu); };
    int *s_class = s_np + 4;                                   // smallest pattern of every class
    uint64_t *s_least = (uint64_t *)(s_class + ((c + 1) & ~1));    // least last key of a class's patterns, without the pattern
    uint16_t *s_ref = (uint16_t *)(s_least + c);      // where in s_arr the refused ones are, if there is room (`lists`)
    int classes = 0;
    constexpr uint64_t EDGE = 0xFFFFFFFFFFFFull;      // score and column of a key
    auto propose = [&](int o, uint32_t at_score, int below) -> uint64_t {      // at that score only patterns up to `below`
        float a[8];
#pragma unroll
        for (int r = 0; r < 8; r++) a[r] = match_abs(s_d[o * so + min(r, m - 1) * sr]);
        auto score_of = [&](uint32_t mk) {
            float acc = 0;
#pragma unroll
            for (int r = 0; r < 7; r++)
                acc += __uint_as_float(__float_as_uint(a[r]) & (uint32_t)__builtin_amdgcn_sbfe((int)mk, r, 1));      // (adding 0 changes nothing)
            return __float_as_uint(acc);
        };
        if (classes == 0) {
            uint32_t best = 0, bmask = 0;
            int bp = 0;
            bool tied = false;
            if constexpr (SM != 0 && SN != 0) {      // the rows that do not exist are zeros, which change no sum
                constexpr MatchMasks<SN, SM> tab;
                constexpr int SC = match_binom(SM, SN);
#pragma unroll
                for (int p = 0; p < SC; p++) {
                    float acc = 0;
                    bool any = false;
#pragma unroll
                    for (int r = 0; r < SM; r++)
                        if ((tab.mask[p] >> r) & 1) {
                            acc = any ? acc + a[r] : a[r];
                            any = true;
                        }
                    const uint32_t sb = __float_as_uint(acc), mk = tab.mask[p] & (uint32_t)real_mask;
                    const uint64_t last = s_mem[p * g + g - 1];
                    if (sb >= best && !(sb == at_score && p > below) && match_key(sb, o << 1, p) > last) {
                        tied = sb == best && (tied || mk != bmask);
                        best = sb;
                        bp = p;
                        bmask = mk;
                    }
                    if (p % 8 == 7) {
#pragma unroll
                        for (int r = 0; r < SM; r++) asm volatile("" : "+v"(a[r]), "+v"(best));
                    }
                }
                return best == 0 ? 0 : match_key(best, o << 1, bp) | (tied ? 1 : 0);
            }
            for (int p0 = 0; p0 < c; p0 += 4) {      // four patterns' reads in flight; beyond the last the last again
                uint32_t mk4[4];
                uint64_t last4[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int p = min(p0 + u, c - 1);
                    mk4[u] = s_mask[p] & (uint32_t)real_mask;
                    last4[u] = s_mem[p * g + g - 1];
                }
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int p = p0 + u;
                    const uint32_t sb = score_of(mk4[u]);
                    if (p < c && sb >= best && !(sb == at_score && p > below) && match_key(sb, o << 1, p) > last4[u]) {
                        tied = sb == best && (tied || mk4[u] != bmask);
                        best = sb;
                        bp = p;
                        bmask = mk4[u];
                    }
                }
            }
            return best == 0 ? 0 : match_key(best, o << 1, bp) | (tied ? 1 : 0);
        }
        auto edge_of = [&](uint32_t sb) { return ((uint64_t)sb << 16) | (uint32_t)(o << 1); };
        // the largest pattern of class k that takes the column; -1: none
        auto within = [&](int k, uint32_t sb) {
            const int end = s_last[s_class[k]];
            int at = k > 0 ? s_last[s_class[k - 1]] + 1 : 0;
            if (sb == at_score && below >= 0 && s_last[below] == end) at = s_at[below];
            for (; at <= end; at++) {
                const int p = s_list[at];
                if (!(sb == at_score && p > below) && edge_of(sb) > (s_mem[p * g + g - 1] & EDGE)) return p;
            }
            return -1;
        };
        for (uint32_t under = ~0u;;) {      // scores below it (a second time where the best score's patterns are above `below`)
            uint32_t best = 0;
            int from = -1;
            bool several = false;
            for (int k0 = 0; k0 < classes; k0 += 4) {      // four classes' reads in flight; beyond the last the last again
                int p4[4];
                uint32_t mk4[4];
                uint64_t least4[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int k = min(k0 + u, classes - 1);
                    p4[u] = s_class[k];
                    least4[u] = s_least[k];
                }
#pragma unroll
                for (int u = 0; u < 4; u++) mk4[u] = s_mask[p4[u]] & (uint32_t)real_mask;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const uint32_t sb = score_of(mk4[u]);
                    if (k0 + u < classes && sb < under && sb >= best && edge_of(sb) > least4[u]) {
                        several = sb == best && from >= 0;
                        best = sb;
                        from = k0 + u;
                    }
                }
            }
            if (best == 0) return 0;
            int bp = -1, found = 0;
            if (!several) {
                bp = within(from, best);
                found = 1;
            } else {
                for (int k = 0; k < classes; k++) {
                    if (score_of(s_mask[s_class[k]] & (uint32_t)real_mask) != best) continue;
                    const int q = within(k, best);
                    if (q >= 0) found++;
                    bp = max(bp, q);
                }
            }
            if (bp >= 0) return match_key(best, o << 1, bp) | (found > 1 ? 1 : 0);
            under = best;
        }
    };
    for (int p = tt; p < c; p += NT) {
        int before = 0, above = 0, size = 0;      // patterns of classes with a smaller mask, of the same one
        for (int q = 0; q < c; q++) {
            const int x = (int)(s_mask[q] & real_mask), y = (int)(s_mask[p] & real_mask);
            before += x < y ? 1 : 0;
            size += x == y ? 1 : 0;
            above += x == y && q > p ? 1 : 0;
        }
        s_list[before + above] = p;
        s_at[p] = before + above;
        s_last[p] = before + size - 1;
    }
    // Few patterns, or few that agree: one by one, which reads half as much per sum (us, one by one against by classes: 1000 x 1001
    // 2:4:16 fp16 26.0, 27.4; 1536 x 2157 2:5:8 bf16, 4 classes of 10, 51, 54; x 2176 3:6:12, 14 of 20, 58, 66, 4 of 20, 60, 58; 2:8:32,
    // 16 of 28, 143, 135, 22 of 28, 143, 150).  Where half of a block and more is kept, so that most columns turn to few classes, also
    // below 13 patterns fewer: 3:6:12, 8 of 20, bf16 65, 70, fp16 64, 66; 6:8:16, 16 of 28, 105, 112.  Folded-in sums cost less: by classes
    // only up to a quarter of the patterns (4:8:32, one by one against by classes, 16 of 70 classes 253, 237, 30 of 70 328, 371; 2:8:32, 16
    // of 28, 75, 90).
    if (c > 15) {
        match_sync<NT>();
        for (int q = 0; q < c; q++) classes += s_at[q] == s_last[q] ? 1 : 0;
        if ((SM != 0 && SN != 0 ? 4 * classes > c : 3 * classes > 2 * c) || (2 * __popc(s_mask[0]) >= m && c - classes < 13)) classes = 0;
        for (int p = tt; p < c; p += NT)
            if (classes > 0 && s_at[p] == s_last[p]) {
                int k = 0;
                for (int q = 0; q < c; q++) k += s_at[q] == s_last[q] && s_at[q] < s_at[p] ? 1 : 0;
                s_class[k] = p;
                s_least[k] = 0;
            }
    }
    match_sync<NT>();
    for (int e = tt; e < real_cols; e += NT) s_arr[e] = propose(e, 0, 0);
    int left = 0;
    for (int round = 0; round < real_cols * c + 2; round++) {
        match_sync<NT>();
        match_sort<NT, KPT>(s_arr, real_cols);
        // groups; first refused column of every pattern that has another class to turn to
        for (int p = tt; p < c; p += NT) {
            s_start[p] = 0;
            s_dem[p] = 0;
            s_occ[p] = real_cols;
        }
        if (tt == 0) s_np[0] = 0;
        match_sync<NT>();
        for (int e = tt; e < real_cols; e += NT) {
            const uint64_t key = s_arr[e], prev = e > 0 ? s_arr[e - 1] : ~0ull;
            if (key != 0 && (e == 0 || match_pattern(prev) != match_pattern(key))) s_start[match_pattern(key)] = e;
        }
        match_sync<NT>();
        for (int e = tt; e < real_cols; e += NT) {
            const uint64_t key = s_arr[e], next = e + 1 < real_cols ? s_arr[e + 1] : 0;
            if (key == 0) continue;
            const int p = match_pattern(key), r = e - s_start[p];
            if (next == 0 || match_pattern(next) != p) s_dem[p] = r + 1;
            if (r == g - 1) s_mem[p * g + g - 1] = key;
            if (r >= g) {
                const int nr = atomicAdd(s_np, 1);
                if (lists) s_ref[nr] = (uint16_t)e;
                if (key & 1) atomicMin(&s_occ[p], e);
            }
        }
        match_sync<NT>();
        left = s_np[0];
        for (int k = tt; k < classes; k += NT) {
            const int end = s_last[s_class[k]], before = k > 0 ? s_last[s_class[k - 1]] : -1;
            uint64_t least = ~0ull;
            for (int at = before + 1; at <= end; at++) least = min(least, s_mem[s_list[at] * g + g - 1] & EDGE);
            s_least[k] = least;
        }
        match_sync<NT>();
        if (left <= few) break;
        for (int i = tt; i < (lists ? left : real_cols); i += NT) {
            const int e = lists ? (int)s_ref[i] : i;
            const uint64_t key = s_arr[e];
            if (key == 0) continue;
            const int p = match_pattern(key), r = e - s_start[p];
            if (r < g) continue;
            uint32_t score = 0;
            int q = p;
            if ((key & 1) == 0) {
                score = (uint32_t)(key >> 16);
                const int to = s_at[p] + (min(e, s_occ[p]) - s_start[p] - g) / g + 1;
                q = to <= s_last[p] ? s_list[to] : -1;
            }
            s_arr[e] = propose(column(key), score, q);
        }
    }
    // the lists, the pending columns in front of s_arr
    constexpr int MOST = 5;      // keys that a thread holds while it re-orders s_arr: five columns at most (match_launch)
    uint64_t mine[MOST];
    int waiting = 0;
    if (tt == 0) s_np[0] = 0;
#pragma unroll
    for (int i = 0; i < MOST; i++) {
        const int e = tt + NT * i;
        mine[i] = e < real_cols ? s_arr[e] : 0;
        if (e < real_cols && mine[i] == 0) waiting++;
    }
    if (waiting != 0) atomicAdd(s_np + 1, waiting);
    match_sync<NT>();
#pragma unroll
    for (int i = 0; i < MOST; i++)
        if (mine[i] != 0) {
            const int e = tt + NT * i, p = match_pattern(mine[i]), r = e - s_start[p];
            if (r < g) s_mem[p * g + r] = (mine[i] & ~0xFFFFull) | (uint64_t)column(mine[i]);
            else s_arr[atomicAdd(s_np, 1)] = (uint64_t)column(mine[i]);
        }
    for (int p = tt; p < c; p += NT) {
        s_occ[p] = min(g, s_dem[p]);
        s_dem[p] = 0;
    }
    match_sync<NT>();
}

// Wavefronts per SIMD that the registers are cut for.  The kernels compiled for a pattern gain from the most, whatever
// they spill (4096 x 4096 fp16 2:4:4 with 5 / 7: 134 / 116 us); so do those of up to a wavefront per tile that take any pattern
// (2:4:12 with 4 / 6: 136 / 125), which spill more where the columns are contiguous (1:8:8 with 5 / 6: 77 / 87), and tiles of two and four wavefronts
// where they are not (six workgroups of a CU instead of five, 2000 x 3000 bf16 1:7:48 48 -> 42, 1024 x 1536 fp32 1:3:128 31 -> 27).
constexpr int match_waves(int nt, bool compiled, bool rc)
{
    return nt > 256 ? 4 : compiled ? (nt == 256 ? 6 : nt == 64 ? 6 : 7) : nt > 64 ? (rc ? 4 : 6) : rc ? 5 : 6;
}

// Columns of a tile per thread of its workgroup, up to a power of two.
constexpr int match_keys(int nt, int cpt)
{
    const int threads = nt <= 64 ? 256 : nt;
    int k = 1;
    while (k * threads < nt * cpt) k *= 2;
    return k;
}

// NT threads per tile, at most CPT columns each.  SN, SM, SG != 0: compiled for that n:m:g.  RC: the columns are
// the contiguous dim of the dense tensor, and the tile data lies in LDS as [position][column]; otherwise
// as [column][position].
template <typename T, int NT, int CPT, int SN, int SM, int SG, bool RC>
__global__ __launch_bounds__(NT <= 64 ? 256 : NT, match_waves(NT, SM != 0, RC)) void match_kernel(MatchParams Q)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int SC = SM ? match_binom(SM, SN) : 0;
    // Where whole patterns make up a column, their sums, compared with themselves once a tile, find weights that are no numbers; columns of such a tile compare whole numbers, and
    // edges have the score itself as their high word.  us, NaNs out of order -> all edges shifted (match_edge) -> this, 4096 x 4096 fp16: 3:6:12
    // 61.0 -> 62.6 -> 61.1, 4:8:32 73.9 -> 77.5 -> 73.4, 2:8:32 47.2 -> 48.7 -> 47.3, 2:4:16 51.3 -> 52.0 -> 51.6.  (2:4 with a g that is not compiled in
    // has no registers for the sums: 2:4:4 1024 x 1536 fp32 17.4 -> 17.8.)
    constexpr bool RAW = SG != 0 && SN > 1 && SM % (SN ? SN : 1) == 0;
    constexpr int THREADS = NT <= 64 ? 256 : NT;
    constexpr int TILES = THREADS / NT;
    constexpr int KPT = match_keys(NT, CPT);
    const int n = SN ? SN : Q.n, m = SM ? SM : Q.m, g = SG ? SG : Q.g, c = SC ? SC : Q.c;
    const int cols = SC && SG ? SC * SG : Q.cols;
    constexpr int V = 16 / (int)sizeof(T);
    const int ldc = (cols + V - 1) / V * V;      // RC: columns per line of the tile data
    const int tid = threadIdx.x;
    const int tile = tid / NT, tt = tid % NT;

    uint32_t *s_pos = (uint32_t *)smem;      // positions of a pattern, four bits each; behind them their masks
    const int head_bytes = (c * 8 + 15) & ~15;
    unsigned char *region = smem + head_bytes + (size_t)tile * Q.region_bytes;
    T *s_d = (T *)region;
    uint64_t *s_mem = (uint64_t *)(region + Q.r_mem);     // kept keys, every pattern's in descending order; 0: free slot.  Sorted keys before
    uint64_t *s_arr = (uint64_t *)(region + Q.r_arr);     // a partial block's proposals; else see match_scratch
    int *s_dem = (int *)(region + Q.r_int);               // proposals of the round per pattern
    int *s_start = s_dem + c;                             // first of them in s_arr
    int *s_occ = s_start + c;                             // slots taken
    int *s_np = s_occ + 4 * c;                            // pending columns, waiting columns, pending columns of the later rounds
    // A round's bins, larger patterns' behind smaller ones', of a pattern larger scores first; two counts in front of them
    int *s_bin = (int *)s_arr + 4;
    const int nbl2 = match_bins_log2(NT, c), nbins = c << nbl2;

    // ---- where the tiles lie ----
    // Workgroups go to the 8 XCDs in turn, each with an L2 of its own, and neighbours along the sparse dim share
    // 128-byte lines where that dim is contiguous: among every 64 workgroups XCD x takes 8x .. 8x+7.  Last tiles
    // first: those of the last chunk hold fewer real columns and should not be the tail.
    int64_t grp = blockIdx.x;
    if (grp < (int64_t)(gridDim.x & ~63u)) grp = (grp & ~63LL) | ((grp & 7) << 3) | ((grp >> 3) & 7);
    const T *dense = (const T *)Q.dense;
    const int64_t nbl = Q.view.num_blocks, per_batch = Q.view.num_chunks * nbl;
    int64_t wg = (int64_t)gridDim.x - 1 - grp;
    if (Q.view.S % m != 0 && nbl >= TILES) {
        // partial blocks take several times as long: their workgroups come first.  Number q of them is holder(q).
        const int64_t lines = Q.outer / nbl;
        auto holder = [&](int64_t q) { return ((q + 1) * nbl - 1) / TILES; };
        if (grp < lines) {
            wg = holder(grp);
        } else {      // number `wg` of the others
            int64_t q = wg * TILES / nbl;
            while (q < lines && holder(q) - q <= wg) q++;
            while (q > 0 && holder(q - 1) - (q - 1) > wg) q--;
            wg += q;
        }
    }
    const int64_t tile0 = wg * TILES;
    const int64_t b_first = tile0 / per_batch;
    const int64_t kc_first = (tile0 - b_first * per_batch) / nbl, mb_first = tile0 - b_first * per_batch - kc_first * nbl;
    auto locate = [&](int tm, int64_t &b, int64_t &kc, int64_t &mb) {
        b = b_first;
        kc = kc_first;
        mb = mb_first + tm;
        while (mb >= nbl) {
            mb -= nbl;
            if (++kc == Q.view.num_chunks) {
                kc = 0;
                b++;
            }
        }
    };

    // ---- tile data to LDS, zeros beyond the ends; UB: bytes of one load ----
    auto load = [&](auto ub) {
        constexpr int UB = decltype(ub)::value, E = UB / (int)sizeof(T);
        if constexpr (!RC && SM != 0 && (E > SM || SM % E != 0)) return;      // (the host does not ask for it)
        using Unit = typename std::conditional<UB == 16, uint4, typename std::conditional<UB == 8, uint2,
                     typename std::conditional<UB == 4, uint32_t, uint16_t>::type>::type>::type;
        auto copy_unit = [&](T *dst, const T *src, int valid) {      // `valid` elements of the unit exist
            if (valid >= E) {
                *(Unit *)dst = *(const Unit *)src;
            } else {
#pragma unroll
                for (int e = 0; e < E; e++) dst[e] = e < valid ? src[e] : Zero<T>::v();
            }
        };
        if (RC) {
            // lines of columns: consecutive threads take consecutive units of a line
            const int upl = ldc / E, total = TILES * m * upl;
#pragma unroll 4
            for (int e = tid; e < total; e += THREADS) {
                const int line = e / upl, o = (e - line * upl) * E;
                const int tm = TILES == 1 ? 0 : line / m, r = line - tm * m;
                int valid = 0;
                const T *src = dense;
                if (tile0 + tm < Q.outer) {
                    int64_t b, kc, mb;
                    locate(tm, b, kc, mb);
                    if (mb * m + r < Q.view.S) {
                        src = dense + b * Q.view.stride_b + (kc * cols + o) + (mb * m + r) * Q.view.stride_s;
                        const int64_t left = min(Q.view.G - kc * cols, (int64_t)cols) - o;
                        valid = left < 0 ? 0 : left < E ? (int)left : E;
                    }
                }
                copy_unit((T *)(smem + head_bytes + (size_t)tm * Q.region_bytes) + r * ldc + o, src, valid);
            }
        } else {
            // columns of m positions: consecutive threads take the units of a column, then the same column of the
            // next tile (its neighbour in memory where the sparse dim is contiguous), then the next columns
            const int upc = max(m / E, 1), across = TILES * upc, walkers = THREADS / across;
            if (tid < walkers * across) {
                const int o0 = tid / across, w = tid - o0 * across;
                const int tm = w / upc, r = (w - tm * upc) * E;
                T *dst = (T *)(smem + head_bytes + (size_t)tm * Q.region_bytes) + r;
                const T *src = dense;
                int real = 0, valid = 0;
                if (tile0 + tm < Q.outer) {
                    int64_t b, kc, mb;
                    locate(tm, b, kc, mb);
                    const int64_t left = Q.view.S - (mb * m + r);
                    valid = left < 0 ? 0 : left < E ? (int)left : E;
                    src = dense + b * Q.view.stride_b + kc * cols * Q.view.stride_g + (mb * m + r) * Q.view.stride_s;
                    real = (int)min(Q.view.G - kc * cols, (int64_t)cols);
                }
                const int64_t sg = Q.view.stride_g;
                if (valid == E && real == cols) {
#pragma unroll 4
                    for (int o = o0; o < cols; o += walkers) copy_unit(dst + o * m, src + o * sg, E);
                } else {
                    for (int o = o0; o < cols; o += walkers) copy_unit(dst + o * m, src + o * sg, o < real ? valid : 0);
                }
            }
        }
    };
    if (Q.unit == 16) load(std::integral_constant<int, 16>{});
    else if (Q.unit == 8) load(std::integral_constant<int, 8>{});
    else if (Q.unit == 4 && (sizeof(T) == 4 || !RC)) load(std::integral_constant<int, 4>{});
    else load(std::integral_constant<int, (int)sizeof(T)>{});
    for (int p = tid; p < c; p += THREADS) {
        uint32_t mk = (Q.masks[p >> 2] >> (8 * (p & 3))) & 0xFFu, pos = 0;
        s_pos[c + p] = mk;
        for (int j = 0; mk != 0; j++) {
            pos |= (uint32_t)(__ffs(mk) - 1) << (4 * j);
            mk &= mk - 1;
        }
        s_pos[p] = pos;
    }
    const bool live = tile0 + tile < Q.outer;
    int real_cols = cols, real_rows = m;
    if (live) {
        int64_t b, kc, mb;
        locate(tile, b, kc, mb);
        real_cols = (int)min(Q.view.G - kc * cols, (int64_t)cols);
        real_rows = (int)min(Q.view.S - mb * m, (int64_t)m);
    }
    if (real_rows == m && real_cols > 0) {
        for (int b = tt; b < match_bin_bytes(nbins) / 16; b += NT) ((int4 *)s_arr)[b] = int4{0, 0, 0, 0};
    } else {
        for (int s = tt; s < cols; s += NT) s_mem[s] = 0;
    }
    for (int p = tt; p < kMatchTables * c + 4; p += NT) s_dem[p] = 0;
    __syncthreads();

    // the partial blocks among the workgroup's tiles, all threads on one after the other
    // (kept out of the way of launches that have none: us, eight copies of the call and any branch -> this, 4096^2 fp16, 2:4:16 59.2 -> 59.0, as
    // without a list of refused columns, 3:6:12, blocks along the slow dim, 76.0 -> 75.4)
    const bool partial = __builtin_amdgcn_readfirstlane(Q.view.S % m != 0 ? 1 : 0) != 0;
    if (__builtin_expect(partial, 0))
#pragma unroll 1
        for (int tm = 0; tm < TILES && tile0 + tm < Q.outer; tm++) {
            int64_t b, kc, mb;
            locate(tm, b, kc, mb);
            if (mb != nbl - 1) continue;
            const int there = (int)min(Q.view.G - kc * cols, (int64_t)cols);
            // (what is left for the lists: a refused column tries there the patterns of a class one by one.  Up to a quarter
            // of the columns, 3:6:12 1003 x 2001 fp32 45.3 -> 45.0 us, 512 x 1792 46.8 -> 39.5; but 2:8:32 1005 x 5000 74 -> 92)
            match_partial<T, THREADS, KPT, SN, SM, SG>(head_bytes + tm * Q.region_bytes, Q.r_mem, Q.r_arr, Q.r_int, c, m, g, RC ? 1 : m,
                                                       RC ? ldc : 1, there, (int)(Q.view.S - mb * m), there / (c <= 20 ? 4 : 8), Q.listed);
        }
    auto group_of = [&](int s) { return SG ? s / SG : (int)(((uint64_t)s * Q.magic_g) >> 32); };
    auto at = [&](int o, int r) { return RC ? r * ldc + o : o * m + r; };

    bool odd = false;      // RAW: a column of the tile has a weight that is no number
    float sums = 0;        // RAW: of this thread's columns
    // Proposal of a column of such a tile: whole numbers are compared.
    auto propose_odd = [&](int o, auto thr_tag) __attribute__((always_inline)) -> uint64_t {
        uint32_t best = 0;
        int bp = 0;
#pragma unroll 1
        for (int p = 0; p < SC; p++) {
            const uint32_t ps = s_pos[p];
            float acc = match_abs(s_d[at(o, (int)(ps & 15u))]);
#pragma unroll 1
            for (int j = 1; j < SN; j++) acc += match_abs(s_d[at(o, (int)((ps >> (4 * j)) & 15u))]);
            const uint32_t sb = __float_as_uint(acc);
            if (sb >= best && (!decltype(thr_tag)::value || match_key(sb, o, p) > s_mem[p * g + g - 1])) {
                best = sb;
                bp = p;
            }
        }
        return best == 0 ? 0 : match_key(best, o, bp);
    };
    // Proposal of column o: its best pattern among those with room or a last key below the column's (the
    // larger pattern on equal scores); 0 where no such pattern has a positive score.  THR = false: all have room.
    auto propose = [&](int o, auto thr_tag) __attribute__((always_inline)) -> uint64_t {      // (a call takes addresses that say no more that they lie in LDS)
        constexpr bool THR = decltype(thr_tag)::value;
        if constexpr (RAW && THR)
            if (odd) return propose_odd(o, thr_tag);
        float a[8];
        if (!RC && sizeof(T) == 2 && SM == 8) {
            const uint4 raw = *(const uint4 *)(s_d + o * 8);
            T v[8];
            __builtin_memcpy(v, &raw, 16);
#pragma unroll
            for (int r = 0; r < 8; r++) a[r] = match_abs(v[r]);
        } else if (!RC && sizeof(T) == 2 && SM == 4) {
            const uint2 raw = *(const uint2 *)(s_d + o * 4);
            T v[4];
            __builtin_memcpy(v, &raw, 8);
#pragma unroll
            for (int r = 0; r < 8; r++) a[r] = r < 4 ? match_abs(v[r & 3]) : 0.f;
        } else {
#pragma unroll
            for (int r = 0; r < 8; r++) a[r] = r < m ? match_abs(s_d[at(o, r)]) : 0.f;
        }
        uint64_t best = 0;
        int later = 0;
        uint32_t zero = 0;      // not to be known for one: the patterns' numbers would take a register each for all columns
        if constexpr (RAW) asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        float whole = 0;      // of the column
        auto consider = [&](float acc, int p) {
            uint32_t sb = __float_as_uint(acc);
            if (THR) {
                const uint64_t last = s_mem[p * g + g - 1 + later];
                if (!(match_key(sb, o, p) > last)) sb = 0;
            }
            best = match_larger(best, RAW ? ((uint64_t)sb << 32) | (zero + (uint32_t)p) : match_edge(sb, (uint32_t)p));
        };
        if constexpr (SM != 0) {
            constexpr MatchMasks<SN ? SN : 1, SM ? SM : 1> tab;
            bool some = false;
#pragma unroll
            for (int p = 0; p < SC; p++) {
                float acc = 0;
                bool any = false;
#pragma unroll
                for (int r = 0; r < SM; r++)
                    if ((tab.mask[p] >> r) & 1) {
                        acc = any ? acc + a[r] : a[r];      // left to right, in ascending positions
                        any = true;
                    }
                consider(acc, p);
                if (RAW && match_run(tab.mask[p], SN)) {
                    whole = some ? whole + acc : acc;
                    some = true;
                }
                // all sums and thresholds in flight at once would not fit the registers
                if (SC > 8 && p % 8 == 7) {
                    if (THR) asm volatile("" : "+v"(later), "+v"(best));
#pragma unroll
                    for (int r = 0; r < SM; r++) asm volatile("" : "+v"(a[r]), "+v"(best), "+v"(zero));
                }
            }
        } else {
            for (int p0 = 0; p0 < c; p0 += 4) {      // (beyond the last pattern no mask: no score)
                const uint32_t four = Q.masks[p0 >> 2];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    float acc = 0;
#pragma unroll
                    for (int r = 0; r < 8; r++)
                        acc += __uint_as_float(__float_as_uint(a[r]) & (0u - ((four >> (8 * u + r)) & 1u)));      // a[r] or 0, without a branch
                    consider(acc, min(p0 + u, c - 1));
                }
            }
        }
        if (RAW && !THR) sums += whole;
        const uint32_t score = RAW ? (uint32_t)(best >> 32) : match_edge_score(best);
        return score == 0 ? 0 : match_key(score, o, match_edge_pattern(best));
    };

    if (live) {
        // a quarter of the tile and fewer go on in the registers below
        const bool lists = SG != 0 || Q.lanes_log2 != 0;
        const int few = lists ? cols / match_few(SG) : 0;
        uint16_t *pending = (uint16_t *)s_arr;
        // every proposal that is not the last word of its column is refused once per (column, pattern) at most
        const int limit = cols * c + 2;
        int pend = real_cols, round = 0;
        uint64_t own[CPT] = {};      // this thread's columns' proposals, kept or new; 0: none
        if (real_rows < m) {
            pend = s_np[0];
            match_sync<NT>();
            if (pend > few) {      // (tiles without lists)
                for (int s = tt; s < cols; s += NT) s_arr[s] = 0;
                match_sync<NT>();
                for (int s = tt; s < cols; s += NT)
                    if (s_mem[s] != 0) s_arr[match_column(s_mem[s])] = s_mem[s];
                match_sync<NT>();
#pragma unroll
                for (int i = 0; i < CPT; i++) own[i] = tt + NT * i < real_cols ? s_arr[tt + NT * i] : 0;
            }
            if (RAW) {
                uint32_t top = 0;
                for (int s = tt; s < cols; s += NT) top = max(top, (uint32_t)(s_mem[s] >> 16));
                top = match_top<(NT < 64 ? NT : 64)>(top);
                if constexpr (NT > 64) {
                    if (tt == 0) s_start[0] = 0;
                    __syncthreads();
                    if ((tt & 63) == 0) atomicMax((unsigned *)s_start, top);
                    __syncthreads();
                    top = ((unsigned *)s_start)[0];
                }
                odd = top > 0x7F800000u;
            }
            round = 1;
        }
        for (; round < limit && pend > (round == 0 ? 0 : few); round++) {
            // 1. proposals
            uint32_t top = 0;
            if (round == 0) {
#pragma unroll 1
                for (int e = tt; e < real_cols; e += NT) {
                    const uint64_t key = propose(e, std::false_type{});
                    s_mem[e] = key;
                    top = max(top, (uint32_t)(key >> 16));
                }
                if (RAW && __builtin_expect(sums != sums, 0)) {
#pragma unroll 1
                    for (int e = tt; e < real_cols; e += NT) {
                        const uint64_t key = propose_odd(e, std::false_type{});
                        s_mem[e] = key;
                        top = max(top, (uint32_t)(key >> 16));
                    }
                }
#pragma unroll
                for (int i = 0; i < CPT; i++) own[i] = tt + NT * i < real_cols ? s_mem[tt + NT * i] : 0;      // this thread's own entries
            } else {
                match_sync<NT>();
                for (int b = tt; b < match_bin_bytes(nbins) / 16; b += NT) ((int4 *)s_arr)[b] = int4{0, 0, 0, 0};
                if (tt < 2) s_np[tt] = 0;
                match_sync<NT>();
#pragma unroll 1
                for (int i = 0; i < CPT; i++) {
                    const int o = tt + NT * i;
                    uint64_t mine = own[0];
#pragma unroll
                    for (int u = 1; u < CPT; u++) mine = u == i ? own[u] : mine;
                    if (o < real_cols) {
                        if (mine != 0 && mine < s_mem[match_pattern(mine) * g + g - 1]) mine = 0;      // refused
                        if (mine == 0) mine = propose(o, std::true_type{});
                        top = max(top, (uint32_t)(mine >> 16));
                    }
#pragma unroll
                    for (int u = 0; u < CPT; u++) own[u] = u == i ? mine : own[u];
                }
            }
            top = match_top<(NT < 64 ? NT : 64)>(top);
            if constexpr (NT > 64) {
                if ((tt & 63) == 0) atomicMax((unsigned *)s_bin - 4, top);
                __syncthreads();
                top = ((unsigned *)s_bin)[-4];
            }
            if (RAW) odd = odd || top > 0x7F800000u;      // (every such column proposes with such a score, which the lists keep before all others)
            // 2. counting sort by pattern and score
            auto bin_of = [&](uint64_t key) {
                return (match_pattern(key) << nbl2) + (int)min((top - (uint32_t)(key >> 16)) >> (24 - nbl2), (1u << nbl2) - 1);
            };
            int pos[CPT];
#pragma unroll
            for (int i = 0; i < CPT; i++) {
                pos[i] = 0;
                if (own[i] != 0) pos[i] = atomicAdd(&s_bin[bin_of(own[i])], 1);
                else if (tt + NT * i < real_cols) atomicAdd(s_np + 1, 1);      // waits
            }
            match_sync<NT>();
            if (tt < 64) {      // four or eight bins a lane
                constexpr int LANES = NT < 64 ? NT : 64;
                int4 *mine = (int4 *)s_bin + (nbl2 == 3 ? tt : 2 * tt), d0{}, d1{};
                const int first = nbl2 == 3 ? 4 * tt : 8 * tt;
                if (first < nbins) d0 = mine[0];
                if (nbl2 == 2 && first + 4 < nbins) d1 = mine[1];
                d0.y += d0.x;
                d0.z += d0.y;
                d0.w += d0.z;
                int sum = d0.w;
                if (nbl2 == 2) {
                    d1.x += d0.w;
                    d1.y += d1.x;
                    d1.z += d1.y;
                    sum = d1.w += d1.z;
                }
                const int excl = match_prefix<LANES>(sum) - sum;
                if (first < nbins + 1) mine[0] = int4{excl, excl + d0.x, excl + d0.y, excl + d0.z};
                if (nbl2 == 2 && first + 4 < nbins + 1) mine[1] = int4{excl + d0.w, excl + d1.x, excl + d1.y, excl + d1.z};
                if (tt == LANES - 1) s_bin[-3] = s_bin[nbins] = excl + sum;      // proposals of this round
            }
            match_sync<NT>();
            const int props = s_bin[-3];
#pragma unroll
            for (int i = 0; i < CPT; i++)
                if (own[i] != 0) s_mem[s_bin[bin_of(own[i])] + pos[i]] = own[i];
            if (tt < 4) s_mem[props + tt] = 0;      // what the last batch of the last bin reads
            match_sync<NT>();
            // 3. ranks.  Thread e takes the proposal that the sort put at e: the lanes of a wavefront then read the
            //    same few bins.  A proposal that has seen as many larger keys as its pattern has slots stops.
            uint64_t key[CPT];
#pragma unroll
            for (int i = 0; i < CPT; i++) {
                const int e = tt + NT * i;
                key[i] = 0;
                if (e < props) {
                    const uint64_t mine = s_mem[e];
                    const int bin = bin_of(mine), s0 = s_bin[bin], s1 = s_bin[bin + 1];
                    int r = s0 - s_bin[match_pattern(mine) << nbl2];      // the larger bins
                    // whole batches: behind the bin lie smaller keys
                    for (int j0 = s0; j0 < s1 && r < g; j0 += 4) {
                        uint64_t k4[4];
#pragma unroll
                        for (int u = 0; u < 4; u++) k4[u] = s_mem[j0 + u];
#pragma unroll
                        for (int u = 0; u < 4; u++) r += k4[u] > mine ? 1 : 0;
                    }
                    key[i] = mine;
                    pos[i] = r;
                }
            }
            for (int p = tt; p < c; p += NT) s_occ[p] = min(g, s_bin[(p + 1) << nbl2] - s_bin[p << nbl2]);
            match_sync<NT>();
            // 4. the new lists in the place of the sorted keys; what a pattern has no slot for is pending
#pragma unroll
            for (int i = 0; i < CPT; i++)
                if (key[i] != 0) {
                    if (pos[i] < g) {
                        s_mem[match_pattern(key[i]) * g + pos[i]] = key[i];
                    } else {
                        const int k = atomicAdd(s_np, 1);
                        if (k < few) pending[k] = (uint16_t)match_column(key[i]);
                    }
                }
            if (SG == 0 && NT >= 32 && g > 16) {      // (slot by slot in one thread a pattern 1:2:1000 took 740 us, 640 now)
#pragma unroll 1
                for (int s = tt; s < cols; s += NT) {
                    const int p = group_of(s);
                    if (s - p * g >= s_occ[p]) s_mem[s] = 0;
                }
            } else {
                for (int p = tt; p < c; p += NT)
                    for (int s = s_occ[p]; s < g; s++) s_mem[p * g + s] = 0;
            }
            match_sync<NT>();
            pend = s_np[0];
        }

        if (lists && pend > 0) {
            // Later rounds: a few columns, whatever the pattern.  L lanes hold a pattern's list, KPL keys each in descending
            // order, and insert a proposal by one shift along the lanes.  A pattern takes at most `bucket` proposals in a round;
            // the rest stay pending.  In a tile of several wavefronts the first one ends the matching alone, without barriers.
            constexpr int EIGHT = 8, LL = SG > 16 && SC <= 8 ? 4 : 3, KPL = SG == 0 ? match_list_keys(NT) : SG > 8 << (LL - 2) ? 4 : 2;
            const bool longs = SG == 0 && match_long(NT, c, g, real_rows < m);
            const int ll = SG != 0 ? LL : Q.lanes_log2, L = 1 << ll, bucket = match_bucket(longs, g, real_rows < m);
            static_assert(SG <= 32 && SG != 1, "a list fits its lanes; lists and buckets fit the proposals' place");
            uint16_t *next = pending + few;
            uint64_t *s_bkt = s_arr + (few + 1) / 2;      // free places hold 0
            if (real_rows < m) {
                constexpr int I = (CPT + 3) / 4;      // a partial block's columns come as entries of eight bytes
                uint16_t o[I];
#pragma unroll
                for (int i = 0; i < I; i++) o[i] = tt + NT * i < pend ? (uint16_t)s_arr[tt + NT * i] : 0;
                match_sync<NT>();
#pragma unroll
                for (int i = 0; i < I; i++)
                    if (tt + NT * i < pend) pending[tt + NT * i] = o[i];
            }
            for (int i = tt; i < c * bucket; i += NT) s_bkt[i] = 0;
            // a column's patterns go to EL lanes; the positions of a lane's patterns stay in registers
            constexpr int EL = SC >= 16 ? 8 : SC >= 8 ? 4 : 2, PER = SG != 0 ? (SC + EL - 1) / EL : 1;
            uint32_t mypos[PER];
            if constexpr (SG != 0) {
#pragma unroll
                for (int i = 0; i < PER; i++) mypos[i] = s_pos[min(tt % EL + EL * i, SC - 1)];
            }
            round = 0;
            auto late = [&](auto active_tag, int until) __attribute__((always_inline)) {      // threads of the tile that take part
                constexpr int A = decltype(active_tag)::value, W = A < 64 ? A : 64, WAVES = A / W;
                const int rows_log2 = (W == 64 ? 6 : W == 32 ? 5 : 4) - ll, rows = 1 << rows_log2;
                const int wave = tt / W, lane = tt % W, row = lane >> ll, r = lane & (L - 1);
                match_sync<A>();
                for (; round < limit && pend > until; round++) {
                    int *count = s_np + 2 + (round & 1);      // zero; the other one is cleared on the way
                    auto put = [&](int o, uint64_t key) {
                        if (key == 0) {
                            atomicAdd(s_np + 1, 1);
                            return;
                        }
                        const int p = match_pattern(key), place = atomicAdd(&s_dem[p], 1);
                        if (place < bucket) s_bkt[p * bucket + place] = key;
                        else next[atomicAdd(count, 1)] = (uint16_t)o;
                    };
                    // score (0: refused) and pattern of a column's edge.  No branch: the reads of a lane's patterns go out together.
                    auto edge = [&](int o, int p, uint32_t ps) {
                        float acc = match_abs(s_d[at(o, (int)(ps & 15u))]);
#pragma unroll
                        for (int j = 1; j < n; j++) acc += match_abs(s_d[at(o, (int)((ps >> (4 * j)) & 15u))]);
                        uint32_t sb = __float_as_uint(acc);
                        if (!(match_key(sb, o, p) > s_mem[p * g + g - 1])) sb = 0;
                        return RAW ? ((uint64_t)sb << 32) | (uint32_t)p : match_edge(sb, (uint32_t)p);
                    };
                    auto other = [&](uint64_t top, auto ctrl) {      // the larger one of two lanes
                        asm("s_nop 1" : "+v"(top));
                        return match_larger(top, match_swap<decltype(ctrl)::value>(top));
                    };
                    constexpr std::integral_constant<int, 0xB1> by_1{};      // lanes 1 apart, 2 apart, the two quads
                    constexpr std::integral_constant<int, 0x4E> by_2{};
                    constexpr std::integral_constant<int, 0x141> by_4{};
                    // A column's patterns over EL lanes, or a column per lane, which is less work where there are enough columns for it: in
                    // tiles of a wavefront from a quarter of the lanes on (us, 4096 x 4096 3:6:12 from 16 / 32 / never: 61.3 / 63.3 / 63.7), with
                    // many patterns from twice as many as lanes on (4:8:32 from 32 / 1024: 85 / 73).
                    if (SG != 0 && !odd && (A <= 64 ? pend <= A / 4 : SC <= 32 || pend <= 2 * A)) {
                        const int sub = tt % EL;
                        for (int e = tt / EL; e < pend; e += A / EL) {
                            const int o = (int)pending[e];
                            uint64_t top = 0;
#pragma unroll
                            for (int i = 0; i < PER; i++) {
                                top = match_larger(top, edge(o, min(sub + EL * i, SC - 1), mypos[i]));
                                if (PER > 4 && i % 3 == 2) asm volatile("" : "+v"(top)::"memory");      // (all reads at once do not fit the registers)
                            }
                            top = other(top, by_1);
                            if (EL >= 4) top = other(top, by_2);
                            if (EL >= 8) top = other(top, by_4);
                            const uint32_t score = RAW ? (uint32_t)(top >> 32) : match_edge_score(top);
                            if (sub == 0) put(o, score == 0 ? 0 : match_key(score, o, match_edge_pattern(top)));
                        }
                    } else if (SG == 0 && c > 8 && pend * EIGHT <= A) {
                        const int e = tt / EIGHT, sub = tt % EIGHT;
                        if (e < pend) {
                            const int o = (int)pending[e];
                            uint64_t top = 0;
#pragma unroll 3
                            for (int i = 0; i < (c + EIGHT - 1) / EIGHT; i++) {
                                const int p = min(sub + EIGHT * i, c - 1);
                                top = match_larger(top, edge(o, p, s_pos[p]));
                            }
                            top = other(top, by_1);
                            top = other(top, by_2);
                            top = other(top, by_4);
                            const uint32_t score = RAW ? (uint32_t)(top >> 32) : match_edge_score(top);
                            if (sub == 0) put(o, score == 0 ? 0 : match_key(score, o, match_edge_pattern(top)));
                        }
                    } else {
                        for (int e = tt; e < pend; e += A) {
                            const int o = (int)pending[e];
                            put(o, propose(o, std::true_type{}));
                        }
                    }
                    match_sync<A>();
                    // a pattern's proposals into its list, two at a time
                    auto merge = [&](int p) {
                        constexpr int AT = 2;
                        constexpr bool EVEN = SG != 0 && (SG / 2 < 8 ? SG / 2 : 8) % AT == 0;      // whole batches, zeros behind the last
                        uint64_t *list = s_mem + p * g + r * KPL, *bkt = s_bkt + p * bucket;
                        uint64_t key[KPL], in[AT], ahead[AT];
                        // what the list will have no place for is known beforehand: one request for its places
                        const int asked = min(s_dem[p], bucket), had = s_occ[p], refused = had + asked - g;
                        int to = 0;
                        if (r == (g - 1) / KPL && refused > 0) to = atomicAdd(count, refused);
#pragma unroll
                        for (int i = 0; i < KPL; i++) key[i] = r * KPL + i < g ? list[i] : 0;
#pragma unroll
                        for (int u = 0; u < AT; u++) in[u] = EVEN || u < asked ? bkt[u] : 0;
                        for (int j = AT; in[0] != 0; j += AT) {
#pragma unroll
                            for (int u = 0; u < AT; u++) ahead[u] = bkt[j + u];      // (the last batch reads past the bucket)
                            uint64_t out[AT];
#pragma unroll
                            for (int u = 0; u < AT; u++) {
                                // key(i) = max(key(i), min(key(i - 1), in)): the keys are positive doubles and no NaN
                                uint64_t tail = key[0];      // the list's last key, in its last lane
#pragma unroll
                                for (int i = 1; i < KPL; i++) tail = (g - 1) % KPL == i ? key[i] : tail;
                                asm("s_nop 1" : "+v"(key[KPL - 1]));      // (a move between lanes reads a result two instructions later at the earliest)
                                uint64_t before = match_swap<(SG != 0 ? 0x111 : 0x138)>(key[KPL - 1]);      // row_shr:1, wave_shr:1
                                if (r == 0) before = in[u];
                                out[u] = match_smaller(tail, in[u]);
#pragma unroll
                                for (int i = KPL - 1; i > 0; i--) key[i] = match_larger(key[i], match_smaller(key[i - 1], in[u]));
                                key[0] = match_larger(key[0], match_smaller(before, in[u]));
                            }
                            if (r == (g - 1) / KPL) {
#pragma unroll
                                for (int u = 0; u < AT; u++)
                                    if (out[u] != 0) next[to++] = (uint16_t)match_column(out[u]);
                            }
#pragma unroll
                            for (int u = 0; u < AT; u++) in[u] = (EVEN ? j < bucket : j + u < asked) ? ahead[u] : 0;
                        }
#pragma unroll
                        for (int i = 0; i < KPL; i++)
                            if (r * KPL + i < g) list[i] = key[i];
                        if (r < bucket) bkt[r] = 0;
                        if (r == 0) {
                            s_dem[p] = 0;
                            s_occ[p] = min(had + asked, g);
                        }
                    };
                    // the same for a list that the lanes have no room for, by a wavefront: places by search, then everything moves there
                    auto merge_long = [&](int p) {
                        uint64_t *list = s_mem + p * g, *bkt = s_bkt + p * bucket;
                        const int asked = __builtin_amdgcn_readfirstlane(min(s_dem[p], bucket)), had = __builtin_amdgcn_readfirstlane(s_occ[p]);
                        const int refused = had + asked - g;
                        int to = 0;
                        if (lane == 0 && refused > 0) to = atomicAdd(count, refused);
                        to = __builtin_amdgcn_readfirstlane(to) - g;
                        const uint64_t mine = lane < asked ? bkt[lane] : 0;
                        int above = 0;      // kept keys in front of the proposal
                        for (int step = 1 << (31 - __clz(had | 1)); step > 0; step >>= 1)
                            if (above + step <= had && list[above + step - 1] > mine) above += step;
                        int at = above;
                        for (int j = 0; j < asked; j++) {
                            const uint64_t k = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(mine >> 32), j) << 32) |
                                               (uint32_t)__builtin_amdgcn_readlane((int)mine, j);
                            at += k > mine ? 1 : 0;
                        }
                        const int first = (int)~match_top<64>(~(uint32_t)above);
                        for (int s0 = (had - 1) & ~63; s0 >= 0 && s0 + 63 >= first; s0 -= 64) {      // the last keys first
                            const int s = s0 + lane;
                            const uint64_t k = s < had ? list[s] : 0;
                            int d = s;
                            for (int j = 0; j < asked; j++) d += __builtin_amdgcn_readlane(above, j) <= s ? 1 : 0;
                            if (s < had) {
                                if (d < g) list[d] = k;
                                else next[to + d] = (uint16_t)match_column(k);
                            }
                        }
                        if (lane < asked) {
                            if (at < g) list[at] = mine;
                            else next[to + at] = (uint16_t)match_column(mine);
                        }
                        if (lane == 0) {
                            s_dem[p] = 0;
                            s_occ[p] = min(had + asked, g);
                        }
                    };
                    if (longs) {
                        if constexpr (W == 64)
                            for (int p = wave; p < c; p += WAVES)
                                if (__builtin_amdgcn_readfirstlane(s_dem[p]) != 0) merge_long(p);
                    } else if constexpr (WAVES > 1) {
                        // a pattern to every list of lanes, in as many turns as that takes
                        for (int p = wave * rows + row; p < c; p += WAVES * rows)
                            if (s_dem[p] != 0) merge(p);
                    } else {
                        // the patterns with proposals, numbered through
                        int open = 0;
                        for (int p0 = 0; p0 < c; p0 += W) {
                            const bool has = p0 + lane < c && s_dem[p0 + lane] != 0;
                            uint64_t b = __ballot(has);
                            if (W < 64) b = (b >> (threadIdx.x & 63 & ~(W - 1))) & ((1ull << (W & 63)) - 1);
                            if (has) s_start[open + __popcll(b & ((1ull << lane) - 1))] = p0 + lane;
                            open += __popcll(b);
                        }
                        match_sync<W>();
                        for (int k = row; k < open; k += rows) merge(s_start[k]);
                    }
                    if (tt == 0) s_np[2 + ((round & 1) ^ 1)] = 0;
                    match_sync<A>();
                    pend = *count;
                    uint16_t *t = pending;
                    pending = next;
                    next = t;
                }
            };
            if constexpr (NT > 64) {
                // (4096 x 4096 fp16, 16 -> 8 columns left to the first wavefront: 2:8:64 164 -> 145 us, 2:8:32 60.5 -> 58.5; with
                // two wavefronts 3:8:8 244 -> 264 / 240 -> 222)
                late(std::integral_constant<int, NT>{}, NT >= 256 ? 8 : 16);
                __syncthreads();
                if (tt < 64) late(std::integral_constant<int, 64>{}, 0);
                __syncthreads();
            } else {
                late(std::integral_constant<int, NT>{}, 0);
                match_sync<NT>();
            }
        }

        // ---- closed form: zero columns beyond the end, then the columns that wait ----
        // Number k in descending column order takes free slot number k, the slots in descending pattern order.
        const int placed = real_cols - s_np[1];
        if (placed < cols) {
            const int npad = cols - real_cols;
            int16_t *s_wait = (int16_t *)s_arr;                  // waiting columns in descending order
            if (placed < real_cols) {
                int16_t *s_flag = s_wait + cols;
                for (int o = tt; o < cols; o += NT) s_flag[o] = 0;
                match_sync<NT>();
                for (int s = tt; s < cols; s += NT)
                    if (s_mem[s] != 0) s_flag[match_column(s_mem[s])] = 1;
                match_sync<NT>();
                // a column's number: those of the higher runs of LANES columns, then of the higher lanes of its own
                constexpr int LANES = NT < 64 ? NT : 64;
                int *s_runs = (int *)(s_flag + cols);
                const int lane = tt % LANES, nruns = (real_cols + LANES - 1) / LANES;
                auto waits = [&](int run) {
                    const int o = run * LANES + lane;
                    const uint64_t b = __ballot(o < real_cols && s_flag[o] == 0);
                    return LANES == 64 ? b : (b >> (threadIdx.x & 63 & ~(LANES - 1))) & ((1ull << (LANES & 63)) - 1);
                };
                for (int run = tt / LANES; run < nruns; run += NT / LANES) {
                    const uint64_t b = waits(run);
                    if (lane == 0) s_runs[run] = __popcll(b);
                }
                match_sync<NT>();
                for (int run = tt / LANES; run < nruns; run += NT / LANES) {
                    const uint64_t b = waits(run);
                    int k = 0;
                    for (int u = run + 1; u < nruns; u++) k += s_runs[u];
                    if ((b >> lane) & 1) s_wait[k + __popcll(b >> lane) - 1] = (int16_t)(run * LANES + lane);
                }
            }
            if (tt < 64) {
                constexpr int LANES = NT < 64 ? NT : 64;
                const int p0 = c - 1 - 2 * tt, p1 = p0 - 1;
                const int r0 = p0 >= 0 ? g - s_occ[p0] : 0, r1 = p1 >= 0 ? g - s_occ[p1] : 0;
                const int excl = match_prefix<LANES>(r0 + r1) - (r0 + r1);
                if (p0 >= 0) s_start[p0] = excl;
                if (p1 >= 0) s_start[p1] = excl + r0;
            }
            match_sync<NT>();
            for (int e = tt; e < cols; e += NT) {
                if (s_mem[e] != 0) continue;
                const int p = group_of(e), k = s_start[p] + (e - p * g) - s_occ[p];
                const int o = k < npad ? cols - 1 - k : (int)s_wait[k - npad];
                s_mem[e] = (1ull << 48) | (uint32_t)o;
            }
        }
    }

    // ---- the workgroup's slots, contiguous in val and idx ----
    __syncthreads();
    T *val = (T *)Q.val;
    auto elem = [&](const unsigned char *reg, uint64_t key, uint32_t ps, int j) {
        const int o = match_column(key), r = (int)((ps >> (4 * j)) & 15u);
        return ((const T *)reg)[at(o, r)];
    };
    if constexpr (SN != 0 && SG % 4 == 0) {
        if (Q.out4) {
            constexpr int BYTES = 4 * SN * (int)sizeof(T);
            constexpr int W = BYTES % 16 == 0 ? 4 : 2;          // words per store
            for (int e = 4 * tid; e < TILES * cols; e += 4 * THREADS) {
                const int tm = TILES == 1 ? 0 : SG != 0 ? e / cols : (int)(((uint64_t)e * Q.magic_cols) >> 32), slot = e - tm * cols;
                const int64_t t = tile0 + tm;
                if (t >= Q.outer) break;
                const unsigned char *reg = smem + head_bytes + (size_t)tm * Q.region_bytes;
                T v[4 * SN];
                int16_t o4[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const uint64_t k = ((const uint64_t *)(reg + Q.r_mem))[slot + u];
                    const uint32_t ps = s_pos[group_of(slot + u)];
                    o4[u] = (int16_t)match_column(k);
#pragma unroll
                    for (int j = 0; j < SN; j++) v[u * SN + j] = elem(reg, k, ps, j);
                }
                const int64_t to = t * (int64_t)cols + slot;
                uint2 raw;
                __builtin_memcpy(&raw, o4, 8);
                *(uint2 *)(Q.idx + to) = raw;
#pragma unroll
                for (int w = 0; w < BYTES / (4 * W); w++) {
                    if constexpr (W == 4) {
                        uint4 x;
                        __builtin_memcpy(&x, (const char *)v + 16 * w, 16);
                        ((uint4 *)(val + to * SN))[w] = x;
                    } else {
                        uint2 x;
                        __builtin_memcpy(&x, (const char *)v + 8 * w, 8);
                        ((uint2 *)(val + to * SN))[w] = x;
                    }
                }
            }
            return;
        }
    }
    for (int e = tid; e < TILES * cols; e += THREADS) {
        const int tm = (int)(((uint64_t)e * Q.magic_cols) >> 32), slot = e - tm * cols;
        const int64_t t = tile0 + tm;
        if (t >= Q.outer) break;
        const unsigned char *reg = smem + head_bytes + (size_t)tm * Q.region_bytes;
        const uint64_t k = ((const uint64_t *)(reg + Q.r_mem))[slot];
        const uint32_t ps = s_pos[group_of(slot)];
        const int64_t to = t * (int64_t)cols + slot;
        Q.idx[to] = (int16_t)match_column(k);
        for (int j = 0; j < n; j++) val[to * n + j] = elem(reg, k, ps, j);
    }
}

template <typename T, int NT, int CPT, int SN, int SM, int SG, bool RC>
static int match_launch(MatchParams &Q, hipStream_t stream, bool *done)
{
    *done = false;
    constexpr int TILES = NT <= 64 ? 256 / NT : 1, THREADS = NT <= 64 ? 256 : NT;
    const int cols = Q.cols, m = Q.m, c = Q.c, V = 16 / (int)sizeof(T);
    if (cols > NT * CPT || c > 128 || (NT < 64 && c > 2 * NT)) return NMG_OK;      // prefix sums: two patterns per lane
    if ((int64_t)TILES * cols >= 65536) return NMG_OK;                              // the magic divisions hold below 2^16
    auto up = [](int x, int a) { return (x + a - 1) / a * a; };
    int off = RC ? m * up(cols, V) * (int)sizeof(T) : up(cols * m * (int)sizeof(T), 16);
    Q.r_mem = off;
    off = up(off + cols * 8 + kMatchPad, 16);
    // Tiles of 16 columns with more than four patterns go through rounds over all columns to the end, those of a wavefront and less also with lists
    // that do not fit their lanes.  us, 4096 x 4096 fp16, rounds -> lists: 1:8:8 101 -> 62, 2:5:2 (20 columns) 275 -> 224, 1:4:4 (16) 104 -> 93, 2:8:1 314 -> 223,
    // 4:8:1 824 -> 434, 2:4:160 211 -> 123, 1:8:256 165 -> 82; but 1:8:2 (16) 115 -> 126.  (1:8:2 109 and 113 along the two dims, 125 and 130 with pending columns only.)
    Q.lanes_log2 = match_long(NT, c, Q.g, false) ? 6 : Q.g > 64 * match_list_keys(NT) ? 0 : Q.g <= 16 ? 3 : Q.g <= 32 ? 4 : Q.g <= 64 ? 5 : 6;
    if ((1 << Q.lanes_log2) > NT || (cols < 18 && c > 4)) Q.lanes_log2 = 0;
    Q.r_arr = off;
    off += match_scratch(match_long(NT, c, Q.g, Q.view.S % m != 0), cols, c, Q.g, match_bins_log2(NT, c), SG != 0 || Q.lanes_log2 != 0, Q.view.S % m != 0, cols / match_few(SG));
    Q.r_int = off;
    off = up(off + (kMatchTables * c + 4) * 4, 16);
    // workgroups that fit a CU's wavefronts (for tiles of several wavefronts four a SIMD, though six may fit: a partial block without
    // the list costs more than the other two give, 2000 x 3000 bf16 2:7:20 94 -> 109)
    constexpr int LDS = 160 * 1024, MOST = (NT > 64 && SM == 0 ? 4 : match_waves(NT, SM != 0, RC)) * 4 / (THREADS / 64);
    const int head = up(c * 8, 16);
    if (Q.view.S % m != 0) {
        // the classes of a partial block, and a list of its refused columns where that costs no workgroup of a CU (us, two workgroups without the
        // list against one with it: 3:6:100 fp32 2001 x 1999 102, 168)
        off = up(off + ((c + 1) & ~1) * 4 + c * 8, 16);
        const int with = up(off + cols * 2, 16);
        auto per_cu = [&](int region) { return std::min(MOST, LDS / (head + TILES * region)); };
        Q.listed = match_keys(NT, CPT) > 1 && (SG != 0 || per_cu(with) == per_cu(off));
        if (Q.listed) off = with;
    }
    // the tiles of a wavefront run the same offsets of their regions: spread them over the banks
    if (NT < 64)
        while (off % 256 != (NT == 16 ? 64 : 128)) off += 16;
    Q.region_bytes = off;
    const size_t lds = (size_t)head + (size_t)TILES * off;
    if (lds > LDS) return NMG_OK;
    // Two wavefronts per tile where every CU gets eight tiles and their data fits beside each other, else four: us with two /
    // four, 4096 x 4096 fp16 2:4:64 118 / 157 and 2:8:16 130 / 135, the latter in fp32 (22 KB a tile) 162 / 137;
    // 777 x 1001 fp16 2:4:64 (750 tiles) 52 / 39, 2:8:16 85 / 56.
    if (NT == 128 && (lds > 20 * 1024 || Q.outer < 8 * 256)) return NMG_OK;
    Q.out4 = cols % 4 == 0 && (uintptr_t)Q.val % 16 == 0 && (uintptr_t)Q.idx % 8 == 0;
    auto kern = match_kernel<T, NT, CPT, SN, SM, SG, RC>;
    if (lds > 64 * 1024)
        NMG_HIP_TRY(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int64_t grid = (Q.outer + TILES - 1) / TILES;
    NMG_REQUIRE(grid <= 0x7fffffffLL, NMG_ERR_UNSUPPORTED, "too many tiles (%lld)", (long long)grid);
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(THREADS), lds, stream, Q);
    NMG_HIP_TRY(hipGetLastError());
    *done = true;
    return NMG_OK;
}

// The patterns of this repository's benchmark and tests at their group sizes, in a source of their own (nmg_match_fixed.hip).
template <typename T> int match_fixed(MatchParams &Q, bool rc, hipStream_t stream, bool *done);

template <typename T, bool RC> static int match_dispatch(MatchParams &Q, hipStream_t stream, bool *done)
{
    const int n = Q.n, m = Q.m;
    const int fixed = match_fixed<T>(Q, RC, stream, done);
    if (fixed != NMG_OK || *done) return fixed;
    // Small tiles, a quarter of a wavefront each: what counts is the instructions of a proposal.  The kernels compiled for
    // a pattern, any g, need the fewest (4096 x 4096 fp16, any pattern -> compiled: 2:4:8 112 -> 75 us, 1:4:8 107 -> 69, 1:2:16
    // 131 -> 94, 1:5:4 164 -> 122).
    if (Q.cols <= 64 && m <= 5 && Q.c <= 6) {
        if (m == 2 && n == 1) return match_launch<T, 16, 4, 1, 2, 0, RC>(Q, stream, done);
        if (m == 3 && n == 1) return match_launch<T, 16, 4, 1, 3, 0, RC>(Q, stream, done);
        if (m == 3 && n == 2) return match_launch<T, 16, 4, 2, 3, 0, RC>(Q, stream, done);
        if (m == 4 && n == 1) return match_launch<T, 16, 4, 1, 4, 0, RC>(Q, stream, done);
        if (m == 4 && n == 2) return match_launch<T, 16, 4, 2, 4, 0, RC>(Q, stream, done);
        if (m == 4 && n == 3) return match_launch<T, 16, 4, 3, 4, 0, RC>(Q, stream, done);
        if (m == 5 && n == 1) return match_launch<T, 16, 4, 1, 5, 0, RC>(Q, stream, done);
        if (m == 5 && n == 4) return match_launch<T, 16, 4, 4, 5, 0, RC>(Q, stream, done);
    }
    // (a tile of many patterns: half a wavefront, 3:6:3 236 -> 184, 2:7:3 241 -> 171, 2:8:2 218 -> 166)
    if (Q.cols <= 64 && Q.c <= (Q.cols > 48 ? 15 : 32)) return match_launch<T, 16, 4, 0, 0, 0, RC>(Q, stream, done);
    if (Q.cols <= 128 && Q.c <= (Q.cols > 64 ? 20 : 60)) return match_launch<T, 32, 4, 0, 0, 0, RC>(Q, stream, done);
    if (Q.cols <= 256) return match_launch<T, 64, 4, 0, 0, 0, RC>(Q, stream, done);
    if (Q.cols <= 512) {
        const int rc = match_launch<T, 128, 4, 0, 0, 0, RC>(Q, stream, done);
        if (rc != NMG_OK || *done) return rc;
    }
    if (Q.cols <= 1024) return match_launch<T, 256, 4, 0, 0, 0, RC>(Q, stream, done);
    if (Q.cols <= 2560) return match_launch<T, 512, 5, 0, 0, 0, RC>(Q, stream, done);
    return match_launch<T, 1024, 4, 0, 0, 0, RC>(Q, stream, done);
}

template <typename T>
static int match_run(const void *dense, void *val, int16_t *idx, const ViewDev &view, int64_t outer, int n, int m, int g, int c, int cols,
               hipStream_t stream, bool *done)
{
    *done = false;
    if (m > 8 || n < 1 || c > 128 || cols < 16) return NMG_OK;
    MatchParams Q{};
    Q.dense = dense;
    Q.val = val;
    Q.idx = idx;
    Q.view = view;
    Q.outer = outer;
    Q.n = n;
    Q.m = m;
    Q.g = g;
    Q.c = c;
    Q.cols = cols;
    const int8_t *order = host_order(n, m);
    NMG_REQUIRE(order != nullptr, NMG_ERR_ARG, "invalid n:m = %d:%d", n, m);
    for (int p = 0; p < c; p++)
        for (int j = 0; j < n; j++) Q.masks[p / 4] |= 1u << (8 * (p % 4) + order[p * n + j]);
    Q.magic_cols = (((uint64_t)1 << 32) + cols - 1) / cols;
    Q.magic_g = (((uint64_t)1 << 32) + g - 1) / g;
    const bool rc = view.stride_g == 1 && view.stride_s != 1;
    // the widest load that every unit of the tile data is aligned to
    Q.unit = (int)sizeof(T);
    auto fits = [&](int64_t elements, int ub) { return elements * (int64_t)sizeof(T) % ub == 0; };
    for (int ub = 16; ub > (int)sizeof(T); ub /= 2) {
        const bool lines = rc ? fits(cols, ub) && fits(view.stride_s, ub)
                              : view.stride_s == 1 && fits(m, ub) && fits(view.stride_g, ub);
        if (lines && fits(view.stride_b, ub) && (uintptr_t)dense % ub == 0) {
            Q.unit = ub;
            break;
        }
    }
    return rc ? match_dispatch<T, true>(Q, stream, done) : match_dispatch<T, false>(Q, stream, done);
}

}  // namespace nmg
