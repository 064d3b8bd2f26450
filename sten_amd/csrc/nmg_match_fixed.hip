// The compressor's kernels for the patterns of this repository's benchmark and tests at their group sizes: pattern, list and tile
// extents folded in (4096 x 4096 fp16, any pattern -> compiled: 2:4:16 107 -> 64 us, 2:8:32 128 -> 71).  Apart from the others because they
// are compiled with other options (build.py).
#include "nmg_match.h"

namespace nmg {

template <typename T, bool RC> static int fixed(MatchParams &Q, hipStream_t stream, bool *done)
{
    auto is = [&](int n, int m, int g) { return Q.n == n && Q.m == m && Q.g == g; };
    if (is(2, 4, 16)) return match_launch<T, 32, 3, 2, 4, 16, RC>(Q, stream, done);
    if (is(1, 8, 32)) return match_launch<T, 64, 4, 1, 8, 32, RC>(Q, stream, done);
    if (is(3, 6, 12)) return match_launch<T, 64, 4, 3, 6, 12, RC>(Q, stream, done);
    if (is(2, 8, 32)) return match_launch<T, 256, 4, 2, 8, 32, RC>(Q, stream, done);
    if (is(4, 8, 32)) return match_launch<T, 512, 5, 4, 8, 32, RC>(Q, stream, done);      // (fp32 tiles leave one workgroup per CU)
    return NMG_OK;
}

template <typename T> int match_fixed(MatchParams &Q, bool rc, hipStream_t stream, bool *done)
{
    return rc ? fixed<T, true>(Q, stream, done) : fixed<T, false>(Q, stream, done);
}

template int match_fixed<float>(MatchParams &, bool, hipStream_t, bool *);
template int match_fixed<__half>(MatchParams &, bool, hipStream_t, bool *);
template int match_fixed<__hip_bfloat16>(MatchParams &, bool, hipStream_t, bool *);

}  // namespace nmg
