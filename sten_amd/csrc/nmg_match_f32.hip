#include "nmg_match.h"

namespace nmg {

int match_f32(const void *dense, void *val, int16_t *idx, const ViewDev &view, int64_t outer, int n, int m, int g, int c, int cols,
              hipStream_t stream, bool *done)
{
    return match_run<float>(dense, val, idx, view, outer, n, m, g, c, cols, stream, done);
}

}  // namespace nmg
