// The columns that a chunk of fp_stream_kernel stages (fp_stream.hpp), and the
// host's bound on them.  No HIP in it: the arithmetic is tested on the host.
#pragma once

#include <algorithm>
#include <cmath>

#include "include/ctr_api.h"

#if defined(__HIPCC__)
#define CTR_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define CTR_HOST_DEVICE inline
#endif

namespace ctr {

struct FpSpan {
    int first, cols;
};

// Columns for rays between xmin and xmax on rows of rowlen pixels, at most `most`
// of them: every tap of a ray with 0 <= x <= rowlen - 1, with one column of margin
// each side (the bounds are FP32).  The right tap of a ray that stands exactly on
// the last column is column rowlen; its weight is 0, but it is read, so it counts
// (fp_stage writes zeros past the row): 0 times what the LDS held before is NaN
// for some leftovers.
CTR_HOST_DEVICE FpSpan fp_span(float xmin, float xmax, int rowlen, int most)
{
    const int lo = static_cast<int>(floorf(fmaxf(xmin, -4.0f))) - 1;
    const int hi = static_cast<int>(floorf(fminf(xmax, 1e6f))) + 2;
    const int first = lo < 0 ? 0 : lo < rowlen ? lo : rowlen - 1;
    const int last = hi < rowlen ? hi : rowlen, n = last - first + 1;
    return {first, n < 1 ? 1 : n < most ? n : most};
}

// Columns the rays of one fp_stream_kernel chunk can span: 64 channels at up to
// sqrt(2) ds / pixel per channel, one column per further row, the drift of a ray
// that is on the image across the other views (at most the image's
// half-diagonal times sqrt(2) per radian, doubled for the second order), and 6:
// fp_span's margins and the right tap.
inline bool fp_stream_applies(const ctr_geom& g, int views, int rows, int span_max)
{
    const double pmin = std::min(std::fabs(g.dx), std::fabs(g.dy));
    const double pmax = std::max(std::fabs(g.dx), std::fabs(g.dy));
    if (!(pmin > 0) || !(g.ds > 0)) return false;
    const double r = 0.5 * std::hypot(g.nx + 2 * std::fabs(g.offset_x),
                                      g.ny + 2 * std::fabs(g.offset_y)) * pmax / pmin;
    const double turn = (views - 1) * std::fabs(g.orbit);
    const double span = 63 * std::sqrt(2.0) * g.ds / pmin + (rows - 1) * pmax / pmin +
                        1.5 * r * turn * (1.0 + 2.0 * turn) + 6.0;
    // steps within 2 columns a row, one plane within a 31-bit buffer range
    return span <= span_max && pmax <= 1.9 * pmin && 16LL * g.nx * g.ny < (1LL << 31);
}

}  // namespace ctr
