// The columns that a chunk of fp_stream_kernel stages (fp_stream.hpp), the host's bound
// on them, and the rows of a ray.  No HIP in it: the arithmetic is tested on the host.
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

// Rows of a ray: the k in [0, n) with 0 <= x_k <= hi, x_k accumulated from x0 in steps
// of off; monotone, so an interval.  [fin, fout): rows with x_k at least a quarter of a
// column (less FP32 rounding) inside both ends.  The sums of the accumulation round to
// half an ulp of hi a row, together less than tol; a crossing that close to a row is
// decided by replaying it up to there.  Where the ray moves so little a row that tol
// is more than a quarter of a row (a view along the axis, give or take rounding), it
// stays on its side of both ends, or all rows are replayed.
CTR_HOST_DEVICE void fp_ray_rows(double x0, double off, double hi, int n, int& kin, int& kout,
                                 int& fin, int& fout)
{
    const double dn = n, tol = fma(2.3e-16 * dn, hi, 1e-8);
    const bool creep = fabs(off) < 4 * tol;
    const double inv = 1.0 / (creep ? 1.0 : off);
    const double ta = -x0 * inv, tb = (hi - x0) * inv;
    const double lo = fmin(ta, tb), up = fmax(ta, tb);
    const double eps = tol * fabs(inv);
    bool tie = fabs(lo - rint(lo)) < eps || fabs(up - rint(up)) < eps;
    kin = static_cast<int>(fmin(fmax(ceil(lo), 0.0), dn));
    kout = static_cast<int>(fmin(fmax(floor(up) + 1.0, 0.0), dn));
    const float fn = static_cast<float>(n), q = 0.25f * fabsf(static_cast<float>(inv));
    fin = static_cast<int>(fminf(fmaxf(ceilf(static_cast<float>(lo) + q), 0.0f), fn));
    fout = static_cast<int>(fminf(fmaxf(floorf(static_cast<float>(up) - q) + 1.0f, 0.0f), fn));
    if (creep) {
        const double drift = fma(dn, fabs(off), tol);
        tie = off != 0.0 && (fabs(x0) < drift || fabs(x0 - hi) < drift);
        kin = fin = 0;
        kout = x0 >= 0 && x0 <= hi ? n : 0;
        fout = x0 >= 0.25 + drift && x0 <= hi - 0.25 - drift ? n : 0;
    }
    if (tie) {
        const int ra = creep ? 0 : static_cast<int>(fmin(fmax(rint(lo), -1.0), dn));
        const int rb = creep ? n - 1 : static_cast<int>(fmin(fmax(rint(up), -1.0), dn));
        double x = x0;
        int k = 0;
        const auto inside = [&] { return x >= 0 && x <= hi; };
        if (creep) {
            kin = n;
            kout = 0;
            for (; k < n; ++k, x += off)
                if (inside()) {
                    kin = k < kin ? k : kin;
                    kout = k + 1;
                }
        } else {
            for (; k < ra; ++k) x += off;
            if (ra >= 0 && ra < n) kin = inside() ? ra : ra + 1;
            for (; k < rb; ++k) x += off;
            if (rb >= 0 && rb < n) kout = inside() ? rb + 1 : rb;
        }
    }
    if (kin >= kout) kin = kout = 0;
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
