// Per-(pixel tile, view) fan-beam geometry of bp_fan_2d and bp_fan_2d_angle: the
// policy of the BP engine and of the gather transpose, which evaluate the same bits
// pixel by pixel (FanGeo), and of the stream kernel, the default forward, which
// takes runs of pixels from a polynomial (FanRun).  Stream and transpose share the
// anchors; their positions differ by rounding and by what the polynomial leaves
// out (fan_run_order: 1e-6 channel and 4e-7 of the weight at most), so the pair is
// adjoint to about 1e-6, and a pixel that lies within that of the detector's end
// may count in one and not in the other.
//
// For a pixel at (x, y) and source angle beta (source at
// (-dso sin b, dso cos b)) the reference computes, in FP64
// (src/bp_fan_2d.cc:66-70):
//     d = dso + x sin b - y cos b,  r = x cos b + y sin b,
//     s = atan2(r, d) * dsd/ds + cents,  w = dsd^2 / (d^2 + r^2).
// Here the tile anchor (xc, yc) is evaluated once in FP64 and every pixel of
// the tile is expressed relative to it.  With (dd, dr) the pixel's offsets
// of (d, r) from the anchor's (dc, rc) and Lc^2 = dc^2 + rc^2,
//     tan(gamma - gamma_c) = u = (dr dc - dd rc) / (Lc^2 + dd dc + dr rc),
// which is a ratio of two functions linear in the pixel offsets (i, j), and
//     d^2 + r^2 = Lc^2 (1 + e)^2 (1 + u^2),  e = (dd dc + dr rc)/Lc^2.
// So s = s_c + (dsd/ds) atan(u) and w = (dsd^2/Lc^2) / ((1+e)^2 (1+u^2)),
// evaluated per pixel in FP32 on small numbers: the channel position keeps
// ~1e-6 channel accuracy where a direct FP32 evaluation of s ~ 700 would
// lose ~5e-5.  The FP64 anchor carries the large part (s_c) exactly.
#pragma once

#include <hip/hip_runtime.h>

#include "bp_stream.hpp"
#include "ctr_common.hpp"
#include "tile_common.hpp"

namespace ctr {

struct alignas(16) FanAnchor {
    float ai, aj;  // numerator slopes per pixel step in x / y, pre-scaled
    float bi, bj;  // denominator slopes per pixel step
    float b0;      // denominator constant
    float fc;      // anchor channel position minus is0
    int is0;       // first channel of the staged detector span
    int inside;    // 1: every pixel of the tile lands strictly inside [0, ns-1]
    int nch;       // channels from is0 the tile's taps can touch (one of margin)
    float frac;    // the anchor's channel position is is0 + whole + frac
    int whole;
    int pad;
};

// Geometry of one fan problem as the kernels see it.
struct FanProblem {
    double dso, dsd, ds, cents, dx, dy;
    int ns, na, nx, ny;
    // polynomial coefficients in v = k*u (k = dsd/ds):
    //   atan:      ds(v) = v * (1 + v2*(p1 + v2*p2)),  p1 = -1/(3k^2), p2 = 1/(5k^4)
    //   1/(1+u^2) = 1 + v2*(g1 + v2*g2),                 g1 = -1/k^2,   g2 = 1/k^4
    float p1, p2, g1, g2;
    float k;          // dsd/ds in FP32 (exact mode)
    double kd, idsd;  // dsd/ds and 1/dsd
    float roff;       // channels a run of 8 pixels stays within of its centre
    float dxd2;       // (dx / dsd)^2
};

// The part of an anchor the stream kernel's pixels read, in one LDS line.
struct alignas(16) FanStreamAnchor {
    float ai, aj, bi, bj, b0, frac;
    int is0, nch;  // nch: FanAnchor::nch | whole << 16
};

struct FanTables {
    const double* xpos;     // [nx]   (src/bp_fan_2d.cc:37-40)
    const double* ypos;     // [ny]
    const double* sincos;   // [2na]  (sin, cos) of the source angle
};

// Anchor of the tile whose local pixel offsets span [ilo, ihi] x [jlo, jhi]
// around (xc, yc).  FP64 for the anchor itself, FP32 for the span bounds:
// the series of fan_pixel (EXACT: atanf), whose error the margins of the span
// and of `inside` cover many times over.
template <bool EXACT>
__device__ inline FanAnchor fan_anchor(const FanProblem& P, double xc, double yc, double sb,
                                       double cb, int ilo, int ihi, int jlo, int jhi)
{
    const double d = P.dso + xc * sb - yc * cb;
    const double r = xc * cb + yc * sb;
    const double L2 = d * d + r * r;
    const double inv = 1.0 / L2;
    const double k = P.kd;
    const double sc = atan2(r, d) * k + P.cents;
    // dd = i*dx*sb + j*dy*cb,  dr = i*dx*cb - j*dy*sb  (y decreases with iy)
    const double nI = P.dx * (cb * d - sb * r) * inv;
    const double nJ = -P.dy * (sb * d + cb * r) * inv;
    const double eI = P.dx * (sb * d + cb * r) * inv;
    const double eJ = P.dy * (cb * d - sb * r) * inv;
    // The channel offset is monotone along any line (a ratio of linear
    // functions through atan), so the tile's extreme channels are at corners.
    const float fnI = static_cast<float>(nI), fnJ = static_cast<float>(nJ);
    const float feI = static_cast<float>(eI), feJ = static_cast<float>(eJ);
    const float fk = static_cast<float>(k);
    float lo = 0.0f, hi = 0.0f;
    const int ci[2] = {ilo, ihi}, cj[2] = {jlo, jhi};
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const float num = fnI * ci[a] + fnJ * cj[b], den = 1.0f + feI * ci[a] + feJ * cj[b];
            float dsv;
            if constexpr (EXACT) {
                dsv = fk * atanf(num / den);
            } else {
                const float v = fk * num * __builtin_amdgcn_rcpf(den), v2 = v * v;
                dsv = fmaf(v, v2 * fmaf(v2, P.p2, P.p1), v);
            }
            lo = fminf(lo, dsv);
            hi = fmaxf(hi, dsv);
        }
    const double smin = sc + lo, smax = sc + hi;
    const int is0 = static_cast<int>(floor(smin)) - 1;
    const double iq = sqrt(L2) * P.idsd;  // 1 / sqrt(dsd^2 / Lc^2)
    FanAnchor A;
    A.ai = static_cast<float>(k * nI * iq);
    A.aj = static_cast<float>(k * nJ * iq);
    A.bi = static_cast<float>(eI * iq);
    A.bj = static_cast<float>(eJ * iq);
    A.b0 = static_cast<float>(iq);
    A.fc = static_cast<float>(sc - is0);
    A.is0 = is0;
    A.inside = (smin >= 0.25 && smax <= P.ns - 1.25) ? 1 : 0;
    A.nch = static_cast<int>(floor(smax)) + 3 - is0;
    A.whole = static_cast<int>(floor(sc)) - is0;
    A.frac = static_cast<float>(sc - floor(sc));
    A.pad = 0;
    return A;
}

// Channel position (relative to is0) and weight of local pixel (fi, fj).
// Default mode: short series (the host checks |u| stays small enough);
// EXACT: atan and 1/(1+u^2) evaluated directly.
template <bool EXACT>
__device__ __forceinline__ void fan_pixel(const FanProblem& P, const FanAnchor& A, float fi,
                                          float fj, float& f, float& w)
{
    const float num = fmaf(A.ai, fi, A.aj * fj);
    const float den = fmaf(A.bi, fi, fmaf(A.bj, fj, A.b0));
    const float rd = __builtin_amdgcn_rcpf(den);
    const float v = num * rd;  // k * u, channels
    if constexpr (EXACT) {
        const float u = v / P.k;
        f = A.fc + P.k * atanf(u);
        w = rd * rd / fmaf(u, u, 1.0f);
    } else {
        const float v2 = v * v;
        const float t = v2 * fmaf(v2, P.p2, P.p1);
        f = A.fc + fmaf(v, t, v);
        w = rd * rd * fmaf(v2, fmaf(v2, P.g2, P.g1), 1.0f);
    }
}

// Host side (fan_bp.hip): geometry checks for a TW x TH tiling, the
// channels one tile's span needs (lmax) and whether the series is accurate
// enough (exact = false) -- and the smallest source-to-pixel distance.
int fan_problem(const ctr_geom& g, int TW, int TH, FanProblem& P, int& lmax, bool& exact);
double fan_min_distance(const ctr_geom& g, int TW, int TH);
// Which FanRun is accurate on runs of 8 pixels: 1 short, 2 long, 0 neither.
int fan_run_order(const ctr_geom& g);

// Policy for the BP engine.
template <bool EXACT>
struct FanGeo {
    using Problem = FanProblem;
    using Tables = FanTables;
    using Anchor = FanAnchor;
    static constexpr bool kGatherFrac = false;
    __device__ static Anchor anchor(const Problem& P, const Tables& T, const TileFrame& F,
                                    int view, int ilo, int ihi, int jlo, int jhi)
    {
        return fan_anchor<EXACT>(P, T.xpos[F.ic], T.ypos[F.jc], T.sincos[2 * view],
                          T.sincos[2 * view + 1], ilo, ihi, jlo, jhi);
    }
    __device__ __forceinline__ static void pixel(const Problem& P, const Anchor& A, float fi,
                                                 float fj, float& f, float& w)
    {
        fan_pixel<EXACT>(P, A, fi, fj, f, w);
    }
    // the series' addends p1 and g1 meet the uniform p2 and g2 in one FMA each
    __device__ __forceinline__ static void pin(Problem& P)
    {
        asm volatile("" : "+v"(P.p1), "+v"(P.g1));
    }
    // Level line s = s_star in pixel-index coordinates: the ray at fan angle
    // g* = (s_star - cents) ds / dsd, r - tan(g*) d = 0, i.e.
    // L(ix, iy) = pi ix + qj iy + rr >= 0 exactly where s >= s_star for every
    // pixel in front of the source (d > 0; the host admits no other).  g* is
    // clamped to +-1.47 rad: every admitted pixel has |g| <= asin(0.95), so a
    // clamped line still bounds the same set of image pixels.
    __device__ static void boundary(const Problem& P, const Tables& T, int view, double s_star,
                                    double& pi, double& qj, double& rr)
    {
        const double sb = T.sincos[2 * view], cb = T.sincos[2 * view + 1];
        const double g = fmin(fmax((s_star - P.cents) * P.ds / P.dsd, -1.47), 1.47);
        const double t = tan(g);
        const double pp = cb - t * sb, qq = sb + t * cb, r0 = -t * P.dso;
        const double x0 = T.xpos[0], y0 = T.ypos[0];
        const double xs = P.nx > 1 ? (T.xpos[P.nx - 1] - x0) / (P.nx - 1) : P.dx;
        const double ys = P.ny > 1 ? (T.ypos[P.ny - 1] - y0) / (P.ny - 1) : -P.dy;
        pi = pp * xs;
        qj = qq * ys;
        rr = pp * x0 + qq * y0 + r0;
    }
};

// Runs of the stream kernel (bp_stream.hpp).  Along a row, with d the offset
// from the run's centre, the squared distance from the source is a quadratic
// in d, so w(d) = w0 / (1 - a1 d + b d^2), b = w0 (dx / dsd)^2, whose series
// w0 (1 + r1 d + r2 d^2 + ...) has r1 = a1, r2 = a1^2 - b, r_n+1 = a1 r_n - b r_n-1;
// and the angle's derivative is a constant over that distance, so f(d) is the
// integral of the same series: f0 + c1 (d + r1 d^2 / 2 + r2 d^3 / 3 + ...).
// Kept: f to d^3 and w to d^2 (LONG: d^4 and d^3); the next term of each goes
// into the lower ones by its least-squares fit over the run's eight pixels,
//     d^3 ~ 9.25 d, d^4 ~ 12.786 d^2 - 18.56, d^5 ~ 15.833 d^3 - 46.75 d,
// which leaves 1/4, 1/6.8 and 1/16 of it.  fan_run_order says which form, if
// any, leaves less than the rounding of f and w.  Against FP64 the BP of filtered
// scans (210^2 to 1024^2, 1 to 30 slices) is 0.6e-7 to 3.6e-7 relative L2 off, the
// engine kernel on the same data 0.9e-7 to 3.8e-7, and on none of them less; on
// sinograms of one sign 16 slices are up to 1.13 times the engine's 2.4e-7 (chains
// of 90 views against 64).
template <bool LONG>
struct FanRun : FanGeo<false> {
    using StreamAnchor = FanStreamAnchor;
    static constexpr int kRunDegree = LONG ? 4 : 3;
    __device__ __forceinline__ static StreamAnchor pack(const Anchor& A)
    {
        return StreamAnchor{A.ai, A.aj, A.bi, A.bj, A.b0, A.frac, A.is0, A.nch | A.whole << 16};
    }
    __device__ __forceinline__ static RunPoly run(const Problem& P, const StreamAnchor& A, float fi,
                                                  float fj)
    {
        const float num = fmaf(A.ai, fi, A.aj * fj);
        const float den = fmaf(A.bi, fi, fmaf(A.bj, fj, A.b0));
        const float rd = __builtin_amdgcn_rcpf(den);
        const float v0 = num * rd, e = A.bi * rd;
        const float g = fmaf(-v0, e, A.ai * rd);  // dv/dd
        const float v2 = v0 * v0;
        const float q = fmaf(v2, fmaf(v2, P.g2, P.g1), 1.0f);  // 1 / (1 + u^2)
        RunPoly R;
        run_base(R, A.nch >> 16, A.frac, fmaf(v0, v2 * fmaf(v2, P.p2, P.p1), v0), P.roff);
        R.w0 = rd * rd * q;
        R.c1 = g * q;
        const float a1 = -2.0f * fmaf(-P.g1 * v0, R.c1, e);
        const float b = R.w0 * P.dxd2;
        const float r2 = fmaf(a1, a1, -b), r3 = a1 * (r2 - b);
        R.c2 = 0.5f * R.c1 * a1;
        R.c3 = (1.0f / 3) * R.c1 * r2;
        R.c4 = 0.25f * R.c1 * r3;
        R.w1 = R.w0 * a1;
        R.w2 = R.w0 * r2;
        R.w3 = R.w0 * r3;
        if constexpr (LONG) {
            const float r4 = fmaf(a1, r3, -b * r2);
            const float c5 = 0.2f * R.c1 * r4, w4 = R.w0 * r4;
            R.c1 = fmaf(-46.75f, c5, R.c1);
            R.c3 = fmaf(15.833f, c5, R.c3);
            R.w0 = fmaf(-18.56f, w4, R.w0);
            R.w2 = fmaf(12.786f, w4, R.w2);
        } else {
            R.c0 = fmaf(-18.56f, R.c4, R.c0);
            R.c2 = fmaf(12.786f, R.c4, R.c2);
            R.w1 = fmaf(9.25f, R.w3, R.w1);
        }
        return R;
    }
};

}  // namespace ctr
