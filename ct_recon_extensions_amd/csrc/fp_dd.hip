// Distance-driven parallel FP (src/fp_par_2d.cc:396-543; the TF FP op's
// method "disdriven") and the gradient the reference defines for it
// (src/fp_par_2d.cc:548-655), for gfx950.  Both are bit-identical to the
// reference's CPU path in float32 and float64: the reference's operation
// order and its float / double mix are kept, with contraction off, and the
// work is split only where the reference's sums are independent (one thread
// per (channel, view) for the FP, one per pixel for the gradient).
//
// FP, per channel and per row (x-branch; per column for the y-branch): the
// channel's footprint [left, right] (centre -+ half a channel width, in pixel
// units) averages the cell values (img[v] + img[v+1]) / 2 of the cells v it
// overlaps, weighted by the overlap; row averages are summed and scaled by
// |dy/cos| (|dx/sin|).  The reference's cell index is unsigned: a row whose
// footprint starts left of the first cell turns floor(left) < 0 into a huge
// index and adds nothing on the x86-64 build; that rule is kept.  The y-branch
// reads a transposed copy of the image so that a footprint's cells are
// contiguous.
//
// Gradient, per pixel and view: the span [mid - o1, mid + o1] of the pixel on
// the detector (one-sided at the first and last pixel along the branch's
// axis) and the channels whose cells it overlaps, each adding
// overlap * proj / 2, times the view's weight.  ceil(left - 1/2) < 0 adds
// nothing (the reference's unsigned index again); channels past ns - 1, which
// the reference reads beyond the row, are not read.  This pair is not an
// exact transpose (the reference's gradient approximates one); it is the
// pair the reference's ops use.
#include "ctr_common.hpp"
#include "interleave.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

#pragma clang fp contract(off)

namespace ctr {
namespace {

struct DdProblem {
    int ns, na, nx, ny, nbatch;
    double dx, dy;
};

template <typename T>
__global__ void dd_transpose_kernel(const T* __restrict__ src, T* __restrict__ dst, int ny, int nx)
{
    __shared__ T tile[32][33];
    const size_t base = static_cast<size_t>(blockIdx.z) * nx * ny;
    const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int y = y0 + r, x = x0 + threadIdx.x;
        if (y < ny && x < nx) tile[r][threadIdx.x] = src[base + static_cast<size_t>(y) * nx + x];
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int x = x0 + r, y = y0 + threadIdx.x;
        if (y < ny && x < nx) dst[base + static_cast<size_t>(x) * ny + y] = tile[threadIdx.x][r];
    }
}

// One thread per (channel, view) and NB slices, a wavefront per 64 channels
// of a view and 4 views per workgroup; data[b][u][v] is the image
// (x-branch: u = iy, v = ix) or its transpose (y-branch: u = ix, v = iy).
constexpr int kDdViews = 4;

template <typename T, int NB>
__global__ __launch_bounds__(64 * kDdViews) void fp_dd_kernel(const T* __restrict__ img,
                                                   const T* __restrict__ imgT,
                                                   T* __restrict__ proj,
                                                   const double* __restrict__ sc,
                                                   const double* __restrict__ bo,
                                                   const int* __restrict__ usex, DdProblem P)
{
    const int is = blockIdx.x * 64 + threadIdx.x;
    const int ia = blockIdx.y * kDdViews + threadIdx.y, b0 = blockIdx.z * NB;
    if (is >= P.ns || ia >= P.na) return;
    const int nb = min(NB, P.nbatch - b0);
    const bool bx = usex[ia] != 0;
    const double dw = bx ? fabs(P.dy / sc[2 * ia + 1]) : fabs(P.dx / sc[2 * ia]);
    const int nu = bx ? P.ny : P.nx, nv = bx ? P.nx : P.ny;
    const T* data = (bx ? img : imgT) + static_cast<size_t>(b0) * P.nx * P.ny;
    const size_t slice = static_cast<size_t>(P.nx) * P.ny;
    const double* b = bo + 3 * (static_cast<size_t>(ia) * P.ns + is);
    double left = b[0] - b[2], right = b[0] + b[2];
    const double off = b[1];
    if (left > right) {
        const double t = left;
        left = right;
        right = t;
    }
    T sum[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) sum[k] = T(0);
    for (int u = 0; u < nu; ++u) {
        T tsum[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k) tsum[k] = T(0);
        T lsum = T(0);
        const double fl = floor(left);
        // cells past nv - 2 are skipped by the reference, so the loop stops
        // there (the same sums, and a bounded trip count for any geometry)
        if (fl >= 0 && fl < nv - 1) {
            const double vend = fmin(ceil(right), static_cast<double>(nv - 1));
            const T* row = data + static_cast<size_t>(u) * nv;
            for (unsigned int v = static_cast<unsigned int>(fl); static_cast<double>(v) < vend; ++v) {
                const double len = fmin(static_cast<double>(v + 1), right) -
                                   fmax(static_cast<double>(v), left);
                // every slice's cell pair loaded first (a slice past the
                // batch re-reads the last one and is not added)
                T c0[NB], c1[NB];
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const T* q = row + static_cast<size_t>(min(k, nb - 1)) * slice + v;
                    c0[k] = q[0];
                    c1[k] = q[1];
                }
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    if (k < nb) {
                        const T pair = c0[k] + c1[k];
                        tsum[k] = static_cast<T>(static_cast<double>(tsum[k]) +
                                                 len * static_cast<double>(pair) / 2);
                    }
                }
                lsum = static_cast<T>(static_cast<double>(lsum) + len);
            }
        }
        if (lsum > 0) {
            if constexpr (std::is_same<T, float>::value) {
                // The float quotients tsum / lsum, correctly rounded, from one
                // FP64 reciprocal: q = tsum * RN(1 / lsum) in FP64 is within
                // 2^-52 (relative) of the exact quotient, and a quotient of two
                // floats is never an exact float midpoint and lies at least
                // 2^-49 (relative) from every one (the midpoint has 25
                // significant bits and lsum 24, so tsum - m lsum is a nonzero
                // multiple of 2^-49 |m lsum|): rounding q to float gives the
                // float division's result.
                const double r = 1.0 / static_cast<double>(lsum);
#pragma unroll
                for (int k = 0; k < NB; ++k)
                    sum[k] = sum[k] + static_cast<float>(static_cast<double>(tsum[k]) * r);
            } else {
#pragma unroll
                for (int k = 0; k < NB; ++k) sum[k] = sum[k] + tsum[k] / lsum;
            }
        }
        left += off;
        right += off;
    }
#pragma unroll
    for (int k = 0; k < NB; ++k)
        if (k < nb)
            proj[(static_cast<size_t>(b0 + k) * P.na + ia) * P.ns + is] =
                static_cast<T>(static_cast<double>(sum[k]) * dw);
}

// One thread per pixel and NB slices; pos[view][stride][2] as ctr_fp_grad_tables.
template <typename T, int NB>
__global__ __launch_bounds__(256) void fp_dd_grad_kernel(const T* __restrict__ proj,
                                                         T* __restrict__ img,
                                                         const double* __restrict__ weights,
                                                         const double* __restrict__ pos,
                                                         const int* __restrict__ usex, int stride,
                                                         DdProblem P)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.nx * P.ny) return;
    const int ix = i % P.nx, iy = i / P.nx;
    const int b0 = blockIdx.y * NB, nb = min(NB, P.nbatch - b0);
    const size_t sslice = static_cast<size_t>(P.na) * P.ns;
    const T* pr = proj + static_cast<size_t>(b0) * sslice;
    double sum[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) sum[k] = 0.0;
    for (int ia = 0; ia < P.na; ++ia) {
        const bool bx = usex[ia] != 0;
        const double* pp = pos + 2 * (static_cast<size_t>(ia) * stride + (bx ? iy : ix));
        const double begin = pp[0], off = pp[1];
        double mid, left, right;
        if (bx) {
            mid = begin + off * ix;
            left = ix == 0 ? mid : mid - off;
            right = ix == P.nx - 1 ? mid : mid + off;
        } else {
            mid = begin + off * iy;
            left = iy == 0 ? mid : mid - off;
            right = iy == P.ny - 1 ? mid : mid + off;
        }
        if (left > right) {
            const double t = left;
            left = right;
            right = t;
        }
        double tmp[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k) tmp[k] = 0.0;
        const double c0 = ceil(left - 0.5);
        if (c0 >= 0 && c0 < P.ns) {
            const double cend = fmin(floor(right + 0.5), static_cast<double>(P.ns - 1));
            const T* row = pr + static_cast<size_t>(ia) * P.ns;
            for (unsigned int is = static_cast<unsigned int>(c0); static_cast<double>(is) <= cend;
                 ++is) {
                const double len = fmin(static_cast<double>(is) + 0.5, right) -
                                   fmax(static_cast<double>(is) - 0.5, left);
                // every slice's value loaded first (a slice past the batch
                // re-reads the last one and is not added)
                T val[NB];
#pragma unroll
                for (int k = 0; k < NB; ++k)
                    val[k] = row[static_cast<size_t>(min(k, nb - 1)) * sslice + is];
#pragma unroll
                for (int k = 0; k < NB; ++k)
                    if (k < nb) tmp[k] += len * static_cast<double>(val[k]) / 2;
            }
        }
        const double w = weights[ia];
#pragma unroll
        for (int k = 0; k < NB; ++k) sum[k] += tmp[k] * w;
    }
#pragma unroll
    for (int k = 0; k < NB; ++k)
        if (k < nb) img[static_cast<size_t>(b0 + k) * P.nx * P.ny + i] = static_cast<T>(sum[k]);
}

// ---- float32, on interleaved planes.
//
// What bounds both directions is VALU issue, most of it the reference's mixed
// float / double arithmetic per cell (channel) and slice, and the fewer
// instructions that takes:
//  * cells (img[v] + img[v+1], a float sum) and channels lie interleaved in fours
//    of slices, so a cell of four slices is one 16-byte load with one address;
//    eight slices share a row's (a view's) geometry;
//  * the first cell of a row starts the sum: (float)(0 + len pair / 2);
//  * a cell the footprint covers whole has len = 1: its term pair / 2 is exact and
//    (float)((double)tsum + pair / 2) is the float FMA of 0.5, pair and tsum (the
//    double sum of two floats rounds to the correctly rounded float sum, 53 >=
//    2 24 + 2); likewise the gradient's double sum takes 0.5 val in one FMA;
//  * len pair / 2 is (0.5 len) pair: halving is exact;
//  * the reciprocal of lsum comes from v_rcp_f64 and two Newton steps, within
//    2^-51 of 1 / lsum, which the rounding argument above (2^-49) admits.
// 8 x 512^2, 720 views, 729 channels: FP 2.47 -> 1.05 ms, gradient 2.06 -> 1.00 ms.

// rows[plane][y][x][IL] = cells (x, x+1) of row y, cols[plane][x][y][IL] = cells (y,
// y+1) of column x; the last cell of a line is not read, slices past the batch
// are zero.
template <int IL>
__global__ __launch_bounds__(256) void dd_cells_kernel(const float* __restrict__ img,
                                                       float* __restrict__ rows,
                                                       float* __restrict__ cols, int ny, int nx,
                                                       int nbatch)
{
    __shared__ float tile[IL][33][34];
    const size_t slice = static_cast<size_t>(nx) * ny;
    const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 32, b0 = blockIdx.z * IL;
    for (int e = threadIdx.y * 32 + threadIdx.x; e < 33 * 33; e += 256) {
        const int y = y0 + e / 33, x = x0 + e % 33;
#pragma unroll
        for (int b = 0; b < IL; ++b)
            tile[b][e / 33][e % 33] = y < ny && x < nx && b0 + b < nbatch
                                          ? img[(b0 + b) * slice + static_cast<size_t>(y) * nx + x]
                                          : 0.0f;
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int c = threadIdx.x;
#pragma unroll
        for (int b = 0; b < IL; ++b) {
            if (y0 + r < ny && x0 + c < nx)
                rows[(blockIdx.z * slice + static_cast<size_t>(y0 + r) * nx + x0 + c) * IL + b] =
                    tile[b][r][c] + tile[b][r][c + 1];
            if (x0 + r < nx && y0 + c < ny)
                cols[(blockIdx.z * slice + static_cast<size_t>(x0 + r) * ny + y0 + c) * IL + b] =
                    tile[b][c][r] + tile[b][c + 1][r];
        }
    }
}

template <int IL>
struct DdGroup {
    float v[IL];
};

template <int IL>
__device__ __forceinline__ DdGroup<IL> dd_load(const float* p)
{
    DdGroup<IL> g;
    if constexpr (IL == 4) {
        const float4 f = *reinterpret_cast<const float4*>(p);
        g.v[0] = f.x;
        g.v[1] = f.y;
        g.v[2] = f.z;
        g.v[3] = f.w;
    } else {
        g.v[0] = *p;
    }
    return g;
}

// 1 / b for a float b > 0, within 2^-51.
__device__ __forceinline__ double dd_reciprocal(float b)
{
    const double d = static_cast<double>(b);
    double r = __builtin_amdgcn_rcp(d);
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}

template <int NB>
__global__ __launch_bounds__(64 * kDdViews) void fp_dd_cells_kernel(
    const float* __restrict__ rows, const float* __restrict__ cols, float* __restrict__ proj,
    const double* __restrict__ sc, const double* __restrict__ bo, const int* __restrict__ usex,
    DdProblem P)
{
    constexpr int IL = NB < 4 ? 1 : 4, G = NB / IL;
    const int is = blockIdx.x * 64 + threadIdx.x;
    const int ia = __builtin_amdgcn_readfirstlane(blockIdx.y * kDdViews + threadIdx.y);
    const int b0 = blockIdx.z * NB;
    if (is >= P.ns || ia >= P.na) return;
    const int nb = min(NB, P.nbatch - b0);
    const bool bx = usex[ia] != 0;
    const double dw = bx ? fabs(P.dy / sc[2 * ia + 1]) : fabs(P.dx / sc[2 * ia]);
    const int nu = bx ? P.ny : P.nx, nv = bx ? P.nx : P.ny;
    const size_t plane = static_cast<size_t>(P.nx) * P.ny * IL;
    const float* data = (bx ? rows : cols) + static_cast<size_t>(b0) * P.nx * P.ny;
    const int planes = (nb + IL - 1) / IL;
    const double* b = bo + 3 * (static_cast<size_t>(ia) * P.ns + is);
    double left = b[0] - b[2], right = b[0] + b[2];
    const double off = b[1];
    if (left > right) {
        const double t = left;
        left = right;
        right = t;
    }
    const double last = nv - 1;
    float sum[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) sum[k] = 0.0f;
    for (int u = 0; u < nu; ++u) {
        const double fl = floor(left);
        // a footprint starting left of the first cell adds nothing, cells past
        // nv - 2 are skipped (the reference's rules, see the kernel above)
        if (fl >= 0 && fl < last) {
            const double vend = fmin(ceil(right), last);
            const float* q = data + static_cast<size_t>(u) * nv * IL + static_cast<int>(fl) * IL;
            const bool more = fl + 1.0 < vend;        // a cell after the first
            const double vl = vend - 1.0;             // the last cell
            DdGroup<IL> c0[G], c1[G];
            const int lastc = more ? static_cast<int>(vl - fl) * IL : 0;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                // a plane past the batch re-reads the first
                const size_t o = g < planes ? g * plane : 0;
                c0[g] = dd_load<IL>(q + o);
                c1[g] = dd_load<IL>(q + o + lastc);
            }
            const double len0 = fmin(fl + 1.0, right) - left, h0 = 0.5 * len0;
            float lsum = static_cast<float>(len0);
            float tsum[NB];
#pragma unroll
            for (int k = 0; k < NB; ++k)
                tsum[k] = static_cast<float>(h0 * static_cast<double>(c0[k / IL].v[k % IL]));
            // cells covered whole between the first and the last
            for (int j = IL; j < lastc; j += IL) {
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const DdGroup<IL> c = dd_load<IL>(q + (g < planes ? g * plane : 0) + j);
#pragma unroll
                    for (int k = 0; k < IL; ++k)
                        tsum[g * IL + k] = __builtin_fmaf(0.5f, c.v[k], tsum[g * IL + k]);
                }
                lsum = static_cast<float>(static_cast<double>(lsum) + 1.0);
            }
            if (more) {
                const double len = fmin(vend, right) - vl, h = 0.5 * len;
#pragma unroll
                for (int k = 0; k < NB; ++k)
                    tsum[k] = static_cast<float>(static_cast<double>(tsum[k]) +
                                                 h * static_cast<double>(c1[k / IL].v[k % IL]));
                lsum = static_cast<float>(static_cast<double>(lsum) + len);
            }
            if (lsum > 0) {
                const double r = dd_reciprocal(lsum);
#pragma unroll
                for (int k = 0; k < NB; ++k)
                    sum[k] = sum[k] + static_cast<float>(static_cast<double>(tsum[k]) * r);
            }
        }
        left += off;
        right += off;
    }
#pragma unroll
    for (int k = 0; k < NB; ++k)
        if (k < nb)
            proj[(static_cast<size_t>(b0 + k) * P.na + ia) * P.ns + is] =
                static_cast<float>(static_cast<double>(sum[k]) * dw);
}

// One pixel's span of one view on the detector and its first and last channels.
template <int G, int IL>
struct DdSpan {
    double left, right, c0, cend, w;
    const float* q;
    int lastc;  // floats from the first channel to the last
    bool on;
    DdGroup<IL> v0[G], v1[G];
};

// One thread per pixel, a wave per 64 pixels of an image row; proj interleaved
// [plane][na][ns][IL].  The loads of view a + 1 are issued before view a is summed
// (a 512^2 image is four waves a SIMD, too few to hide them: 1.11 ms without).
template <int NB>
__global__ __launch_bounds__(256) void fp_dd_grad_planes_kernel(
    const float* __restrict__ proj, float* __restrict__ img, const double* __restrict__ weights,
    const double* __restrict__ pos, const int* __restrict__ usex, int stride, DdProblem P)
{
    constexpr int IL = NB < 4 ? 1 : 4, G = NB / IL;
    const int ix = blockIdx.x * 64 + (threadIdx.x & 63);
    const int iy = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + (threadIdx.x >> 6));
    if (ix >= P.nx || iy >= P.ny) return;
    const int b0 = blockIdx.z * NB, nb = min(NB, P.nbatch - b0);
    const size_t plane = static_cast<size_t>(P.na) * P.ns * IL;
    const float* pr = proj + static_cast<size_t>(b0) * P.na * P.ns;
    const int planes = (nb + IL - 1) / IL;
    const double2* table = reinterpret_cast<const double2*>(pos);
    const double fx = ix, fy = iy, last = P.ns - 1;
    double sum[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) sum[k] = 0.0;

    double2 pp = table[usex[0] != 0 ? iy : ix];  // of the next view to fetch
    const auto fetch = [&](int a, DdSpan<G, IL>& S) {
        const int ia = min(a, P.na - 1), an = min(a + 1, P.na - 1);
        const bool bx = usex[ia] != 0;
        const double begin = pp.x, off = pp.y;
        pp = table[static_cast<size_t>(an) * stride + (usex[an] != 0 ? iy : ix)];
        const double mid = begin + off * (bx ? fx : fy);
        double left = (bx ? ix : iy) == 0 ? mid : mid - off;
        double right = bx ? (ix == P.nx - 1 ? mid : mid + off) : (iy == P.ny - 1 ? mid : mid + off);
        if (left > right) {
            const double t = left;
            left = right;
            right = t;
        }
        S.left = left;
        S.right = right;
        S.w = weights[ia];
        S.c0 = ceil(left - 0.5);
        S.cend = fmin(floor(right + 0.5), last);
        S.on = S.c0 >= 0 && S.c0 <= S.cend && a < P.na;
        // (a span off the detector loads the row's first channel)
        const int c = S.on ? static_cast<int>(S.c0) : 0;
        S.lastc = S.on ? (static_cast<int>(S.cend) - c) * IL : 0;
        S.q = pr + (static_cast<size_t>(ia) * P.ns + c) * IL;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            // a plane past the batch re-reads the first
            const size_t o = g < planes ? g * plane : 0;
            S.v0[g] = dd_load<IL>(S.q + o);
            S.v1[g] = dd_load<IL>(S.q + o + S.lastc);
        }
    };
    const auto add = [&](const DdSpan<G, IL>& S) {
        if (!S.on) return;
        double tmp[NB];
        const double h0 = 0.5 * (fmin(S.c0 + 0.5, S.right) - fmax(S.c0 - 0.5, S.left));
#pragma unroll
        for (int k = 0; k < NB; ++k) tmp[k] = h0 * static_cast<double>(S.v0[k / IL].v[k % IL]);
        // channels covered whole -- but where left - 1/2 or right + 1/2 rounded
        // onto a channel's edge, its neighbour is a rounding short of that
        const bool whole = !(S.c0 + 0.5 < S.left) && !(S.cend - 0.5 > S.right);
        for (int j = IL; j < S.lastc; j += IL) {
            if (!whole) {
                const double c = S.c0 + j / IL;
                const double h = 0.5 * (fmin(c + 0.5, S.right) - fmax(c - 0.5, S.left));
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const DdGroup<IL> v = dd_load<IL>(S.q + (g < planes ? g * plane : 0) + j);
#pragma unroll
                    for (int k = 0; k < IL; ++k)
                        tmp[g * IL + k] = tmp[g * IL + k] + h * static_cast<double>(v.v[k]);
                }
                continue;
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const DdGroup<IL> v = dd_load<IL>(S.q + (g < planes ? g * plane : 0) + j);
#pragma unroll
                for (int k = 0; k < IL; ++k)
                    tmp[g * IL + k] =
                        __builtin_fma(0.5, static_cast<double>(v.v[k]), tmp[g * IL + k]);
            }
        }
        if (S.lastc > 0) {
            const double h = 0.5 * (fmin(S.cend + 0.5, S.right) - fmax(S.cend - 0.5, S.left));
#pragma unroll
            for (int k = 0; k < NB; ++k)
                tmp[k] = tmp[k] + h * static_cast<double>(S.v1[k / IL].v[k % IL]);
        }
#pragma unroll
        for (int k = 0; k < NB; ++k) sum[k] = sum[k] + tmp[k] * S.w;
    };
    DdSpan<G, IL> even, odd;
    fetch(0, even);
    for (int ia = 0; ia < P.na; ia += 2) {
        fetch(ia + 1, odd);
        add(even);
        fetch(ia + 2, even);
        add(odd);
    }
#pragma unroll
    for (int k = 0; k < NB; ++k)
        if (k < nb)
            img[(static_cast<size_t>(b0 + k) * P.ny + iy) * P.nx + ix] = static_cast<float>(sum[k]);
}

// Whether 1 to 4 slices that 8s leave over go along as one more, padded group of 8:
// a launch of their own takes as long as the whole one where that does not fill the
// chip (blocks: workgroups of a group; FP of 9 slices of 256^2, 60 views: 396 us in
// two launches, 273 in one; 9 of 512^2, 360 views, 1068 and 1150).
bool dd_padded(int nbatch, long long blocks)
{
    return nbatch > 8 && nbatch % 8 >= 1 && nbatch % 8 <= 4 && blocks * div_up(nbatch, 8) < 800;
}

// Slices in groups of 8, 4 and 1 (2 and 3 left over are one group of 4).
template <typename F>
int dd_groups(int nbatch, bool padded, F&& launch)
{
    for (int b0 = 0; b0 < nbatch;) {
        const int left = nbatch - b0;
        const int nb = left >= 5 ? 8 : left >= 2 ? 4 : 1;
        const int take = padded ? left : nb == 8 && left >= 8 ? left / 8 * 8 : std::min(left, nb);
        const int rc = launch(b0, take, nb);
        if (rc) return rc;
        b0 += take;
    }
    return CTR_OK;
}

int fp_dd_f32_part(const ctr_geom& g, const float* img, float* proj, int nbatch, const double* sc,
              const double* bo, const int* usex, hipStream_t st)
{
    DdProblem P{static_cast<int>(g.ns), static_cast<int>(g.na), static_cast<int>(g.nx),
                static_cast<int>(g.ny), nbatch, g.dx, g.dy};
    const size_t slice = static_cast<size_t>(g.nx) * g.ny;
    const bool padded = dd_padded(
        nbatch, static_cast<long long>(div_up(g.ns, 64)) * div_up(g.na, kDdViews));
    const bool single = nbatch % 8 == 1 && !padded;  // a last slice alone
    const int np = nbatch > 1 ? div_up(nbatch, 4) : 0;
    float* ws = nullptr;
    const int e = ws_part(reinterpret_cast<void**>(&ws),
                          (8 * np + (single ? 2 : 0)) * slice * sizeof(float), st);
    if (e) return e;
    float *rows = ws, *cols = ws + 4 * np * slice, *one = ws + 8 * np * slice;
    const dim3 tiles(div_up(g.nx, 32), div_up(g.ny, 32)), block(32, 8);
    if (np)
        hipLaunchKernelGGL(dd_cells_kernel<4>, dim3(tiles.x, tiles.y, np), block, 0, st, img, rows,
                           cols, P.ny, P.nx, nbatch);
    if (single)
        hipLaunchKernelGGL(dd_cells_kernel<1>, tiles, block, 0, st, img + (nbatch - 1) * slice, one,
                           one + slice, P.ny, P.nx, 1);
    int rc = check_launch("dd_cells_kernel");
    if (rc == CTR_OK)
        rc = dd_groups(nbatch, padded, [&](int b0, int take, int nb) {
            P.nbatch = take;
            float* out = proj + static_cast<size_t>(b0) * g.na * g.ns;
            const dim3 grid(div_up(g.ns, 64), div_up(g.na, kDdViews), div_up(take, nb));
            const dim3 wg(64, kDdViews);
            if (nb == 8)
                hipLaunchKernelGGL(fp_dd_cells_kernel<8>, grid, wg, 0, st, rows + b0 * slice,
                                   cols + b0 * slice, out, sc, bo, usex, P);
            else if (nb == 4)
                hipLaunchKernelGGL(fp_dd_cells_kernel<4>, grid, wg, 0, st, rows + b0 * slice,
                                   cols + b0 * slice, out, sc, bo, usex, P);
            else
                hipLaunchKernelGGL(fp_dd_cells_kernel<1>, grid, wg, 0, st, one, one + slice, out,
                                   sc, bo, usex, P);
            return check_launch("fp_dd_cells_kernel");
        });
    CTR_HIP(ctr::ws_free(ws, st));
    return rc;
}

int fp_dd_grad_f32_part(const ctr_geom& g, const float* proj, float* img, int nbatch, const double* w,
                   const double* pos, const int* usex, int stride, hipStream_t st)
{
    DdProblem P{static_cast<int>(g.ns), static_cast<int>(g.na), static_cast<int>(g.nx),
                static_cast<int>(g.ny), nbatch, g.dx, g.dy};
    const size_t sino = static_cast<size_t>(g.na) * g.ns;
    const int np = nbatch > 1 ? div_up(nbatch, 4) : 0;
    float* ws = nullptr;
    if (np) {
        const int e = ws_part(reinterpret_cast<void**>(&ws), 4 * np * sino * sizeof(float), st);
        if (e) return e;
        hipLaunchKernelGGL(interleave_kernel<4>, dim3(div_up(sino, 256), np), dim3(256), 0, st,
                           proj, ws, static_cast<unsigned int>(sino), nbatch);
    }
    int rc = check_launch("interleave_kernel");
    const bool padded =
        dd_padded(nbatch, static_cast<long long>(div_up(g.nx, 64)) * div_up(g.ny, 4));
    if (rc == CTR_OK)
        rc = dd_groups(nbatch, padded, [&](int b0, int take, int nb) {
            P.nbatch = take;
            float* out = img + static_cast<size_t>(b0) * g.nx * g.ny;
            const dim3 grid(div_up(g.nx, 64), div_up(g.ny, 4), div_up(take, nb));
            if (nb == 8)
                hipLaunchKernelGGL(fp_dd_grad_planes_kernel<8>, grid, dim3(256), 0, st,
                                   ws + b0 * sino, out, w, pos, usex, stride, P);
            else if (nb == 4)
                hipLaunchKernelGGL(fp_dd_grad_planes_kernel<4>, grid, dim3(256), 0, st,
                                   ws + b0 * sino, out, w, pos, usex, stride, P);
            else
                hipLaunchKernelGGL(fp_dd_grad_planes_kernel<1>, grid, dim3(256), 0, st,
                                   proj + b0 * sino, out, w, pos, usex, stride, P);
            return check_launch("fp_dd_grad_planes_kernel");
        });
    if (ws) CTR_HIP(ctr::ws_free(ws, st));
    return rc;
}

int fp_dd_f32(const ctr_geom& g, const float* img, float* proj, int nbatch, const double* sc,
              const double* bo, const int* usex, hipStream_t st)
{
    const size_t slice = static_cast<size_t>(g.nx) * g.ny, sino = static_cast<size_t>(g.na) * g.ns;
    const auto part = [&](int b, int count) {
        return fp_dd_f32_part(g, img + b * slice, proj + b * sino, count, sc, bo, usex, st);
    };
    return in_parts(nbatch, 2 * slice * sizeof(float), part, [&](int b, int count) {
        return one_by_one(b, count, [&](int i) { return part(i, 1); });
    });
}

int fp_dd_grad_f32(const ctr_geom& g, const float* proj, float* img, int nbatch, const double* w,
                   const double* pos, const int* usex, int stride, hipStream_t st)
{
    const size_t slice = static_cast<size_t>(g.nx) * g.ny, sino = static_cast<size_t>(g.na) * g.ns;
    const auto part = [&](int b, int count) {
        return fp_dd_grad_f32_part(g, proj + b * sino, img + b * slice, count, w, pos, usex, stride,
                                   st);
    };
    return in_parts(nbatch, sino * sizeof(float), part, [&](int b, int count) {
        return one_by_one(b, count, [&](int i) { return part(i, 1); });
    });
}

template <typename T, int NB>
int launch_fp_dd(const DdProblem& P, const T* img, const T* imgT, T* proj, const double* sc,
                 const double* bo, const int* usex, hipStream_t st)
{
    dim3 grid(div_up(P.ns, 64), div_up(P.na, kDdViews), div_up(P.nbatch, NB));
    hipLaunchKernelGGL((fp_dd_kernel<T, NB>), grid, dim3(64, kDdViews), 0, st, img, imgT, proj,
                       sc, bo, usex, P);
    return check_launch("fp_dd_kernel");
}

template <typename T>
int fp_dd_typed(const ctr_geom& g, const T* img, T* proj, int nbatch, const double* sc,
                const double* bo, const int* usex, hipStream_t st)
{
    const DdProblem P{static_cast<int>(g.ns), static_cast<int>(g.na), static_cast<int>(g.nx),
                      static_cast<int>(g.ny), nbatch, g.dx, g.dy};
    T* imgT = nullptr;
    const size_t n = static_cast<size_t>(nbatch) * g.nx * g.ny;
    CTR_HIP(ctr::ws_alloc(reinterpret_cast<void**>(&imgT), n * sizeof(T), st));
    hipLaunchKernelGGL(dd_transpose_kernel<T>, dim3(div_up(g.nx, 32), div_up(g.ny, 32), nbatch),
                       dim3(32, 8), 0, st, img, imgT, static_cast<int>(g.ny),
                       static_cast<int>(g.nx));
    int rc = check_launch("dd_transpose_kernel");
    if (rc == CTR_OK)
        rc = nbatch >= 4 ? launch_fp_dd<T, 4>(P, img, imgT, proj, sc, bo, usex, st)
             : nbatch >= 2 ? launch_fp_dd<T, 2>(P, img, imgT, proj, sc, bo, usex, st)
                           : launch_fp_dd<T, 1>(P, img, imgT, proj, sc, bo, usex, st);
    CTR_HIP(ctr::ws_free(imgT, st));
    return rc;
}

template <typename T, int NB>
int launch_fp_dd_grad(const DdProblem& P, const T* proj, T* img, const double* w,
                      const double* pos, const int* usex, int stride, hipStream_t st)
{
    dim3 grid(div_up(static_cast<long long>(P.nx) * P.ny, 256), div_up(P.nbatch, NB));
    hipLaunchKernelGGL((fp_dd_grad_kernel<T, NB>), grid, dim3(256), 0, st, proj, img, w, pos,
                       usex, stride, P);
    return check_launch("fp_dd_grad_kernel");
}

template <typename T>
int fp_dd_grad_typed(const ctr_geom& g, const T* proj, T* img, int nbatch, const double* w,
                     const double* pos, const int* usex, unsigned int stride, hipStream_t st)
{
    const DdProblem P{static_cast<int>(g.ns), static_cast<int>(g.na), static_cast<int>(g.nx),
                      static_cast<int>(g.ny), nbatch, g.dx, g.dy};
    const int s = static_cast<int>(stride);
    return nbatch >= 4 ? launch_fp_dd_grad<T, 4>(P, proj, img, w, pos, usex, s, st)
           : nbatch >= 2 ? launch_fp_dd_grad<T, 2>(P, proj, img, w, pos, usex, s, st)
                         : launch_fp_dd_grad<T, 1>(P, proj, img, w, pos, usex, s, st);
}

}  // namespace

int fp_dd(const ctr_geom& g, int dtype, const void* img, void* proj, int nbatch,
          const double* sc, const double* bo, const int* usex, hipStream_t st)
{
    CTR_REQUIRE(g.ns >= 1 && g.na >= 1 && g.nx >= 1 && g.ny >= 1, CTR_ERR_ARG,
                "distance-driven FP: sizes must be positive");
    if (dtype == CTR_F32)
        return fp_dd_f32(g, static_cast<const float*>(img), static_cast<float*>(proj), nbatch, sc,
                         bo, usex, st);
    return fp_dd_typed(g, static_cast<const double*>(img), static_cast<double*>(proj), nbatch, sc,
                       bo, usex, st);
}

int fp_dd_grad(const ctr_geom& g, int dtype, const void* proj, void* img, int nbatch,
               const double* w, const double* pos, const int* usex, unsigned int pos_stride,
               hipStream_t st)
{
    CTR_REQUIRE(g.ns >= 1 && g.na >= 1 && g.nx >= 1 && g.ny >= 1, CTR_ERR_ARG,
                "distance-driven FP gradient: sizes must be positive");
    if (dtype == CTR_F32) {
        // The kernel without interleaved planes (the same bits): where a few views are not
        // worth the copy (2 slices of 128^2: 12 views 12 -> 17 us with it, 60 views 51 ->
        // 47; 512^2, 4 slices, 12 views 24 and 24), and sinograms past its 32-bit positions.
        const long long sino = static_cast<long long>(g.na) * g.ns;
        const long long pixels = static_cast<long long>(g.nx) * g.ny;
        if (nbatch > 1 && ((g.na <= 40 && pixels <= (1 << 17)) || sino >= (1LL << 31)))
            return fp_dd_grad_typed(g, static_cast<const float*>(proj), static_cast<float*>(img),
                                    nbatch, w, pos, usex, pos_stride, st);
        return fp_dd_grad_f32(g, static_cast<const float*>(proj), static_cast<float*>(img), nbatch,
                              w, pos, usex, static_cast<int>(pos_stride), st);
    }
    return fp_dd_grad_typed(g, static_cast<const double*>(proj), static_cast<double*>(img),
                            nbatch, w, pos, usex, pos_stride, st);
}

}  // namespace ctr
