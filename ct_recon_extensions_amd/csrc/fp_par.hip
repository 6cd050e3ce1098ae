// Ray-driven parallel-beam forward projection for gfx950 and its
// gather-form transpose.
//
// FP (fp_stream.hpp; float32): waves stream image rows through their own LDS,
// one ray a lane for several views and slices.  fp_kernel (float64, and spans
// beyond that kernel's): one thread per ray (view, channel) for NB slices; a
// workgroup covers 256 consecutive channels of one view, so the sinogram row
// is written coalesced.  The ray marches the rows of the image (x-branch) or
// its columns (y-branch); the branch, the start position and the step of
// every ray come from the reference's FP64 tables (src/fp_par_2d.cc:149-208)
// and the position advances by repeated FP64 addition exactly as the
// reference does (src/fp_par_2d.cc:236-273), so sample inclusion
// (0 <= x <= nx-1) and tap choice match it; the lerp and the sum are FP32
// (the reference also sums in T).  For y-branch views the kernel reads a
// transposed copy of the slice so both branches walk contiguous rows.
//
// Transpose (fpt_kernel): one thread per pixel for NB slices; per view the
// channels whose rays pass within one pixel step are gathered with the
// triangle weight 1 - |mid - is|/o1 of the reference's transpose
// (src/fp_par_2d.cc:355-385), the channel range clamped to the detector.
//
// Transpose on the BP engine (FptGeo): the pixel's centre projects to the
// channel mid = begin + i*o1 + j*o2 (linear in the pixel), and the channels
// within |o1| of it get 1 - |c - mid|/|o1|; with |o1| <= 1 (pixel pitch along
// the marched axis at most the channel pitch) those are at most floor(mid)
// and floor(mid)+1, i.e. two taps, so the engine's LDS-staged spans, slice
// batching and FP64 anchors apply unchanged.  The first and last pixel
// along the marched axis keep one side only (src/fp_par_2d.cc:360-368).
#include "bp_engine.hpp"
#include "ctr_common.hpp"
#include "fp_stream.hpp"
#include "fpt_geom.hpp"
#include "tile_common.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <type_traits>
#include <unordered_map>

namespace ctr {

// Transposed copy src[b][iy][ix] -> dst[b][ix][iy] through a 32x33 LDS tile.
template <typename T>
__global__ void transpose_kernel(const T* __restrict__ src, T* __restrict__ dst, int ny, int nx)
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

// img   : [b][ny][nx] (x-branch rows) ; imgT : [b][nx][ny] (y-branch rows)
template <typename T, int NB>
__global__ __launch_bounds__(256) void fp_kernel(const T* __restrict__ img,
                                                 const T* __restrict__ imgT,
                                                 T* __restrict__ proj,
                                                 const double* __restrict__ sincos,
                                                 const double* __restrict__ bo,
                                                 const int* __restrict__ usex, FpProblem P)
{
    using Acc = typename std::conditional<sizeof(T) == 8, double, float>::type;
    const int s = blockIdx.x * 256 + threadIdx.x;
    const int a = blockIdx.y;
    const int b0 = blockIdx.z * NB;
    const int nb = min(NB, P.nbatch - b0);
    if (s >= P.ns) return;
    const bool xb = usex[a] != 0;
    // x-branch walks ny rows of length nx; y-branch walks nx rows of length ny
    const int nsteps = xb ? P.ny : P.nx;
    const int rowlen = xb ? P.nx : P.ny;
    const T* src = xb ? img : imgT;
    const double dw = xb ? fabs(P.dy / sincos[2 * a + 1]) : fabs(P.dx / sincos[2 * a]);
    double x = bo[2 * (static_cast<size_t>(a) * P.ns + s)];
    const double off = bo[2 * (static_cast<size_t>(a) * P.ns + s) + 1];
    const double hi = rowlen - 1;
    const size_t slice = static_cast<size_t>(P.nx) * P.ny;
    Acc sum[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) sum[b] = Acc(0);
    for (int k = 0; k < nsteps; ++k) {
        if (x >= 0 && x <= hi) {
            const double fl = floor(x);
            const int i1 = static_cast<int>(fl);
            const int i2 = min(i1 + 1, rowlen - 1);
            const Acc u = static_cast<Acc>(x - fl);
            const T* row = src + static_cast<size_t>(k) * rowlen;
            // every slice's taps loaded first (a slice past the batch
            // re-reads the last one and is not added)
            T t0[NB], t1[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                t0[b] = row[(b0 + min(b, nb - 1)) * slice + i1];
                t1[b] = row[(b0 + min(b, nb - 1)) * slice + i2];
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (b < nb) {
                    const Acc p0 = t0[b];
                    const Acc p1 = t1[b];
                    sum[b] += p0 + u * (p1 - p0);
                }
            }
        }
        x += off;
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
        if (b < nb)
            proj[(static_cast<size_t>(b0 + b) * P.na + a) * P.ns + s] =
                static_cast<T>(static_cast<double>(sum[b]) * dw);
}

// Pixels of the image border (first / last row and column), i < 2nx + 2(ny-2).
__device__ __forceinline__ void border_pixel(int i, int nx, int ny, int& ix, int& iy)
{
    if (i < nx) {
        ix = i;
        iy = 0;
    } else if (i < 2 * nx) {
        ix = i - nx;
        iy = ny - 1;
    } else {
        const int j = i - 2 * nx;
        ix = j < ny - 2 ? 0 : nx - 1;
        iy = 1 + (j < ny - 2 ? j : j - (ny - 2));
    }
}

// Contribution of view a to pixel (ix, iy) for slices b0 .. b0+nb-1,
// added to sum[]: the reference's gather (src/fp_par_2d.cc:355-385).
template <typename T, int NB>
__device__ __forceinline__ void fpt_view(const T* __restrict__ proj,
                                         const double* __restrict__ weights,
                                         const double* __restrict__ pos,
                                         const int* __restrict__ usex, const FpProblem& P,
                                         int stride, int a, int ix, int iy, int b0, int nb,
                                         double (&sum)[NB])
{
    using Acc = typename std::conditional<sizeof(T) == 8, double, float>::type;
    const size_t pslice = static_cast<size_t>(P.na) * P.ns;
    double mid, left, right, o1;
    // mid exactly as the reference rounds it (a product, then a sum): the
    // one-sided border rule below is decided on it
    if (usex[a]) {
        const double* pp = pos + 2 * (static_cast<size_t>(a) * stride + iy);
        o1 = pp[1];
        mid = __dadd_rn(pp[0], __dmul_rn(o1, static_cast<double>(ix)));
        left = ix == 0 ? mid : mid - o1;
        right = ix == P.nx - 1 ? mid : mid + o1;
    } else {
        const double* pp = pos + 2 * (static_cast<size_t>(a) * stride + ix);
        o1 = pp[1];
        mid = __dadd_rn(pp[0], __dmul_rn(o1, static_cast<double>(iy)));
        left = iy == 0 ? mid : mid - o1;
        right = iy == P.ny - 1 ? mid : mid + o1;
    }
    if (left > right) {
        const double t = left;
        left = right;
        right = t;
    }
    const int c0 = max(static_cast<int>(ceil(left)), 0);
    const int c1 = min(static_cast<int>(floor(right)), P.ns - 1);
    Acc tmp[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) tmp[b] = Acc(0);
    for (int c = c0; c <= c1; ++c) {
        const Acc w = static_cast<Acc>(1.0 - fabs((mid - c) / o1));
        const T* pr = proj + static_cast<size_t>(a) * P.ns + c;
        // every slice's value loaded first (a slice past the batch re-reads
        // the last one and is not added)
        T val[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) val[b] = pr[(b0 + min(b, nb - 1)) * pslice];
#pragma unroll
        for (int b = 0; b < NB; ++b)
            if (b < nb) tmp[b] += w * static_cast<Acc>(val[b]);
    }
    const double wa = weights[a];
#pragma unroll
    for (int b = 0; b < NB; ++b) sum[b] += static_cast<double>(tmp[b]) * wa;
}

// Every pixel, one thread per pixel for NB slices.
template <typename T, int NB>
__global__ __launch_bounds__(256) void fpt_kernel(const T* __restrict__ proj,
                                                  T* __restrict__ img,
                                                  const double* __restrict__ weights,
                                                  const double* __restrict__ pos,
                                                  const int* __restrict__ usex, FpProblem P,
                                                  int stride)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int b0 = blockIdx.y * NB;
    const int nb = min(NB, P.nbatch - b0);
    if (i >= P.nx * P.ny) return;
    const int ix = i % P.nx, iy = i / P.nx;
    double sum[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) sum[b] = 0.0;
    for (int a = 0; a < P.na; ++a) fpt_view<T, NB>(proj, weights, pos, usex, P, stride, a, ix, iy,
                                                   b0, nb, sum);
#pragma unroll
    for (int b = 0; b < NB; ++b)
        if (b < nb) img[(static_cast<size_t>(b0 + b) * P.ny + iy) * P.nx + ix] = static_cast<T>(sum[b]);
}

// The border pixels (nx, ny >= 3) after the engine pass, in two steps so
// that neighbouring threads read neighbouring channels: (1) thread = border
// pixel, a chunk of views per workgroup row, FP64 partial sums per (view
// chunk, slice, pixel); (2) the partials added in chunk order.  Chunks of
// kBorderViews views where the partials live in a caller's workspace (the
// allocation-free entry point's fixed scratch), of kBorderViewsAlloc views
// (four times the workgroups) where they are allocated per call.
constexpr int kBorderViews = 16;
constexpr int kBorderViewsAlloc = 4;

template <int NB>
__global__ __launch_bounds__(256) void fpt_border_partial_kernel(
    const float* __restrict__ proj, double* __restrict__ partial,
    const double* __restrict__ weights, const double* __restrict__ pos,
    const int* __restrict__ usex, FpProblem P, int stride, int nborder, int cviews)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int vc = blockIdx.y;
    const int b0 = blockIdx.z * NB;
    const int nb = min(NB, P.nbatch - b0);
    if (i >= nborder) return;
    int ix, iy;
    border_pixel(i, P.nx, P.ny, ix, iy);
    double sum[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) sum[b] = 0.0;
    const int a1 = min(P.na, (vc + 1) * cviews);
    for (int a = vc * cviews; a < a1; ++a)
        fpt_view<float, NB>(proj, weights, pos, usex, P, stride, a, ix, iy, b0, nb, sum);
#pragma unroll
    for (int b = 0; b < NB; ++b)
        if (b < nb) partial[(static_cast<size_t>(vc) * P.nbatch + b0 + b) * nborder + i] = sum[b];
}

__global__ void fpt_border_reduce_kernel(const double* __restrict__ partial,
                                         float* __restrict__ img, FpProblem P, int nborder,
                                         int nchunks)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int b = blockIdx.y;
    if (i >= nborder) return;
    int ix, iy;
    border_pixel(i, P.nx, P.ny, ix, iy);
    // eight chunks' partials loaded together (chunks past the last re-read
    // it and are not added), then added in chunk order
    const double* q = partial + static_cast<size_t>(b) * nborder + i;
    const size_t cstride = static_cast<size_t>(P.nbatch) * nborder;
    double t = 0.0;
    for (int c = 0; c < nchunks; c += 8) {
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = q[static_cast<size_t>(min(c + k, nchunks - 1)) * cstride];
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (c + k < nchunks) t += v[k];
    }
    img[(static_cast<size_t>(b) * P.ny + iy) * P.nx + ix] = static_cast<float>(t);
}

namespace {

template <typename T, int NB>
int launch_fp(const FpProblem& P, const T* img, const T* imgT, T* proj, const double* sc,
              const double* bo, const int* usex, hipStream_t st)
{
    dim3 grid(div_up(P.ns, 256), P.na, div_up(P.nbatch, NB));
    hipLaunchKernelGGL((fp_kernel<T, NB>), grid, dim3(256), 0, st, img, imgT, proj, sc, bo, usex, P);
    return check_launch("fp_kernel");
}

// Waves (row segments) per workgroup: 2 where that fills the chip, more for small
// scans (8 x 512^2, 720 views: 296 us at 2, 303 at 4, 345 at 8; 4 slices 184, 183,
// 192; one slice 135, 120, 121; 1 x 256^2, 360 views: 68, 54, 54; 8 x 192^2, 200
// views: 61, 55, 61).  groups: slice groups of the launch.
int fp_stream_waves(const ctr_geom& g, int shape, int groups)
{
    const int vgroups = div_up(g.na, shape < 2 ? 4 : 1);
    return static_cast<long long>(div_up(g.ns, 64)) * vgroups * groups >= 4096 ? 2 : 4;
}

// Segments are whole fours of rows for any NB: a slice alone has the sums that it
// has in a group of four with as many waves.
template <int NB, int V, int SPAN>
int launch_fp_stream_s(FpStreamLaunch L, int n, int waves, hipStream_t st)
{
    using S = FpShape<NB, SPAN>;
    static_assert(4 % S::kRows == 0, "segments of whole chunks");
    L.nb = n;
    L.cgroups = div_up(L.P.ns, 64);
    const int groups = div_up(n, NB), vgroups = div_up(L.P.na, V);
    L.chunks = div_up(div_up(std::max(L.P.nx, L.P.ny), 4), waves) * (4 / S::kRows);
    const size_t lds = static_cast<size_t>(waves) * S::kLds;
    hipLaunchKernelGGL((fp_stream_kernel<NB, V, SPAN>), dim3(L.cgroups * vgroups, groups, 2),
                       dim3(64 * waves), lds, st, L);
    return check_launch("fp_stream_kernel");
}

// shape: 0 4 views and 128 columns, 1 4 and 256, 2 1 and 128, 3 1 and 256.
template <int NB>
int launch_fp_stream(int shape, const FpStreamLaunch& L, int n, int waves, hipStream_t st)
{
    switch (shape) {
        case 0: return launch_fp_stream_s<NB, 4, 128>(L, n, waves, st);
        case 1: return launch_fp_stream_s<NB, 4, 256>(L, n, waves, st);
        case 2: return launch_fp_stream_s<NB, 1, 128>(L, n, waves, st);
        default: return launch_fp_stream_s<NB, 1, 256>(L, n, waves, st);
    }
}

// Four views share a staged row unless their rays drift too far apart (few
// views); 256 columns take coarse detectors.  -1: none.
int fp_stream_shape(const ctr_geom& g)
{
    constexpr int rows = FpShape<1, 128>::kRows;
    for (int shape = 0; shape < 4; ++shape)
        if (fp_stream_applies(g, shape < 2 ? 4 : 1, rows, shape & 1 ? 256 : 128)) return shape;
    return -1;
}

// waves: of the groups of four; waves1: of a last slice alone; padded: that slice is a
// group of four (the same bits).
int fp_stream_part(const ctr_geom& g, int shape, int waves, int waves1, bool padded, const float* img,
                   float* proj, int nbatch, const double* sc, const double* bo, const int* usex,
                   hipStream_t st)
{
    FpStreamLaunch L{};
    L.P = FpProblem{static_cast<int>(g.ns), static_cast<int>(g.na), static_cast<int>(g.nx),
                    static_cast<int>(g.ny), nbatch, g.dx, g.dy};
    L.proj = proj;
    L.sincos = sc;
    L.bo = bo;
    L.usex = usex;
    const size_t slice = static_cast<size_t>(g.nx) * g.ny;
    const int np = nbatch > 1 ? div_up(nbatch, 4) : 0;
    const bool single = nbatch % 4 == 1 && !(padded && nbatch > 1);  // the last slice alone
    float* ws = nullptr;
    const int e = ws_part(reinterpret_cast<void**>(&ws),
                          (8 * np + (single ? 1 : 0)) * slice * sizeof(float), st);
    if (e) return e;
    float *rows = ws, *cols = ws + 4 * np * slice, *one = ws + 8 * np * slice;
    const dim3 tiles(div_up(g.nx, 32), div_up(g.ny, 32), std::max(np, 1));
    if (np)
        hipLaunchKernelGGL(image_planes_kernel<4>, tiles, dim3(32, 8), 0, st, img, rows, cols,
                           L.P.ny, L.P.nx, nbatch);
    if (single)
        hipLaunchKernelGGL(image_planes_kernel<1>, dim3(tiles.x, tiles.y), dim3(32, 8), 0, st,
                           img + (nbatch - 1) * slice, nullptr, one, L.P.ny, L.P.nx, 1);
    int rc = check_launch("image_planes_kernel");
    for (int b0 = 0; b0 < nbatch && rc == CTR_OK;) {
        const int left = nbatch - b0;
        int take = left;
        L.b0 = b0;
        L.rows = rows;
        L.cols = cols;
        if (left >= 2) {
            take = single ? left - 1 : left;
            rc = launch_fp_stream<4>(shape, L, take, waves, st);
        } else {
            L.rows = img;                   // indexed by slice
            L.cols = one - b0 * slice;
            rc = launch_fp_stream<1>(shape, L, 1, waves1, st);
        }
        b0 += take;
    }
    CTR_HIP(ctr::ws_free(ws, st));
    return rc;
}

int fp_stream(const ctr_geom& g, int shape, const float* img, float* proj, int nbatch,
              const double* sc, const double* bo, const int* usex, hipStream_t st)
{
    const size_t slice = static_cast<size_t>(g.nx) * g.ny, sino = static_cast<size_t>(g.na) * g.ns;
    // of the whole call, whatever its parts are.  A last slice alone is two more
    // launches, which a small scan does not hide: there it is a padded group (5 slices
    // of 32^2: 26 us alone, 17 padded)
    const long long blocks = static_cast<long long>(div_up(g.ns, 64)) *
                             div_up(g.na, shape < 2 ? 4 : 1) * div_up(nbatch, 4);
    const bool padded = blocks < 512;
    const int four = nbatch % 4 == 1 && !padded ? nbatch - 1 : nbatch;  // in groups of four
    const int waves = fp_stream_waves(g, shape, div_up(four, 4));
    const int waves1 = fp_stream_waves(g, shape, 1);
    const auto part = [&](int b, int count, int w1) {
        return fp_stream_part(g, shape, waves, w1, padded, img + b * slice, proj + b * sino, count,
                              sc, bo, usex, st);
    };
    return in_parts(
        nbatch, 2 * slice * sizeof(float), [&](int b, int count) { return part(b, count, waves1); },
        [&](int b, int count) {
            return one_by_one(b, count, [&](int i) {
                return part(i, 1, nbatch > 1 && i < four ? waves : waves1);
            });
        });
}

template <typename T>
int fp_typed(const ctr_geom& g, const T* img, T* proj, int nbatch, const double* sc,
             const double* bo, const int* usex, hipStream_t st)
{
    FpProblem P{static_cast<int>(g.ns), static_cast<int>(g.na), static_cast<int>(g.nx),
                static_cast<int>(g.ny), nbatch, g.dx, g.dy};
    if constexpr (std::is_same<T, float>::value) {
        const int shape = fp_stream_shape(g);
        if (shape >= 0) return fp_stream(g, shape, img, proj, nbatch, sc, bo, usex, st);
    }
    T* imgT = nullptr;
    const size_t n = static_cast<size_t>(nbatch) * g.nx * g.ny;
    CTR_HIP(ctr::ws_alloc(reinterpret_cast<void**>(&imgT), n * sizeof(T), st));
    hipLaunchKernelGGL(transpose_kernel<T>, dim3(div_up(g.nx, 32), div_up(g.ny, 32), nbatch),
                       dim3(32, 8), 0, st, img, imgT, static_cast<int>(g.ny),
                       static_cast<int>(g.nx));
    int rc = check_launch("transpose_kernel");
    if (rc == CTR_OK) {
        const int nb = nbatch >= 8 ? 8 : nbatch >= 4 ? 4 : nbatch >= 2 ? 2 : 1;
        switch (nb) {
            case 1: rc = launch_fp<T, 1>(P, img, imgT, proj, sc, bo, usex, st); break;
            case 2: rc = launch_fp<T, 2>(P, img, imgT, proj, sc, bo, usex, st); break;
            case 4: rc = launch_fp<T, 4>(P, img, imgT, proj, sc, bo, usex, st); break;
            default: rc = launch_fp<T, 8>(P, img, imgT, proj, sc, bo, usex, st); break;
        }
    }
    CTR_HIP(ctr::ws_free(imgT, st));
    return rc;
}

template <typename T, int NB>
int launch_fpt(const FpProblem& P, const T* proj, T* img, const double* w, const double* pos,
               const int* usex, int stride, hipStream_t st)
{
    dim3 grid(div_up(static_cast<long long>(P.nx) * P.ny, 256), div_up(P.nbatch, NB));
    hipLaunchKernelGGL((fpt_kernel<T, NB>), grid, dim3(256), 0, st, proj, img, w, pos, usex, P,
                       stride);
    return check_launch("fpt_kernel");
}

// Bytes of FP64 partials the border pass needs (nchunks x nbatch x nborder)
// with chunks of cviews views.
size_t fpt_border_bytes(int nx, int ny, int na, int nbatch, int cviews = kBorderViews)
{
    const size_t nborder = 2 * static_cast<size_t>(nx) + 2 * (static_cast<size_t>(ny) - 2);
    return static_cast<size_t>(div_up(na, cviews)) * nbatch * nborder * sizeof(double);
}

// ws: caller workspace of at least fpt_border_bytes(...) bytes, or null for a
// stream-ordered allocation.  Every partial is written before it is read.
template <int NB>
int launch_fpt_border(const FpProblem& P, const float* proj, float* img, const double* w,
                      const double* pos, const int* usex, int stride, void* ws, hipStream_t st)
{
    const int nborder = 2 * P.nx + 2 * (P.ny - 2);
    const int cviews = ws ? kBorderViews : kBorderViewsAlloc;
    const int nchunks = div_up(P.na, cviews);
    double* partial = static_cast<double*>(ws);
    if (!ws)
        CTR_HIP(ctr::ws_alloc(reinterpret_cast<void**>(&partial),
                               fpt_border_bytes(P.nx, P.ny, P.na, P.nbatch, cviews), st));
    hipLaunchKernelGGL((fpt_border_partial_kernel<NB>),
                       dim3(div_up(nborder, 256), nchunks, div_up(P.nbatch, NB)), dim3(256), 0, st,
                       proj, partial, w, pos, usex, P, stride, nborder, cviews);
    int rc = check_launch("fpt_border_partial_kernel");
    if (rc == CTR_OK) {
        hipLaunchKernelGGL(fpt_border_reduce_kernel, dim3(div_up(nborder, 256), P.nbatch),
                           dim3(256), 0, st, partial, img, P, nborder, nchunks);
        rc = check_launch("fpt_border_reduce_kernel");
    }
    if (!ws) CTR_HIP(ctr::ws_free(partial, st));
    return rc;
}

template <int NB, int LROW>
int launch_fpt_engine(const ctr_geom& g, const float* proj, float* img, int nbatch,
                      const double* w, const double* pos, const int* usex, int stride,
                      hipStream_t st)
{
    constexpr int TW = 16, TH = 16;
    BpLaunch<FptGeo> L{};
    L.P = FptProblem{static_cast<int>(g.ns), static_cast<int>(g.na), static_cast<int>(g.nx),
                     static_cast<int>(g.ny)};
    L.nbatch = nbatch;
    L.tiles_x = div_up(g.nx, TW);
    L.tiles_y = div_up(g.ny, TH);
    L.lmax = LROW;
    L.vchunk = engine_vchunk<FptAnchor>(NB, LROW);
    L.scale = 1.0;
    L.proj = proj;
    L.img = img;
    const FptTables T{w, pos, usex, stride};
    const size_t lds = kAnchorChunk * sizeof(FptAnchor) +
                       2 * static_cast<size_t>(L.vchunk) * NB * LROW * sizeof(float);
    auto kern = bp_forward_kernel<FptGeo, TW, TH, NB, LROW>;
    if (lds > 64 * 1024)
        CTR_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>(lds)));
    hipLaunchKernelGGL(kern, dim3(super_grid(L.tiles_x, L.tiles_y), div_up(nbatch, NB)),
                       dim3(TileShape<TW, TH>::kBlock), lds, st, T, L);
    return check_launch("bp_forward_kernel<fp transpose>");
}

// The engine path needs |o1| <= 1 for every view (at most two channels per
// pixel-view) and a staged span that fits 64 channels per 16x16 tile:
// |o1| <= max(dx, dy)/ds and the span is at most 15 (|o1| + |o2|) + 3.
bool fpt_engine_applies(const ctr_geom& g)
{
    const double r = std::max(std::fabs(g.dx), std::fabs(g.dy)) / g.ds;
    return g.ds > 0 && r <= 1.0 && 15.0 * 2.0 * r + 4.0 <= 64.0;
}

template <typename T>
int fpt_typed(const ctr_geom& g, const T* proj, T* img, int nbatch, const double* w,
              const double* pos, const int* usex, unsigned int stride, void* ws, hipStream_t st)
{
    if constexpr (std::is_same<T, float>::value) {
        if (fpt_engine_applies(g) && g.nx >= 3 && g.ny >= 3) {
            // interior on the engine, then the border pixels exactly
            const int s = static_cast<int>(stride);
            int rc = CTR_OK;
            FpProblem P{static_cast<int>(g.ns), static_cast<int>(g.na), static_cast<int>(g.nx),
                        static_cast<int>(g.ny), nbatch, g.dx, g.dy};
            if (stream_applies(48, g.na, g.ns) && stream_pays(nbatch, P.nx, P.ny, P.na, 48, 8)) {
                StreamLaunch<FptGeo> S{};
                S.P = FptProblem{P.ns, P.na, P.nx, P.ny};
                S.scale = 1.0;
                S.img = img;
                const FptTables tab{w, pos, usex, s};
                // a caller's workspace means that nothing may be allocated
                rc = ws ? launch_stream_batch<FptGeo, true>(S, tab, proj, nbatch, 48, st)
                        : launch_stream_batch<FptGeo>(S, tab, proj, nbatch, 48, st);
                if (rc) return rc;
                return nbatch >= 8 ? launch_fpt_border<8>(P, proj, img, w, pos, usex, s, ws, st)
                                   : launch_fpt_border<1>(P, proj, img, w, pos, usex, s, ws, st);
            }
            const int nb = engine_nb(nbatch >= 8 ? 8 : nbatch >= 4 ? 4 : nbatch, g.na, g.ns);
            // the applicability bound keeps a tile-view's span within
            // 30 max(dx,dy)/ds + 5 <= 35 channels: 48-channel rows when the
            // slices are interleaved four to a word, 64 otherwise
            if (nb >= 8) rc = launch_fpt_engine<8, 48>(g, proj, img, nbatch, w, pos, usex, s, st);
            else if (nb >= 4) rc = launch_fpt_engine<4, 48>(g, proj, img, nbatch, w, pos, usex, s, st);
            else if (nb >= 2) rc = launch_fpt_engine<2, 64>(g, proj, img, nbatch, w, pos, usex, s, st);
            else rc = launch_fpt_engine<1, 64>(g, proj, img, nbatch, w, pos, usex, s, st);
            if (rc) return rc;
            return nbatch >= 8 ? launch_fpt_border<8>(P, proj, img, w, pos, usex, s, ws, st)
                               : launch_fpt_border<1>(P, proj, img, w, pos, usex, s, ws, st);
        }
    }
    FpProblem P{static_cast<int>(g.ns), static_cast<int>(g.na), static_cast<int>(g.nx),
                static_cast<int>(g.ny), nbatch, g.dx, g.dy};
    const int nb = nbatch >= 8 ? 8 : nbatch >= 4 ? 4 : nbatch >= 2 ? 2 : 1;
    const int s = static_cast<int>(stride);
    switch (nb) {
        case 1: return launch_fpt<T, 1>(P, proj, img, w, pos, usex, s, st);
        case 2: return launch_fpt<T, 2>(P, proj, img, w, pos, usex, s, st);
        case 4: return launch_fpt<T, 4>(P, proj, img, w, pos, usex, s, st);
        default: return launch_fpt<T, 8>(P, proj, img, w, pos, usex, s, st);
    }
}

}  // namespace

int fp_par(const ctr_geom& g, int dtype, const void* img, void* proj, int nbatch,
           const double* sc, const double* bo, const int* usex, hipStream_t st)
{
    CTR_REQUIRE(g.ns >= 1 && g.na >= 1 && g.nx >= 1 && g.ny >= 1, CTR_ERR_ARG,
                "ray-driven FP: sizes must be positive");
    if (dtype == CTR_F32)
        return fp_typed(g, static_cast<const float*>(img), static_cast<float*>(proj), nbatch, sc,
                        bo, usex, st);
    return fp_typed(g, static_cast<const double*>(img), static_cast<double*>(proj), nbatch, sc, bo,
                    usex, st);
}

int fp_par_t(const ctr_geom& g, int dtype, const void* proj, void* img, int nbatch,
             const double* w, const double* pos, const int* usex, unsigned int pos_stride,
             hipStream_t st)
{
    CTR_REQUIRE(g.ns >= 1 && g.na >= 1 && g.nx >= 1 && g.ny >= 1, CTR_ERR_ARG,
                "ray-driven FP transpose: sizes must be positive");
    if (dtype == CTR_F32)
        return fpt_typed(g, static_cast<const float*>(proj), static_cast<float*>(img), nbatch, w,
                         pos, usex, pos_stride, nullptr, st);
    return fpt_typed(g, static_cast<const double*>(proj), static_cast<double*>(img), nbatch, w,
                     pos, usex, pos_stride, nullptr, st);
}

// ---------------------------------------------- allocation-free FP transpose
// The only device memory the FP transpose uses beyond its inputs and output
// is the border pass's FP64 partials (float32 buffers, geometries on the BP
// engine).  ctr_fp_t_noalloc keeps them in this file-scope array instead of a
// stream-ordered allocation: kFptScratchBytes per device, held until the
// process ends.  Kernels take its device address, which hipGetSymbolAddress
// returns once per device (the name itself is a host-side stand-in).
constexpr size_t kFptScratchBytes = size_t{16} << 20;
static __device__ __align__(256) unsigned char scratch[kFptScratchBytes];

namespace {
std::mutex g_scratch_mu;
std::unordered_map<int, void*> g_scratch_ptr;  // device -> address of `scratch` there

int scratch_address(void** out)
{
    int dev = 0;
    CTR_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    auto it = g_scratch_ptr.find(dev);
    if (it == g_scratch_ptr.end()) {
        void* p = nullptr;
        CTR_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        it = g_scratch_ptr.emplace(dev, p).first;
    }
    *out = it->second;
    return CTR_OK;
}
}  // namespace

int fp_par_t_noalloc(const ctr_geom& g, int dtype, const void* proj, void* img, int nbatch,
                     const double* w, const double* pos, const int* usex,
                     unsigned int pos_stride, hipStream_t st)
{
    CTR_REQUIRE(g.ns >= 1 && g.na >= 1 && g.nx >= 1 && g.ny >= 1, CTR_ERR_ARG,
                "ray-driven FP transpose: sizes must be positive");
    if (dtype != CTR_F32)  // the float64 transpose uses no scratch
        return fpt_typed(g, static_cast<const double*>(proj), static_cast<double*>(img), nbatch,
                         w, pos, usex, pos_stride, nullptr, st);
    // only the engine path (with its border pass) uses the scratch
    const bool border = fpt_engine_applies(g) && g.nx >= 3 && g.ny >= 3;
    const size_t need = border ? fpt_border_bytes(static_cast<int>(g.nx), static_cast<int>(g.ny),
                                                  static_cast<int>(g.na), nbatch)
                               : 0;
    if (need > kFptScratchBytes) {
        set_error("ctr_fp_t_noalloc: the border partials need " + std::to_string(need) +
                  " bytes, more than the " + std::to_string(kFptScratchBytes) +
                  "-byte scratch (use ctr_fp_t, or fewer slices per call)");
        return CTR_ERR_SHAPE;
    }
    void* ws = nullptr;
    const int rc = scratch_address(&ws);
    if (rc) return rc;
    return fpt_typed(g, static_cast<const float*>(proj), static_cast<float*>(img), nbatch, w, pos,
                     usex, pos_stride, ws, st);
}

}  // namespace ctr
