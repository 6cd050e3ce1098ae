// Ray-driven parallel FP with wave-private row streams (float32).
//
// A wave owns 64 consecutive channels (one ray a lane) of V consecutive views
// for NB slices, over one segment of the marched rows; the waves of a workgroup
// take the segments of the same rays, and their partial sums are added in FP64
// at the end.  What bounds the FP is the issue of the per-sample work and the
// LDS reads of the taps, and the layout keeps everything else off those units:
//  * each wave stages the columns its rays can touch, R rows at a time, into
//    its own double-buffered LDS by DMA, 16 bytes a lane, with no barrier before
//    the end.  Slices are interleaved in fours (image_planes_kernel, which also
//    makes the transposed copy for the views that march columns), so a tap of
//    four slices is one 16-byte read;
//  * the rows a ray has samples on, [kin, kout), come from its FP64 position
//    once (fp_ray_rows: the reference accumulates x += step and tests 0 <= x <=
//    nx - 1; where a crossing falls within that sum's rounding of a row it is
//    replayed, elsewhere it cannot matter).  Inside them the position
//    is 32.32 fixed point: an add, an add with carry, and the fraction's
//    conversion per sample, good to 2^-33 of a pixel a step, restarted from FP64
//    in each segment.  Noise images against FP64, relative L2: 2.0e-7 at 256^2,
//    2.8e-7 at 512^2, 1.1e-6 at 8192^2 (positions accumulated in FP64 and one FP32
//    sum a ray, as before: 3.7e-7, 5.3e-7, 1.5e-6);
//  * rows on which all rays of the wave are inside run without any test; the
//    columns of every chunk are computed 64 chunks at a time, one a lane.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "bp_engine.hpp"
#include "ctr_common.hpp"
#include "fp_span.hpp"
#include "tile_common.hpp"

namespace ctr {

struct FpProblem {
    int ns, na, nx, ny, nbatch;
    double dx, dy;
};

// 4 rows of one slice or 2 of four: 8 x 512^2, 720 views 303 us (4 rows: 415, the
// registers of the unrolled rows cost two waves a SIMD).
template <int NB, int SPAN>
struct FpShape {
    static constexpr int kIl = NB < 4 ? 1 : 4;          // slices a column holds
    static constexpr int kPlanes = NB / kIl;            // 4-slice planes
    static constexpr int kSpan = SPAN;                  // columns staged
    static constexpr int kRows = NB == 1 ? 4 : 2;       // rows a chunk
    static constexpr int kRowF = kPlanes * kSpan * kIl; // floats of a staged row
    // floats of a buffer: the rows, then zeros for the taps of rays off the image
    // (both taps of every plane)
    static constexpr int kZero = kRows * kRowF;
    static constexpr int kBuf = kZero + ((kPlanes - 1) * kSpan * kIl + 2 * kIl + 7) / 8 * 8;
    static constexpr int kLds = 2 * kBuf * 4;  // bytes of a wave
    static_assert(NB == 1 || NB % 4 == 0, "one slice or planes of four");
};

struct FpStreamLaunch {
    FpProblem P;
    const float* rows;   // x-branch rows: [plane][ny][nx][kIl]
    const float* cols;   // y-branch rows: [plane][nx][ny][kIl]
    float* proj;
    const double* sincos;
    const double* bo;
    const int* usex;
    int b0, nb;          // slices of this launch
    int chunks;          // chunks of kRows rows a segment (one wave)
    int cgroups;         // channel groups
};

__device__ __forceinline__ int wave_min(int x)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x = min(x, __shfl_xor(x, o));
    return uniform_i(x);
}

// A chunk's column count, with kFpNarrow where a single slice's lanes move one column
// each: four of a lane would cross the row's end.
constexpr int kFpNarrow = 1 << 16;

template <int IL>
__device__ __forceinline__ int fp_columns(const FpSpan& c, int rowlen)
{
    const bool narrow = IL == 1 && c.first + ((c.cols + 3) & ~3) > rowlen && ((rowlen - c.first) & 3);
    return c.cols + (narrow ? kFpNarrow : 0);
}

// DMA of the chunk's rows k0 .. k0 + kRows - 1, columns cm .. cm + cols - 1, of
// every plane; columns past the row (the last column's right tap is one) and rows
// past the image read as zero.
template <int NB, int SPAN>
__device__ __forceinline__ void fp_stage(const float* src, size_t plane, int nsteps, int rowlen,
                                         int k0, int cm, int cols_flag, int planes, float* buf,
                                         int lane)
{
    using S = FpShape<NB, SPAN>;
    const unsigned int row_bytes = static_cast<unsigned int>(rowlen) * S::kIl * 4u;
    const unsigned int bytes = static_cast<unsigned int>(nsteps) * row_bytes;
    // columns a lane moves: 16 bytes of them, or one where a lane's four would
    // cross the row's end (single slices; flagged by fp_columns)
    const int lane_cols = S::kIl == 4 || cols_flag >= kFpNarrow ? 1 : 4;
    const int cols = cols_flag & (kFpNarrow - 1);
    for (int c = 0; c < cols; c += 64 * lane_cols) {
        const int lc = c + lane * lane_cols, col = cm + lc;
        if (lc >= S::kSpan) continue;
#pragma unroll
        for (int p = 0; p < S::kPlanes; ++p) {
            // a plane past the batch has no memory: range 0 reads as zero
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(src + p * plane), 0, p < planes ? bytes : 0u, 0x00020000);
#pragma unroll
            for (int r = 0; r < S::kRows; ++r) {
                const unsigned int voff =
                    col < rowlen ? static_cast<unsigned int>(k0 + r) * row_bytes +
                                       static_cast<unsigned int>(col) * S::kIl * 4u
                                 : 0x80000000u;
                auto* dst = (__attribute__((address_space(3))) void*)(
                    buf + r * S::kRowF + (p * S::kSpan + c) * S::kIl);
                if (S::kIl == 4 || lane_cols == 4)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 16, voff, 0, 0, 0);
                else
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 4, voff, 0, 0, 0);
            }
        }
    }
}

// The rows of one staged chunk, after issuing the next chunk's DMA.  xi, xf: the
// rays' 32.32 positions; buf holds columns from cm on.  test: some ray is not
// inside on some row of the chunk; rays with k outside [kin, kout) then read
// zeros.  (Only the addresses are in the two branches: the sums stay in place.)
template <int NB, int V, int SPAN>
__device__ __forceinline__ void fp_chunk(const float* src, size_t plane, int nsteps, int rowlen,
                                         int planes, float* __restrict__ next,
                                         const float* __restrict__ buf, int k0, int cm, int cm_next,
                                         int cols_next, bool test, int lane, const int (&kin)[V],
                                         const int (&kout)[V], long long (&x)[V],
                                         const long long (&off)[V], float (&sum)[V][NB])
{
    using S = FpShape<NB, SPAN>;
    if (cols_next > 0)
        fp_stage<NB, SPAN>(src, plane, nsteps, rowlen, k0 + S::kRows, cm_next, cols_next, planes, next,
                     lane);
#pragma unroll
    for (int r = 0; r < S::kRows; ++r) {
        int at[V];  // floats from buf
        float u[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            at[v] = (static_cast<int>(x[v] >> 32) - cm) * S::kIl + r * S::kRowF;
            u[v] = static_cast<float>(static_cast<unsigned int>(x[v])) * 0x1p-32f;
        }
        if (test) {
#pragma unroll
            for (int v = 0; v < V; ++v) {
                // a position within rounding of the first column belongs to it
                const bool neg = x[v] < 0;
                u[v] = neg ? 0.0f : u[v];
                at[v] = neg ? r * S::kRowF - cm * S::kIl : at[v];
                at[v] = k0 + r >= kin[v] && k0 + r < kout[v] ? at[v] : S::kZero;
            }
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const float w0 = 1.0f - u[v];
            const float* q = buf + at[v];
#pragma unroll
            for (int p = 0; p < S::kPlanes; ++p) {
                if constexpr (S::kIl == 4) {
                    const float4 a = *reinterpret_cast<const float4*>(q + p * S::kSpan * 4);
                    const float4 c = *reinterpret_cast<const float4*>(q + p * S::kSpan * 4 + 4);
                    float* s = sum[v] + 4 * p;
                    s[0] = fmaf(u[v], c.x, fmaf(w0, a.x, s[0]));
                    s[1] = fmaf(u[v], c.y, fmaf(w0, a.y, s[1]));
                    s[2] = fmaf(u[v], c.z, fmaf(w0, a.z, s[2]));
                    s[3] = fmaf(u[v], c.w, fmaf(w0, a.w, s[3]));
                } else {
                    sum[v][0] = fmaf(u[v], q[1], fmaf(w0, q[0], sum[v][0]));
                }
            }
            x[v] += off[v];
        }
    }
}

// Grid: (channel group, view group), slice group, branch.  A workgroup serves
// the views of its group that march its branch's rows; the few groups with
// views of both take two workgroups at once, the others' second one ends at
// the mask.  The prologue loops over the views and passes its results through
// LDS: unrolled, its code alone (fetched once) took longer than a small scan.
template <int NB, int V, int SPAN>
__global__ __launch_bounds__(512) void fp_stream_kernel(const FpStreamLaunch L)
{
    using S = FpShape<NB, SPAN>;
    static_assert(S::kLds >= V * 64 * 16, "the prologue's results fit the buffers");
    extern __shared__ __align__(16) unsigned char smem[];
    const FpProblem& P = L.P;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform_i(tid >> 6);
    const int nwaves = blockDim.x >> 6;
    const bool xb = blockIdx.z == 0;
    // neighbouring channels and views on one XCD: they share image columns
    const int id = xcd_tile(blockIdx.x, gridDim.x);
    const int s0 = (id % L.cgroups) * 64, a0 = (id / L.cgroups) * V;
    const int al = min(a0 + min(lane, V - 1), P.na - 1);  // lane v: view v
    const bool branch_x = L.usex[al] != 0;
    const unsigned int act = static_cast<unsigned int>(
        __ballot(lane < V && a0 + lane < P.na && branch_x == xb));
    if (act == 0) return;  // the whole workgroup
    const double trig = L.sincos[2 * al + (xb ? 1 : 0)];

    float* mine = reinterpret_cast<float*>(smem + static_cast<size_t>(wave) * S::kLds);
    const int s = min(s0 + lane, P.ns - 1);
    const int bg = blockIdx.y * NB, nb = min(NB, L.nb - bg);
    const int planes = (nb + S::kIl - 1) / S::kIl;
    const size_t plane = static_cast<size_t>(P.nx) * P.ny * S::kIl;
    const int nsteps = xb ? P.ny : P.nx, rowlen = xb ? P.nx : P.ny;
    const float* src = (xb ? L.rows : L.cols) + static_cast<size_t>(L.b0 + bg) * P.nx * P.ny;
    const int ka = min(wave * L.chunks * S::kRows, nsteps);
    const int kb = min(ka + L.chunks * S::kRows, nsteps);

    // every ray's rows and position at row ka (32.32; rays far off the image are
    // held within the range, they have no rows)
    struct alignas(16) Ray {
        long long x;
        int kin, kout;
    };
    Ray* rays = reinterpret_cast<Ray*>(mine);
    int first = 1 << 30, last = 0, fin = 0, fout = 1 << 30;
    float slope = 0.0f, lo_l = 1e30f, hi_l = -1e30f;  // lane v: view v's
    int olo = 0, ohi = 0;
    double2 ray = reinterpret_cast<const double2*>(L.bo)[static_cast<size_t>(a0) * P.ns + s];
#pragma unroll 1
    for (int v = 0; v < V; ++v) {
        const double x0 = ray.x, off = ray.y;
        ray = reinterpret_cast<const double2*>(
            L.bo)[static_cast<size_t>(min(a0 + v + 1, P.na - 1)) * P.ns + s];
        Ray r;
        int f0, f1;
        fp_ray_rows(x0, off, rowlen - 1, nsteps, r.kin, r.kout, f0, f1);
        const bool on = act >> v & 1;
        if (!on) r.kin = r.kout = f1 = 0;
        if (r.kin < r.kout) {
            first = min(first, r.kin);
            last = max(last, r.kout);
        }
        fin = max(fin, f0);
        fout = min(fout, f1);
        const double at = fma(static_cast<double>(ka), off, x0);
        r.x = static_cast<long long>(rint(fmin(fmax(at, -1e6), 1e6) * 0x1p32));
        rays[v * 64 + lane] = r;
        // columns of the view's rays at row k: [lo_l, hi_l] + k slope
        const float xf = static_cast<float>(x0), xa = lane_value(xf, 0), xz = lane_value(xf, 63);
        const float sl = uniform_f(static_cast<float>(off)), drift = (S::kRows - 1) * sl;
        const long long o = static_cast<long long>(rint(fmin(fmax(off, -2.0), 2.0) * 0x1p32));
        if (lane == v) {
            slope = sl;
            lo_l = on ? fminf(xa, xz) + fminf(0.0f, drift) : 1e30f;
            hi_l = on ? fmaxf(xa, xz) + fmaxf(0.0f, drift) : -1e30f;
            olo = static_cast<int>(o);
            ohi = static_cast<int>(o >> 32);
        }
    }
    first = wave_min(first);
    last = -wave_min(-last);
    fin = -wave_min(-fin);
    fout = wave_min(fout);
    const int kbeg = max(ka, min(first, nsteps) / S::kRows * S::kRows), kend = min(kb, last);
    const int nchunks = kbeg < kend ? (kend - kbeg + S::kRows - 1) / S::kRows : 0;
    long long x[V], off[V];
    int kin[V], kout[V];
    float sum[V][NB];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const Ray r = rays[v * 64 + lane];
        kin[v] = r.kin;
        kout[v] = r.kout;
        off[v] = static_cast<long long>(__builtin_amdgcn_readlane(ohi, v)) << 32 |
                 static_cast<unsigned int>(__builtin_amdgcn_readlane(olo, v));
        x[v] = r.x + (kbeg - ka) * off[v];
#pragma unroll
        for (int b = 0; b < NB; ++b) sum[v][b] = 0.0f;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    for (int e = S::kZero + lane; e < S::kBuf; e += 64) mine[e] = mine[S::kBuf + e] = 0.0f;

    int cm_l = 0, cols_l = 0;  // chunk (64 j + lane)'s first column and count
    const auto spans = [&](int h0) {
        const float k = static_cast<float>(kbeg + (h0 + lane) * S::kRows);
        float xmin = 1e30f, xmax = -1e30f;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const float sl = lane_value(slope, v);
            xmin = fminf(xmin, fmaf(k, sl, lane_value(lo_l, v)));
            xmax = fmaxf(xmax, fmaf(k, sl, lane_value(hi_l, v)));
        }
        const FpSpan c = fp_span(xmin, xmax, rowlen, S::kSpan);
        cm_l = c.first;
        cols_l = h0 + lane < nchunks ? fp_columns<S::kIl>(c, rowlen) : 0;
    };
    spans(0);
    int cm = uniform_i(cm_l);
    float *buf = mine, *next = mine + S::kBuf;
    if (nchunks > 0)
        fp_stage<NB, SPAN>(src, plane, nsteps, rowlen, kbeg, cm, uniform_i(cols_l), planes, buf, lane);
#pragma unroll 1
    for (int h = 0; h < nchunks; ++h) {
        if (((h + 1) & 63) == 0) spans(h + 1);
        const int cm_next = __builtin_amdgcn_readlane(cm_l, (h + 1) & 63);
        const int cols_next = __builtin_amdgcn_readlane(cols_l, (h + 1) & 63);
        const int k0 = kbeg + h * S::kRows;
        const bool test = k0 < fin || k0 + S::kRows > fout;
        // this wave's DMAs have landed; nothing else writes its LDS
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        fp_chunk<NB, V, SPAN>(src, plane, nsteps, rowlen, planes, next, buf, k0, cm, cm_next,
                        h + 1 < nchunks ? cols_next : 0, test, lane, kin, kout, x, off, sum);
        float* t = buf;
        buf = next;
        next = t;
        cm = cm_next;
    }

    // Segments' sums through LDS, one view at a time, in FP64 and in row order.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const double dw_l = fabs((xb ? P.dy : P.dx) / trig);
#pragma unroll 1
    for (int v = 0; v < V; ++v) {
        if (!(act >> v & 1)) continue;  // uniform
        __syncthreads();  // the previous view has been read
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float t = sum[0][b];
#pragma unroll
            for (int j = 1; j < V; ++j) t = v == j ? sum[j][b] : t;
            mine[b * 64 + lane] = t;
        }
        __syncthreads();
        const double dw = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(dw_l), v),
                                           __builtin_amdgcn_readlane(__double2loint(dw_l), v));
        for (int e = tid; e < nb * 64; e += nwaves * 64) {
            double t = 0.0;
            for (int w = 0; w < nwaves; ++w)
                t += static_cast<double>(
                    reinterpret_cast<const float*>(smem + static_cast<size_t>(w) * S::kLds)[e]);
            const int ch = s0 + (e & 63);
            if (ch < P.ns)
                L.proj[(static_cast<size_t>(L.b0 + bg + (e >> 6)) * P.na + a0 + v) * P.ns + ch] =
                    static_cast<float>(t * dw);
        }
    }
}

// rows[plane][y][x][4] and cols[plane][x][y][4] of 4-slice planes (zero past the
// batch); one slice (IL = 1) needs the transposed copy only.
template <int IL>
__global__ __launch_bounds__(256) void image_planes_kernel(const float* __restrict__ img,
                                                           float* __restrict__ rows,
                                                           float* __restrict__ cols, int ny, int nx,
                                                           int nbatch)
{
    __shared__ float tile[IL][32][33];
    const size_t slice = static_cast<size_t>(nx) * ny, base = blockIdx.z * slice * IL;
    const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int y = y0 + r, x = x0 + threadIdx.x;
        if (y >= ny || x >= nx) continue;
        float v[IL];
#pragma unroll
        for (int b = 0; b < IL; ++b) {
            const int sl = blockIdx.z * IL + b;
            v[b] = sl < nbatch ? img[sl * slice + static_cast<size_t>(y) * nx + x] : 0.0f;
            tile[b][r][threadIdx.x] = v[b];
        }
        if constexpr (IL == 4)
            *reinterpret_cast<float4*>(rows + base + (static_cast<size_t>(y) * nx + x) * 4) =
                make_float4(v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int x = x0 + r, y = y0 + threadIdx.x;
        if (y >= ny || x >= nx) continue;
        float* d = cols + base + (static_cast<size_t>(x) * ny + y) * IL;
        if constexpr (IL == 4)
            *reinterpret_cast<float4*>(d) = make_float4(tile[0][threadIdx.x][r], tile[1][threadIdx.x][r],
                                                        tile[2][threadIdx.x][r], tile[3][threadIdx.x][r]);
        else
            *d = tile[0][threadIdx.x][r];
    }
}

}  // namespace ctr
