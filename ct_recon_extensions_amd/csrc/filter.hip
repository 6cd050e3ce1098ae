// Ramp filter and fan weighting for gfx950.
//
// ramp_kernel: one workgroup filters ROWS detector rows.  The rows are
// staged in LDS (optionally multiplied by the fan / flat cosine weight on the
// way in, FanWeighting<T> src/fan_weighting.cc:19-35, so the weighting costs
// no extra pass over HBM), zero-padded by ns on both sides so no lane needs a
// range test.  The linear convolution of src/filter.cc:67-91,
//     out[is] = ds * sum_k in[k] h[is - k],
// is evaluated as h0*x[is] + sum over odd m of h[m] x[is - m]: even taps
// other than the centre are zero (src/filter.cc:26-30, :45-49), which halves
// the work.  The tap index is uniform across the workgroup (scalar loads),
// each tap is applied to all ROWS rows, and every lane reads consecutive
// LDS words (no bank conflicts).  The centre tap and the odd taps |m| <= 15
// (~97% of the filter's weight; on smooth rows they nearly cancel) are
// accumulated in FP64 with FP64 taps; the far field in FP32, added in FP64 at the
// end.  float64 rows have a kernel of their own, FP64 throughout.
// The transpose (RampFilterGrad) is the same operator since h is symmetric.
#include "ctr_common.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace ctr {

constexpr int kRampRows = 4;

struct RampParams {
    int ns, nrow, wtype;
    double ds, dso, dsd, cents;
};

__device__ inline double cos_weight(const RampParams& P, int is)
{
    const double s = P.ds * (static_cast<double>(is) - P.cents);
    if (P.wtype == 2) return P.dso * fabs(cos(atan2(s, P.dsd))) / P.dsd;
    return P.dso * fabs(cos(s / P.dsd)) / P.dsd;
}

// hf: taps in FP32, hf[ns + m] = h[m]; zero-padded rows in LDS.
constexpr int kRampNear = 15;  // |m| <= kRampNear: FP64 near field

__global__ __launch_bounds__(256) void ramp_kernel(const float* __restrict__ in,
                                                   float* __restrict__ out,
                                                   const float* __restrict__ hf,
                                                   const double* __restrict__ h64, RampParams P)
{
    extern __shared__ __align__(16) unsigned char smem[];
    float* xs = reinterpret_cast<float*>(smem);  // [ROWS][3*ns]
    const int ns = P.ns, pitch = 3 * ns;
    const int r0 = blockIdx.x * kRampRows;
    const int nr = min(kRampRows, P.nrow - r0);
    for (int e = threadIdx.x; e < kRampRows * pitch; e += 256) {
        const int r = e / pitch, c = e - r * pitch - ns;
        float v = 0;
        if (r < nr && c >= 0 && c < ns) {
            const float x = in[static_cast<size_t>(r0 + r) * ns + c];
            v = P.wtype ? static_cast<float>(cos_weight(P, c) * static_cast<double>(x))
                        : x;
        }
        xs[e] = v;
    }
    __syncthreads();
    const double h0 = h64[ns];
    // odd m in [-(ns-1), ns-1]; x index ns + is - m stays in [1, 3ns-1]
    const int mlo = -(ns - 1) | 1;  // smallest odd >= -(ns-1)
    const int nlo = max(mlo, -kRampNear), nhi = min(ns - 1, kRampNear);
    for (int is = threadIdx.x; is < ns; is += 256) {
        float acc[kRampRows];
        double near[kRampRows];
#pragma unroll
        for (int r = 0; r < kRampRows; ++r) {
            acc[r] = 0.0f;
            near[r] = h0 * static_cast<double>(xs[r * pitch + ns + is]);
        }
        for (int m = mlo; m < nlo; m += 2) {
            const float h = hf[ns + m];
            const int xi = ns + is - m;
#pragma unroll
            for (int r = 0; r < kRampRows; ++r) acc[r] = fma(h, xs[r * pitch + xi], acc[r]);
        }
        for (int m = nlo; m <= nhi; m += 2) {
            const double h = h64[ns + m];
            const int xi = ns + is - m;
#pragma unroll
            for (int r = 0; r < kRampRows; ++r)
                near[r] = fma(h, static_cast<double>(xs[r * pitch + xi]), near[r]);
        }
        for (int m = nhi + 2; m <= ns - 1; m += 2) {
            const float h = hf[ns + m];
            const int xi = ns + is - m;
#pragma unroll
            for (int r = 0; r < kRampRows; ++r) acc[r] = fma(h, xs[r * pitch + xi], acc[r]);
        }
#pragma unroll
        for (int r = 0; r < kRampRows; ++r)
            if (r < nr)
                out[static_cast<size_t>(r0 + r) * ns + is] =
                    static_cast<float>((near[r] + static_cast<double>(acc[r])) * P.ds);
    }
}

// float64 rows: one workgroup a row, a wave 256 outputs at a time.  One 8-byte LDS
// read a multiply-add is what bounded ramp_kernel here (with two workgroups a CU,
// 1.4 of them for each); a lane takes the four outputs 8 q + p + 2 j (p its parity),
// which share their samples: for the four taps m = 8 k + 1 + 2 u it needs the samples
// 8 (q - k) - 1 + p + 2 (j - u), i.e. the four of its parity in block q - k, which it
// holds, and those in block q - k - 1, which it reads: 16 multiply-adds for 4 reads.
// Blocks of 8 are stored 10 apart: the lanes' reads meet every bank once.  A wave
// leaves out the taps that meet only padding.  Each output adds the same products in
// the same order as in ramp_kernel.  1440 rows of 736: 165 -> 40 us (73 with
// every group's taps clamped), and the copy of the taps (4 us) is not made.
constexpr int kWideOut = 256;   // outputs of a wave
constexpr int kWidePitch = 10;  // doubles a block of 8 samples
// Blocks of padding before the row.  A wave at output i0 takes taps from
// i0 - ns - 8 to i0 + 256 (and from -15 to 15), so blocks from -33 to ns / 8 + 33.
constexpr int kWidePad = 36;
inline __host__ __device__ int wide_blocks(int ns) { return ns / 8 + 2 * kWidePad; }

__global__ __launch_bounds__(512) void ramp_f64_kernel(const double* __restrict__ in,
                                                       double* __restrict__ out,
                                                       const double* __restrict__ h,
                                                       RampParams P)
{
    extern __shared__ __align__(16) unsigned char smem[];
    double* xs = reinterpret_cast<double*>(smem);
    const int ns = P.ns;
    const size_t r0 = static_cast<size_t>(blockIdx.x) * ns;
    for (int e = threadIdx.x; e < 8 * wide_blocks(ns); e += blockDim.x) {
        const int c = e - 8 * kWidePad - 1;
        double v = 0;
        if (c >= 0 && c < ns) {
            v = in[r0 + c];
            if (P.wtype) v = cos_weight(P, c) * v;
        }
        xs[kWidePitch * (e >> 3) + (e & 7)] = v;
    }
    __syncthreads();
    const double h0 = h[ns];
    const int lane = threadIdx.x & 63, p = lane & 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int i0 = wave * kWideOut; i0 < ns; i0 += (blockDim.x >> 6) * kWideOut) {
        const int q = i0 / 8 + (lane >> 1), i1 = min(i0 + kWideOut, ns) - 1;
        const double* row = xs + kWidePitch * (q + kWidePad) + p;
        double cur[4], acc[4], near[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = p + 2 * j + 1;  // output 8 q + p + 2 j as a sample
            acc[j] = 0.0;
            near[j] = h0 * row[kWidePitch * (e >> 3) + (e & 7) - p];
        }
        const auto load = [&](int k) {
#pragma unroll
            for (int j = 0; j < 4; ++j) cur[j] = row[-kWidePitch * k + 2 * j];
        };
        // EDGE: taps past |m| = ns - 1 count as zero (else the four are read at once)
        const auto taps = [&](auto EDGE, double(&a)[4], int k) {
            double nxt[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) nxt[j] = row[-kWidePitch * (k + 1) + 2 * j];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int m = 8 * k + 1 + 2 * u;
                double hm;
                if constexpr (EDGE.value) {
                    const double t = h[ns + min(max(m, 1 - ns), ns - 1)];
                    hm = abs(m) < ns ? t : 0.0;
                } else {
                    hm = h[ns + m];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) a[j] = fma(hm, j >= u ? cur[j - u] : nxt[4 + j - u], a[j]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) cur[j] = nxt[j];
        };
        // near groups: m = -15 ... 15
        constexpr int kNearLo = -(kRampNear + 1) / 8, kNearHi = kRampNear / 8;
        const int klo = min((i0 - ns) >> 3, kNearLo);
        const int khi = max((i1 - 1) >> 3, kNearHi);
        // only the first and the last group of a row reach past its taps
        constexpr std::true_type edge{};
        constexpr std::false_type inner{};
        load(klo);
        if (klo < kNearLo) taps(edge, acc, klo);
#pragma unroll 2
        for (int k = klo + 1; k < kNearLo; ++k) taps(inner, acc, k);
#pragma unroll
        for (int k = kNearLo; k <= kNearHi; ++k) taps(edge, near, k);
#pragma unroll 2
        for (int k = kNearHi + 1; k < khi; ++k) taps(inner, acc, k);
        if (khi > kNearHi) taps(edge, acc, khi);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int is = 8 * q + p + 2 * j;
            if (is < ns) out[r0 + is] = (near[j] + acc[j]) * P.ds;
        }
    }
}

__global__ void taps_kernel(const double* __restrict__ h, float* __restrict__ hf, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) hf[i] = static_cast<float>(h[i]);
}

template <typename T>
__global__ void fanw_kernel(const T* __restrict__ in, T* __restrict__ out, RampParams P)
{
    const size_t n = static_cast<size_t>(P.nrow) * P.ns;
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const int is = static_cast<int>(i % P.ns);
        out[i] = static_cast<T>(cos_weight(P, is) * static_cast<double>(in[i]));
    }
}

namespace {

int ramp_f32(const ctr_geom& g, const float* in, float* out, unsigned int nrow, const double* filter,
             int wtype, hipStream_t st)
{
    RampParams P{static_cast<int>(g.ns), static_cast<int>(nrow), wtype, g.ds, g.dso, g.dsd,
                 cent_s(g)};
    const size_t lds = static_cast<size_t>(kRampRows) * 3 * g.ns * sizeof(float);
    CTR_REQUIRE(lds <= 160 * 1024, CTR_ERR_SHAPE, "ramp filter: ns too large for LDS");
    const int ntaps = 2 * g.ns + 1;
    float* hf = nullptr;
    CTR_HIP(ctr::ws_alloc(reinterpret_cast<void**>(&hf), ntaps * sizeof(float), st));
    hipLaunchKernelGGL(taps_kernel, dim3(div_up(ntaps, 256)), dim3(256), 0, st, filter, hf,
                       ntaps);
    int rc = check_launch("taps_kernel");
    if (rc == CTR_OK) {
        auto kern = ramp_kernel;
        if (lds > 64 * 1024)
            CTR_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(lds)));
        hipLaunchKernelGGL(kern, dim3(div_up(nrow, kRampRows)), dim3(256), lds, st, in, out,
                           static_cast<const float*>(hf), filter, P);
        rc = check_launch("ramp_kernel");
    }
    CTR_HIP(ctr::ws_free(hf, st));
    return rc;
}

}  // namespace

int ramp(const ctr_geom& g, int dtype, const void* in, void* out, unsigned int nrow,
         const double* filter, int weight_type, hipStream_t st)
{
    if (dtype == CTR_F32)
        return ramp_f32(g, static_cast<const float*>(in), static_cast<float*>(out), nrow, filter,
                        weight_type, st);
    const int ns = static_cast<int>(g.ns);
    // rows of up to 1706 channels, as the entry point has always taken
    CTR_REQUIRE(static_cast<size_t>(ns) * 96 <= 160 * 1024, CTR_ERR_SHAPE,
                "ramp filter: ns too large for LDS");
    RampParams P{ns, static_cast<int>(nrow), weight_type, g.ds, g.dso, g.dsd, cent_s(g)};
    const size_t lds = static_cast<size_t>(wide_blocks(ns)) * kWidePitch * sizeof(double);
    // a grid holds fewer than 2^32 lanes
    constexpr unsigned int kRowsPerGrid = 1u << 22;
    for (unsigned int r = 0; r < nrow; r += kRowsPerGrid) {
        const size_t o = static_cast<size_t>(r) * ns;
        hipLaunchKernelGGL(ramp_f64_kernel, dim3(std::min(kRowsPerGrid, nrow - r)),
                           dim3(64 * div_up(ns, kWideOut)), lds, st,
                           static_cast<const double*>(in) + o, static_cast<double*>(out) + o,
                           filter, P);
        const int rc = check_launch("ramp_f64_kernel");
        if (rc) return rc;
    }
    return CTR_OK;
}

int fan_weighting(const ctr_geom& g, int dtype, const void* in, void* out, unsigned int nrow,
                  hipStream_t st)
{
    RampParams P{static_cast<int>(g.ns), static_cast<int>(nrow), g.type, g.ds, g.dso, g.dsd,
                 cent_s(g)};
    const size_t n = static_cast<size_t>(nrow) * g.ns;
    const dim3 grid(static_cast<unsigned int>(std::min<size_t>(8192, (n + 255) / 256)));
    if (dtype == CTR_F32)
        hipLaunchKernelGGL(fanw_kernel<float>, grid, dim3(256), 0, st,
                           static_cast<const float*>(in), static_cast<float*>(out), P);
    else
        hipLaunchKernelGGL(fanw_kernel<double>, grid, dim3(256), 0, st,
                           static_cast<const double*>(in), static_cast<double*>(out), P);
    return check_launch("fanw_kernel");
}

}  // namespace ctr
