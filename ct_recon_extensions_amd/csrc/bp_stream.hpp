// Forward backprojection with wave-private view streams (float32), for the
// geometries whose detector position is a low-order polynomial along a short
// run of pixels (others: bp_engine.hpp).  What bounds a BP is the issue of the
// geometry of a pixel-view, the more so the fewer slices (16, 8, 4, 2 or 1) share
// it, and the work is split to make it cheap:
//  * a lane owns a run of M pixels of an image row.  Per view it evaluates
//    the geometry once, at the run's centre, with its derivatives along the
//    row (Geo::run), and every pixel of the run takes the position and the
//    weight from that polynomial; pixels at +d and -d share its even and odd
//    halves.  For the fan: ~43 VALU slots a run + 3.5 a pixel against 17 (a
//    reciprocal among them, 4 slots) a pixel, i.e. 9 against 20 at M = 8;
//  * a 16 x 16 pixel tile then needs 256 / M lanes, so a wave walks
//    64 * M / 256 views at once (two at M = 8, one in each half);
//  * a workgroup is one tile x NB slices, its waves take consecutive parts
//    of the views, and each wave stages the detector spans of its own views
//    into its own LDS ring (buffer loads that write LDS, double-buffered):
//    no barrier until the waves' partial images are added, in FP64 and in
//    wave order, at the end.  The wave count per tile (stream_waves) is
//    also what fills the chip when the image is small: a 256^2 slice has 256
//    tiles, a quarter of the waves it takes to hide latency.
//  * a wave evaluates the FP64 anchors of all its views first (64 at a time,
//    one a lane) and keeps them in LDS, while no sum is live in registers.
// Sums: one FP32 chain of at most kStreamChain views a lane, the halves of a
// wave added in FP32, the waves in FP64.  The split depends on the batch: runs are
// of 4 pixels in groups of 16 slices and of 8 in smaller ones (the sums of 16 x 8
// pixels do not fit the registers), and the wave count follows the number of
// workgroups.  So a slice's last bits are those of its batch size.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "bp_engine.hpp"
#include "ctr_common.hpp"
#include "interleave.hpp"
#include "tile_common.hpp"

namespace ctr {

constexpr int kStreamTile = 16;      // tile side in pixels
constexpr int kStreamChain = 96;     // views a lane may add in one FP32 chain
constexpr int kStreamMaxWaves = 16;  // waves per workgroup
constexpr int kStreamMaxPitch = 128; // channels of a staged span

// Position and weight along a run: base + c0 + c1 d + ... + c4 d^4 channels
// from the span's first and w0 + w1 d + w2 d^2 + w3 d^3 (d in pixels from the
// run's centre).  The whole channels of the centre are in `base`, and c0 is
// the fraction plus an offset that keeps the sum positive (its truncation is
// the floor): a position is rounded at the size of a run, not of a span.
struct RunPoly {
    float c0, c1, c2, c3, c4, w0, w1, w2, w3;
    int base;
};

// base and c0 of a centre at whole + frac + t channels, for runs that stay
// within off channels of their centre.
__device__ __forceinline__ void run_base(RunPoly& R, int whole, float frac, float t, float off)
{
    const float fl = floorf(t);
    R.base = whole + static_cast<int>(fl - off);
    R.c0 = frac + (t - fl) + off;
}

template <class Geo>
struct StreamLaunch {
    typename Geo::Problem P;
    int nbatch, tiles_x, tiles_y;
    int pitch;       // channels per staged span (a multiple of 16)
    int vchunk;      // views per LDS buffer (a multiple of the views in flight)
    int views;       // anchors a wave keeps
    int wave_bytes;  // LDS per wave
    double scale;
    const float* src;  // [slice group][na][ns][slices of a group]
    float* img;
};

template <int NB, int M>
struct StreamShape {
    static constexpr int kIl = NB < 4 ? NB : 4;      // slices interleaved per LDS word group
    static constexpr int kGroups = NB / kIl;
    static constexpr int kViews = M / 4;             // views a wave walks at once
    static constexpr int kCh = 64 / kIl;             // channels per DMA
    static constexpr int kRuns = kStreamTile / M;    // runs per tile row
    static_assert(NB == 1 || NB == 2 || NB % 4 == 0, "slices: 1, 2 or a multiple of 4");
    static_assert(M == 4 || M == 8, "run length");
    // views of a wave: FP32 chains of kStreamChain on each lane
    static constexpr int kMaxViews = kStreamChain * kViews;
};

// LDS of one wave: the packed anchors of its views, two span buffers; the
// partial image of one slice group (kIl x 256 floats) reuses it at the end.
inline int stream_wave_bytes(int il, int nb, int pitch, int vchunk, int views)
{
    const int spans = 2 * vchunk * pitch * nb * 4;
    return std::max(views * 32 + spans, il * kStreamTile * kStreamTile * 4);
}

// Views per buffer: what 10 KB a wave (16 waves on a CU) leaves beside the
// anchors of 96 views, at least the views in flight, at most 16.
inline int stream_vchunk(int views, int nb, int pitch)
{
    const int fit = (10 * 1024 - 96 * 32) / (2 * pitch * nb * 4) / views * views;
    return std::max(views, std::min(16, fit));
}

// A lane's part in the staging DMAs, fixed for the tile: with 16 bytes a lane a
// view's span of one slice group takes pitch * kIl / 4 lanes, and where that
// leaves room one DMA brings `per` views (their spans follow each other in LDS;
// with one slice group only).
struct StageLane {
    int per, sub, li, lanes;
};

template <int NB, int M>
__device__ __forceinline__ StageLane stage_lane(int pitch, int lane)
{
    using S = StreamShape<NB, M>;
    StageLane G;
    G.lanes = pitch * S::kIl / 4;
    G.per = S::kGroups == 1 && G.lanes <= 64 ? 64 / G.lanes : 1;
    G.sub = G.per > 1 ? lane / G.lanes : 0;
    G.li = lane - G.sub * G.lanes;
    return G;
}

// Stage the spans of views va + vc .. va + vc + nv - 1 into
// buf[view][group][channel][kIl slices].  The source has the slices of a group
// interleaved per channel (interleave_kernel; a single slice is the sinogram
// itself), so a lane moves 16 bytes: 4, 2 or 1 channels of 1, 2 or 4 slices.  With
// 4 bytes a lane, the slices apart, the DMAs of 4-slice groups cost as much as
// the sums (the 4-slice BP of 512^2, 720 views: 227 us against 150).
// RAW (calls that must not or cannot allocate, or are captured) stages the sinograms
// as they are, 4 bytes a lane: the same spans, hence the same sums (FP transpose of
// 512^2, 720 views, engine -> RAW -> interleaved: 8 slices 249, 222, 206 us, 16 slices
// 453, 352, 335).
// Off the detector: without EDGE every tap is inside, and what the span holds
// past the row is not read (past the last row's end a 16-byte load still brings
// the channels before the end; stream_tile keeps spans before the first row's
// start out); with EDGE those channels read as zero (an offset of
// 2^31 is out of range), per lane for 4 slices, else with 4 bytes a lane.
template <class Geo, int NB, int M, bool EDGE, bool RAW>
__device__ __forceinline__ void stream_stage(const StreamLaunch<Geo>& L, const StageLane& G,
                                             const typename Geo::StreamAnchor* anchors, float* buf,
                                             int va, int vc, int nv, const float* src, int nb,
                                             int lane)
{
    using S = StreamShape<NB, M>;
    const auto& P = L.P;
    const unsigned int row_bytes = static_cast<unsigned int>(P.ns) * S::kIl * 4u;
    const unsigned int bytes = static_cast<unsigned int>(P.na) * row_bytes;  // of a slice group
    const size_t group = static_cast<size_t>(P.na) * P.ns * S::kIl;
    if constexpr (RAW && NB > 1) {
        // lane -> slice lane % kIl, channel lane / kIl: its offset in the group's first
        // 64 words is fixed for the tile.  Without EDGE a channel before or past the row
        // reads a neighbour (or zero) and is no tap.
        const unsigned int slice_bytes = static_cast<unsigned int>(P.na) * P.ns * 4u;
        const int lane_ch = lane / S::kIl, words = L.pitch * S::kIl;
        const unsigned int lane_off =
            (lane % S::kIl) * slice_bytes + static_cast<unsigned int>(lane_ch) * 4u;
#pragma unroll 1
        for (int t = 0; t < nv; ++t) {
            const int is0 = uniform_i(anchors[vc + t].is0);
            const unsigned int at =
                lane_off + static_cast<unsigned int>((va + vc + t) * P.ns + is0) * 4u;
#pragma unroll 1
            for (int w0 = 0; w0 < words; w0 += 64) {
                unsigned int voff = at + w0 / S::kIl * 4;
                if constexpr (EDGE)
                    if (static_cast<unsigned int>(is0 + lane_ch + w0 / S::kIl) >=
                        static_cast<unsigned int>(P.ns))
                        voff = 0x80000000u;
                if (w0 + lane >= words) continue;
#pragma unroll
                for (int g = 0; g < S::kGroups; ++g) {
                    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                        const_cast<float*>(src + g * group), 0,
                        static_cast<unsigned int>(max(0, min(S::kIl, nb - S::kIl * g))) * slice_bytes,
                        0x00020000);
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        rs,
                        (__attribute__((address_space(3))) void*)(
                            buf + (t * NB + g * S::kIl) * L.pitch + w0),
                        4, voff, 0, 0, 0);
                }
            }
        }
    } else if constexpr (EDGE && S::kIl < 4) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(src), 0, bytes, 0x00020000);
#pragma unroll 1
        for (int t = 0; t < nv; ++t) {
            const int is0 = anchors[vc + t].is0;
            const unsigned int row = static_cast<unsigned int>(va + vc + t) * row_bytes;
#pragma unroll 1
            for (int w0 = 0; w0 < L.pitch * S::kIl; w0 += 64) {
                const int w = w0 + lane, ch = is0 + w / S::kIl;
                const unsigned int voff =
                    static_cast<unsigned int>(ch) < static_cast<unsigned int>(P.ns)
                        ? row + static_cast<unsigned int>(ch * S::kIl + w % S::kIl) * 4u
                        : 0x80000000u;
                if (w < L.pitch * S::kIl)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        rs, (__attribute__((address_space(3))) void*)(buf + t * NB * L.pitch + w0), 4,
                        voff, 0, 0, 0);
            }
        }
    } else {
#pragma unroll 1
        for (int t = 0; t < nv; t += G.per) {
            const int tv = t + G.sub;
            if (G.sub >= G.per || tv >= nv) continue;
            const int is0 = anchors[vc + tv].is0;
            const int row = (va + vc + tv) * static_cast<int>(row_bytes);
#pragma unroll 1
            for (int li = G.li; li < G.lanes; li += 64) {
                int voff = row + is0 * (S::kIl * 4) + li * 16;
                if constexpr (EDGE)
                    if (static_cast<unsigned int>(is0 + li) >= static_cast<unsigned int>(P.ns))
                        voff = static_cast<int>(0x80000000u);
#pragma unroll
                for (int g = 0; g < S::kGroups; ++g) {
                    // a group past the batch has no memory: range 0 reads as zero
                    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                        const_cast<float*>(src + g * group), 0, S::kIl * g < nb ? bytes : 0u,
                        0x00020000);
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        rs,
                        (__attribute__((address_space(3))) void*)(
                            buf + (t * NB + g * S::kIl) * L.pitch +
                            uniform_i(li - G.li) * 4),
                        16, voff, 0, 0, 0);
                }
            }
        }
    }
}

// Tap index (from R.base) and weights of the pixels of a run for one view.
template <class Geo, int M, bool EDGE>
__device__ __forceinline__ void stream_taps(const typename Geo::Problem& P,
                                            const typename Geo::StreamAnchor& A, const RunPoly& R,
                                            int pitch, int (&idx)[M], float (&w0)[M],
                                            float (&w1)[M])
{
#pragma unroll
    for (int h = 0; h < M / 2; ++h) {
        const float d = h + 0.5f, d2 = d * d;
        float fe = R.c0, fo = R.c1, we = R.w0, wo = R.w1;
        if constexpr (Geo::kRunDegree >= 3) {
            fe = fmaf(Geo::kRunDegree == 4 ? fmaf(R.c4, d2, R.c2) : R.c2, d2, R.c0);
            fo = fmaf(R.c3, d2, R.c1);
            we = fmaf(R.w2, d2, R.w0);
            if constexpr (Geo::kRunDegree == 4) wo = fmaf(R.w3, d2, R.w1);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const float sd = s ? d : -d;
            const int m = s ? M / 2 + h : M / 2 - 1 - h;
            const float f = fmaf(sd, fo, fe);
            const float fr = __builtin_amdgcn_fractf(f);
            idx[m] = static_cast<int>(f);
            if constexpr (HasCustomTaps<Geo>::value) {
                Geo::stream_weights(A, fr, R.w0, w0[m], w1[m]);
            } else {
                float w = Geo::kRunDegree >= 3 ? fmaf(sd, wo, we) : R.w0;
                if constexpr (EDGE) w = on_detector(A.is0 + R.base + idx[m], fr, P.ns) ? w : 0.0f;
                w1[m] = w * fr;
                w0[m] = w - w1[m];
            }
            // keeps the reads inside the span for any geometry
            if constexpr (EDGE)
                idx[m] = min(max(idx[m], -R.base), pitch - 2 - R.base);
        }
    }
}

// One step of a wave: the DMA of the nv_next views from vn on into `next` (at the
// start of a chunk), then the sums of the views v .. v + kViews - 1 < nva, whose
// spans are in buf.  The restrict qualifiers tell the compiler that the span
// and anchor reads cannot depend on the DMA in flight.
template <class Geo, int NB, int M, bool EDGE, bool RAW>
__device__ __forceinline__ void stream_step(
    const StreamLaunch<Geo>& L, const StageLane& G, const typename Geo::Problem& Pg,
    const typename Geo::StreamAnchor* __restrict__ anchors, float* __restrict__ next,
    const float* __restrict__ buf, int va, int v, int nva, int vn, int nv_next, const float* src,
    int nb, int lane, float fi, float fj, float (&acc)[M][NB])
{
    using S = StreamShape<NB, M>;
    if (nv_next > 0)
        stream_stage<Geo, NB, M, EDGE, RAW>(L, G, anchors, next, va, vn, nv_next, src, nb, lane);
    {
        const int half = S::kViews == 2 ? lane >> 5 : 0;
        const bool on = v + half < nva;
        const int tv = on ? half : 0;
        const typename Geo::StreamAnchor A = anchors[v + tv];
        int idx[M];
        float w0[M], w1[M];
        RunPoly R = Geo::run(Pg, A, fi, fj);
        // a half without a view in this step adds zeros
        if (!on) R.w0 = R.w1 = R.w2 = R.w3 = 0.0f;
        stream_taps<Geo, M, EDGE>(Pg, A, R, L.pitch, idx, w0, w1);
        const float* sv = buf + tv * NB * L.pitch + R.base * S::kIl;
#pragma unroll
        for (int m = 0; m < M; ++m) {
#pragma unroll
            for (int g = 0; g < S::kGroups; ++g) {
                const float* q = sv + g * S::kIl * L.pitch + idx[m] * S::kIl;
                if constexpr (S::kIl == 4) {
                    const float4 a = *reinterpret_cast<const float4*>(q);
                    const float4 c = *reinterpret_cast<const float4*>(q + 4);
                    float* s = acc[m] + 4 * g;
                    s[0] = fmaf(w1[m], c.x, fmaf(w0[m], a.x, s[0]));
                    s[1] = fmaf(w1[m], c.y, fmaf(w0[m], a.y, s[1]));
                    s[2] = fmaf(w1[m], c.z, fmaf(w0[m], a.z, s[2]));
                    s[3] = fmaf(w1[m], c.w, fmaf(w0[m], a.w, s[3]));
                } else if constexpr (S::kIl == 2) {
                    const float2 a = *reinterpret_cast<const float2*>(q);
                    const float2 c = *reinterpret_cast<const float2*>(q + 2);
                    acc[m][0] = fmaf(w1[m], c.x, fmaf(w0[m], a.x, acc[m][0]));
                    acc[m][1] = fmaf(w1[m], c.y, fmaf(w0[m], a.y, acc[m][1]));
                } else {
                    acc[m][0] = fmaf(w1[m], q[1], fmaf(w0[m], q[0], acc[m][0]));
                }
            }
            // 64 sums leave registers for the taps of two pixels in flight
            if constexpr (M * NB >= 64) {
                if (m & 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// All views of a wave, in chunks of L.vchunk.
template <class Geo, int NB, int M, bool EDGE, bool RAW>
__device__ __forceinline__ void stream_views(const StreamLaunch<Geo>& L, const StageLane& G,
                                             const typename Geo::Problem& Pg,
                                             const typename Geo::StreamAnchor* anchors,
                                             float* spans, int va, int nva, const float* src,
                                             int nb, int lane, float fi, float fj, float (&acc)[M][NB])
{
    using S = StreamShape<NB, M>;
    const int bufsz = L.vchunk * NB * L.pitch;
    float *buf = spans + bufsz, *next = spans;
    stream_stage<Geo, NB, M, EDGE, RAW>(L, G, anchors, next, va, 0, min(L.vchunk, nva), src, nb,
                                        lane);
    int left = 0;  // views of the chunk still to come
    const float* sv = buf;
#pragma unroll 1
    for (int v = 0; v < nva; v += S::kViews) {
        int nv_next = 0;
        if (left == 0) {
            // this wave's DMAs have landed; nothing else writes its LDS
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            float* t = buf;
            buf = next;
            next = t;
            sv = buf;
            left = L.vchunk;
            nv_next = min(L.vchunk, nva - v - L.vchunk);
        }
        stream_step<Geo, NB, M, EDGE, RAW>(L, G, Pg, anchors, next, sv, va, v, nva, v + L.vchunk,
                                           nv_next, src, nb, lane, fi, fj, acc);
        sv += S::kViews * NB * L.pitch;
        left -= S::kViews;
    }
}

// One tile x NB slices (from slice b0): the whole work of a workgroup of
// nwaves waves.  smem: nwaves regions of L.wave_bytes, of which L.views anchors
// are the first part.  A wave with more views (ROUNDS; the persistent ragged
// kernel, whose wave count is fixed) takes them in balanced rounds and adds the
// rounds' sums.  A persistent caller puts a barrier between tiles.
template <class Geo, int NB, int M, bool ROUNDS = false, bool RAW = false>
__device__ __forceinline__ void stream_tile(const typename Geo::Tables& T,
                                            const StreamLaunch<Geo>& L, int tile, int b0,
                                            int nwaves, unsigned char* smem)
{
    using S = StreamShape<NB, M>;
    using Anchor = typename Geo::StreamAnchor;
    static_assert(sizeof(Anchor) == 32, "packed anchors");
    const auto& P = L.P;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform_i(tid >> 6);
    unsigned char* mine = smem + static_cast<size_t>(wave) * L.wave_bytes;
    const int per = (P.na + nwaves - 1) / nwaves;  // views a wave, the last one fewer
    Anchor* anchors = reinterpret_cast<Anchor*>(mine);
    float* spans = reinterpret_cast<float*>(mine + L.views * sizeof(Anchor));

    const TileFrame F(tile, L.tiles_x, P.nx, P.ny, kStreamTile, kStreamTile);
    const int nb = min(NB, L.nbatch - b0);
    const float* src = L.src + static_cast<size_t>(b0) * P.na * P.ns;
    const StageLane G = stage_lane<NB, M>(L.pitch, lane);
    const int ilo = F.x0 - F.ic, jlo = F.y0 - F.jc;
    typename Geo::Problem Pg = P;
    if constexpr (HasPin<Geo>::value) Geo::pin(Pg);

    // lane -> run: 16 consecutive lanes (one pass of a 16-byte LDS read) take
    // 8 rows x 2 runs, whose taps of one pixel of the run span ~10 channels
    const int rl = lane % (64 / S::kViews);  // run of the tile
    int rx, ry;
    if constexpr (M == 8) {
        rx = (rl >> 3) & 1;
        ry = (rl & 7) + 8 * (rl >> 4);
    } else {
        rx = ((rl >> 3) & 1) + 2 * (rl >> 5);
        ry = (rl & 7) + 8 * ((rl >> 4) & 1);
    }
    const float fi = static_cast<float>(ilo + rx * M) + 0.5f * (M - 1);
    const float fj = static_cast<float>(jlo + ry);

    float acc[M][NB], total[ROUNDS ? M : 1][ROUNDS ? NB : 1];
    const auto clear = [](auto& x) {
#pragma unroll
        for (auto& r : x)
#pragma unroll
            for (float& v : r) v = 0.0f;
    };
    clear(acc);
    clear(total);
    int va = min(wave * per, P.na);
    const int vend = min(va + per, P.na);
    const int rounds = ROUNDS ? (vend - va + L.views - 1) / L.views : 1;
    for (int k = 0; k < rounds; ++k) {
        const int nva = (vend - va + rounds - k - 1) / (rounds - k);
        bool inside = true;  // no view of the round takes the tile past the detector
        for (int v = lane; v < nva; v += 64) {
            const typename Geo::Anchor A =
                Geo::anchor(P, T, F, va + v, ilo, ilo + kStreamTile - 1, jlo,
                            jlo + kStreamTile - 1);
            anchors[v] = Geo::pack(A);
            // a span that starts at channel -1 of the first view starts before the
            // buffer, and a 16-byte load there (4 or 2 channels) is out of range as
            // a whole: channels 0 to 2 with it.  EDGE stages channel by channel.
            const bool before = S::kIl < 4 && A.is0 < 0 && va + v == 0;
            inside = inside && A.inside != 0 && !before;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (__ballot(!inside) != 0)
            stream_views<Geo, NB, M, true, RAW>(L, G, Pg, anchors, spans, va, nva, src, nb, lane,
                                                fi, fj, acc);
        else
            stream_views<Geo, NB, M, false, RAW>(L, G, Pg, anchors, spans, va, nva, src, nb, lane,
                                                 fi, fj, acc);
        // every read of this wave's LDS is done before it is written again
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if constexpr (ROUNDS) {
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int b = 0; b < NB; ++b) total[m][b] += acc[m][b];
            clear(acc);
        }
        va += nva;
    }

    // Partial images, one slice group at a time: halves of a wave by a
    // shuffle, waves through LDS in FP64 and in wave order.
#pragma unroll
    for (int g = 0; g < S::kGroups; ++g) {
        if (g > 0) __syncthreads();  // the previous group has been read
        float* part = reinterpret_cast<float*>(mine);
#pragma unroll
        for (int b = 0; b < S::kIl; ++b) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                float v;
                if constexpr (ROUNDS) v = total[m][g * S::kIl + b];
                else v = acc[m][g * S::kIl + b];
                if constexpr (S::kViews == 2) v += __shfl_xor(v, 32);
                if (S::kViews == 1 || lane < 32)
                    part[b * 256 + ry * kStreamTile + rx * M + m] = v;
            }
        }
        __syncthreads();
        for (int e = tid; e < S::kIl * 256; e += nwaves * 64) {
            const int b = e >> 8, px = e & 255;
            double sum = 0.0;
            for (int w = 0; w < nwaves; ++w)
                sum += static_cast<double>(
                    reinterpret_cast<const float*>(smem + static_cast<size_t>(w) * L.wave_bytes)[e]);
            const int ix = F.x0 + (px & 15), iy = F.y0 + (px >> 4);
            const int sl = g * S::kIl + b;
            if (sl < nb && ix < P.nx && iy < P.ny)
                L.img[(static_cast<size_t>(b0 + sl) * P.ny + iy) * P.nx + ix] =
                    static_cast<float>(sum * L.scale);
        }
    }
}

template <class Geo, int NB, int M, bool RAW>
__global__ __launch_bounds__(64 * kStreamMaxWaves) void bp_stream_kernel(
    const typename Geo::Tables T, const StreamLaunch<Geo> L)
{
    extern __shared__ __align__(16) unsigned char smem[];
    int group;
    const int tile = super_tile(L.tiles_x, L.tiles_y, group);
    if (tile < 0) return;  // padding of the supertile grid: the whole workgroup
    stream_tile<Geo, NB, M, false, RAW>(T, L, tile, group * NB, blockDim.x >> 6, smem);
}

// ---------------------------------------------------------------- host side

// Waves per tile: 8 (two workgroups a CU, four waves a SIMD) or 16.  Measured on
// the fan BP with 3 to 16 waves: counts that are no multiple of 4 load the SIMDs
// unevenly (512^2, 720 views, 8 slices: 199 us at 8, 211 to 306 at 5 to 7, 217 at
// 3, 227 at 16); 16 is better where 8 leave CUs half empty (up to 256 tiles: 8
// slices of 256^2, 360 views, 54 against 58 us) or where the anchors of a wave's
// views keep a second workgroup off the CU (1024^2, 1440 views, 8 slices: 1.49
// against 1.81 ms).  0: neither fits.
template <int NB, int M>
int stream_waves(int na, long long workgroups, int pitch, int vchunk)
{
    using S = StreamShape<NB, M>;
    const auto fits = [&](int w, int waves) {  // `waves` waves of w-wave workgroups on a CU
        const int views = div_up(na, w);
        return views <= S::kMaxViews &&
               waves * stream_wave_bytes(S::kIl, NB, pitch, vchunk, views) <= 160 * 1024;
    };
    if (workgroups <= 256 && fits(16, 16)) return 16;
    if (fits(8, 16)) return 8;
    return fits(16, 16) ? 16 : fits(8, 8) ? 8 : 0;
}

// Launch the n slices of L in groups of NB.
template <class Geo, int NB, int M, bool RAW>
int launch_stream(StreamLaunch<Geo> L, const typename Geo::Tables& T, int n, int pitch,
                  hipStream_t st)
{
    using S = StreamShape<NB, M>;
    const auto& P = L.P;
    L.nbatch = n;
    L.tiles_x = div_up(P.nx, kStreamTile);
    L.tiles_y = div_up(P.ny, kStreamTile);
    L.pitch = pitch;
    L.vchunk = stream_vchunk(S::kViews, NB, pitch);
    const int groups = div_up(n, NB);
    const int w = stream_waves<NB, M>(
        P.na, static_cast<long long>(L.tiles_x) * L.tiles_y * groups, pitch, L.vchunk);
    CTR_REQUIRE(w > 0, CTR_ERR_SHAPE, "BP: the views of a tile exceed a workgroup's LDS");
    L.views = div_up(P.na, w);
    L.wave_bytes = stream_wave_bytes(S::kIl, NB, pitch, L.vchunk, L.views);
    const size_t lds = static_cast<size_t>(w) * L.wave_bytes;
    auto kern = bp_stream_kernel<Geo, NB, M, RAW>;
    if (lds > 64 * 1024)
        CTR_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>(lds)));
    hipLaunchKernelGGL(kern, dim3(super_grid(L.tiles_x, L.tiles_y), groups), dim3(64 * w), lds, st,
                       T, L);
    return check_launch("bp_stream_kernel");
}

template <int NB, int M>
bool stream_fits(int na, int pitch)
{
    return stream_waves<NB, M>(na, 1 << 20, pitch,
                               stream_vchunk(StreamShape<NB, M>::kViews, NB, pitch)) > 0;
}

// Whether the spans of 16 x 16 tiles fit (kStreamMaxPitch channels) and a group of
// il interleaved sinograms lies within a 31-bit buffer range: row offsets are 32-bit,
// and the offset of 2^31 of a channel off the detector has to be outside it.
inline bool stream_reaches(int lmax, long long na, long long ns, int il)
{
    return lmax <= kStreamMaxPitch && na * ns * il * 4 < (1LL << 31);
}

// Whether the stream kernels take a batch: groups of four slices in reach, and
// views that groups of up to 4 slices always have room for (8 waves of 192).
inline bool stream_applies(int lmax, long long na, long long ns)
{
    return stream_reaches(lmax, na, ns, 4) && na <= 8 * 2 * kStreamChain;
}

// Whether the stream kernels are the faster for n slices of nx x ny pixels.  A tile's
// 8 or 16 waves have to be worth their sums at the end, and the interleaved copy its
// two passes over the sinogram; the engine kernel has neither (4 waves a tile, no copy),
// and the fewer views, the more both weigh.  It pads a batch to whole groups of `most`
// (16; the FP transpose 8), 8, 4 or 2 slices, and on a small image it leaves the chip
// half empty.  Measured on fan, parallel and FP-transpose calls of 32^2 to 1024^2 with 8
// to 720 views and 1 to 32 slices, engine -> stream in us:
//  * one slice from 56 views on (fan 512^2: 30 views 11 -> 14, 60 views 17 -> 16);
//  * 2 or 3 from 144 (512^2, 2 slices: 90 views 26 -> 30, 180 views 47 -> 41);
//  * 4 or more from 176 on images of up to 256 tiles (256^2, 8 slices: 90 views 24 ->
//    26, 180 views 44 -> 31), on larger ones from 144 for a batch that the engine pads
//    (512^2, 5 slices: 90 views 53 -> 49) and from 208 for one that it does not (512^2,
//    8 slices: 120 views 46 -> 56, 240 views 87 -> 82);
//  * a batch of 16s and a rest is two or three launches here: from 208 views on, 240 on
//    images of up to 512 tiles, 480 for the FP transpose there (24 slices of 320^2, 320
//    views 179 -> 208);
//  * where the anchors of many views keep groups of 16 out of the LDS (spans of 64
//    channels, 1536 views), two groups of 8 take longer than one of the engine's 16
//    (400^2, 16 slices: 879 and 983 us).
inline bool stream_pays(int n, int nx, int ny, int na, int lmax, int most)
{
    const long long tiles = static_cast<long long>(div_up(nx, kStreamTile)) * div_up(ny, kStreamTile);
    const int group = std::min(most, n >= 16 ? 16 : n >= 8 ? 8 : n >= 4 ? 4 : n >= 2 ? 2 : 1);
    int least = n == 1         ? 56
                : n < 4        ? 144
                : tiles <= 256 ? 176
                : n % group    ? 144
                               : 208;
    if (n > 16 && n % 16) least = tiles > 512 ? 208 : most == 8 ? 480 : 240;
    if (na < least) return false;
    const bool sixteens = most == 16 && n >= 16 && (n % 16 == 0 || n % 16 > 8);
    return !sixteens || stream_fits<16, 4>(na, (lmax + 15) / 16 * 16);
}

// A batch of n sinograms proj, in groups of 16, 8, 4 (2, 1) slices.  A group
// costs about 326, 199, 141, 110, 83 us of 512^2 pixels and 720 views, empty
// slices included: 10 to 15 slices are one group of 16 (8 + 4: 340), 5 to 7 one
// of 8 (4 + 1: 224), 3 one of 4.  RAW: nothing is allocated.
template <class Geo, bool RAW = false>
int launch_stream_part(StreamLaunch<Geo> L, const typename Geo::Tables& T, const float* proj,
                        int n, int lmax, hipStream_t st)
{
    const auto& P = L.P;
    const int pitch = (lmax + 15) / 16 * 16;
    const size_t sino = static_cast<size_t>(P.na) * P.ns, image = static_cast<size_t>(P.nx) * P.ny;
    float* img = L.img;
    float* ws = nullptr;
    if (n > 1 && !RAW) {
        const size_t slices = n == 2 ? 2 : div_up(n, 4) * 4;
        const int e = ws_part(reinterpret_cast<void**>(&ws), slices * sino * sizeof(float), st);
        if (e) return e;
        const dim3 grid(div_up(sino, 256), n == 2 ? 1 : div_up(n, 4));
        if (n == 2)
            hipLaunchKernelGGL(interleave_kernel<2>, grid, dim3(256), 0, st, proj, ws,
                               static_cast<unsigned int>(sino), n);
        else
            hipLaunchKernelGGL(interleave_kernel<4>, grid, dim3(256), 0, st, proj, ws,
                               static_cast<unsigned int>(sino), n);
    }
    int rc = check_launch("interleave_kernel");
    for (int b0 = 0; b0 < n && rc == CTR_OK;) {
        const int left = n - b0;
        L.img = img + b0 * image;
        L.src = (RAW || left == 1 ? proj : ws) + b0 * sino;
        int take = left;
        if (left >= 10 && stream_fits<16, 4>(P.na, pitch)) {
            take = left >= 16 ? left / 16 * 16 : left;
            rc = launch_stream<Geo, 16, 4, RAW>(L, T, take, pitch, st);
        } else if (left >= 5 && stream_fits<8, 8>(P.na, pitch)) {
            take = std::min(left, 8);
            rc = launch_stream<Geo, 8, 8, RAW>(L, T, take, pitch, st);
        } else if (left >= 2 && n > 2) {
            take = std::min(left, 4);
            rc = launch_stream<Geo, 4, 8, RAW>(L, T, take, pitch, st);
        } else if (left == 2) {
            rc = launch_stream<Geo, 2, 8, RAW>(L, T, 2, pitch, st);
        } else {
            rc = launch_stream<Geo, 1, 8, RAW>(L, T, 1, pitch, st);
        }
        b0 += take;
    }
    if (ws) CTR_HIP(ctr::ws_free(ws, st));
    return rc;
}

template <class Geo, bool RAW = false>
int launch_stream_batch(StreamLaunch<Geo> L, const typename Geo::Tables& T, const float* proj,
                        int n, int lmax, hipStream_t st)
{
    if constexpr (RAW) return launch_stream_part<Geo, true>(L, T, proj, n, lmax, st);
    const size_t sino = static_cast<size_t>(L.P.na) * L.P.ns;
    const size_t image = static_cast<size_t>(L.P.nx) * L.P.ny;
    float* const img = L.img;
    const auto part = [&](auto raw, int b, int count) {
        L.img = img + b * image;
        return launch_stream_part<Geo, decltype(raw)::value>(L, T, proj + b * sino, count, lmax, st);
    };
    const auto raw = [&](int b, int count) { return part(std::true_type{}, b, count); };
    const size_t bytes = sino * sizeof(float);
    // a captured BP allocates nothing: no memory nodes in the graph
    if (n > 1 && ws_capturing(st)) return in_parts(n, bytes, raw, raw);
    return in_parts(
        n, bytes, [&](int b, int count) { return part(std::false_type{}, b, count); }, raw);
}

}  // namespace ctr
