// Shared definitions of the MI355X CT library: the geometry record, error
// plumbing for the C ABI, and small device helpers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <string>

#include "include/ctr_api.h"

namespace ctr {

// Last-error string of the calling thread (the C ABI never throws).
void set_error(const std::string& msg);
const char* get_error();

#define CTR_HIP(expr)                                                              \
    do {                                                                           \
        hipError_t e_ = (expr);                                                    \
        if (e_ != hipSuccess) {                                                    \
            ::ctr::set_error(std::string(#expr) + ": " + hipGetErrorString(e_));   \
            return CTR_ERR_HIP;                                                    \
        }                                                                          \
    } while (0)

#define CTR_REQUIRE(cond, code, msg)                                               \
    do {                                                                           \
        if (!(cond)) {                                                             \
            ::ctr::set_error(msg);                                                 \
            return (code);                                                         \
        }                                                                          \
    } while (0)

// Launches report asynchronous configuration errors through this check.
inline int check_launch(const char* what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string(what) + ": " + hipGetErrorString(e));
        return CTR_ERR_HIP;
    }
    return CTR_OK;
}

inline int div_up(long long a, long long b) { return static_cast<int>((a + b - 1) / b); }

// Centres of the pixel grid and of the detector, as every reference routine
// defines them (e.g. src/bp_fan_2d.cc:22-25, :56-57).
inline double cent_x(const ctr_geom& g) { return static_cast<double>(g.nx - 1) / 2 + g.offset_x; }
inline double cent_y(const ctr_geom& g) { return static_cast<double>(g.ny - 1) / 2 + g.offset_y; }
inline double cent_s(const ctr_geom& g) { return static_cast<double>(g.ns - 1) / 2 + g.offset_s; }

// Device memory for the duration of a call, ordered on `st` (workspace.cpp).
hipError_t ws_alloc(void** p, size_t bytes, hipStream_t st);
hipError_t ws_free(void* p, hipStream_t st);
// Whether st is being captured: scratch is then a memory node of the graph.
bool ws_capturing(hipStream_t st);

// A batch in parts whose scratch (bytes a slice) stays within 1 GiB, at least 16
// slices each: call(first, count).  A part whose scratch the device has no room for
// (ws_part: kNoScratch) is small(first, count)'s, which gets by with less and gives the
// same bits: what is free on the device does not show in a result.
constexpr int kNoScratch = -1;

inline int ws_part(void** p, size_t bytes, hipStream_t st)
{
    const hipError_t e = ws_alloc(p, bytes, st);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        return kNoScratch;
    }
    CTR_HIP(e);
    return 0;
}

template <typename F, typename G>
int in_parts(int n, size_t bytes, F&& call, G&& small)
{
    const size_t fit = (size_t{1} << 30) / bytes / 16 * 16;
    const int part = static_cast<int>(fit < 16 ? 16 : fit < static_cast<size_t>(n) ? fit : n);
    int rc = 0;
    for (int b = 0; b < n && rc == 0; b += part) {
        const int count = n - b < part ? n - b : part;
        rc = call(b, count);
        if (rc == kNoScratch) rc = small(b, count);
    }
    if (rc != kNoScratch) return rc;
    set_error("out of device memory");
    return CTR_ERR_HIP;
}

// small() of operators that take the slices of a part one at a time.
template <typename F>
int one_by_one(int first, int count, F&& call)
{
    int rc = 0;
    for (int i = 0; i < count && rc == 0; ++i) rc = call(first + i);
    return rc;
}

// Scale of bp_fan_2d: |orbit| / round(|na*orbit|/pi) (src/bp_fan_2d.cc:58,83).
double fan_bp_scale(const ctr_geom& g);

}  // namespace ctr
