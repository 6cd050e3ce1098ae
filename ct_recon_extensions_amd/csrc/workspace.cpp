// Device memory the operators need only during a call (transposed copies,
// interleaved sinograms, partial sums): stream-ordered allocations from one
// pool per device.
//
// The device's default pool gives everything back whenever a stream is
// synchronised, so a program that waits for each result paid for mapping the
// memory again on every call (about 100 us for the ray-driven FP and its
// transpose, 150 us of the 1.2 ms of a least-squares gradient).  This pool
// keeps up to kKeep bytes that are free, no more, and ctr_release_workspace
// gives those back too.  The pool orders reuse between streams itself and is
// safe to use from several threads.
#include <mutex>
#include <unordered_map>

#include "ctr_common.hpp"

namespace ctr {
namespace {

// 1 GiB: the scratch of the largest sinogram batch of the benchmark (32 x 1440
// x 1472) four times over
constexpr uint64_t kKeep = 1ull << 30;

std::mutex g_mu;
std::unordered_map<int, hipMemPool_t> g_pools;  // device -> pool, for the process's life

hipError_t pool_of_device(hipMemPool_t* out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(g_mu);
    auto it = g_pools.find(dev);
    if (it == g_pools.end()) {
        hipMemPoolProps props{};
        props.allocType = hipMemAllocationTypePinned;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t pool = nullptr;
        e = hipMemPoolCreate(&pool, &props);
        if (e != hipSuccess) return e;
        uint64_t keep = kKeep;
        e = hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
        if (e != hipSuccess) {
            (void)hipMemPoolDestroy(pool);
            return e;
        }
        it = g_pools.emplace(dev, pool).first;
    }
    *out = it->second;
    return hipSuccess;
}

}  // namespace

hipError_t ws_alloc(void** p, size_t bytes, hipStream_t st)
{
    // a captured allocation belongs to the graph, which has a pool of its own
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &status) != hipSuccess) {
        (void)hipGetLastError();
        return hipMallocAsync(p, bytes, st);
    }
    if (status != hipStreamCaptureStatusNone) return hipMallocAsync(p, bytes, st);
    hipMemPool_t pool = nullptr;
    const hipError_t e = pool_of_device(&pool);
    return e == hipSuccess ? hipMallocFromPoolAsync(p, bytes, pool, st) : e;
}

hipError_t ws_free(void* p, hipStream_t st) { return hipFreeAsync(p, st); }

}  // namespace ctr

extern "C" int ctr_release_workspace(void)
{
    using namespace ctr;
    try {
        std::lock_guard<std::mutex> lock(g_mu);
        for (auto& entry : g_pools) CTR_HIP(hipMemPoolTrimTo(entry.second, 0));
        return CTR_OK;
    } catch (...) {
        set_error("ctr_release_workspace: out of memory");
        return CTR_ERR_ALLOC;
    }
}
