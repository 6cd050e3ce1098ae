// Device memory the operators need only during a call (transposed copies,
// interleaved sinograms, partial sums).
//
// A stream-ordered allocation and its release cost the host 15 to 25 us a call
// once kernels lie between the two, as much as the rest of a small operator,
// and the default pool maps the memory anew after every synchronisation (about
// 100 us).  So freed blocks are kept, per device, with an event recorded where
// their last use ends: a call on the same stream takes one at once (the wait
// for the event is then satisfied by the stream's order), a call on another
// stream only a block whose event has passed.  At most kKeep bytes and
// kBlocks blocks are kept free, the oldest go first, and ctr_release_workspace
// gives them all back to the device (an allocator beside this one, PyTorch's for
// one, cannot ask for them).  Any number of threads and streams: a block belongs to
// one call from ws_alloc to ws_free.
#include <cstdint>
#include <deque>
#include <exception>
#include <mutex>
#include <unordered_map>

#include "ctr_common.hpp"

namespace ctr {
namespace {

// 1 GiB: the scratch of the largest sinogram batch of the benchmark (32 x 1440
// x 1472: 259 MiB, a block of 320) three times over
constexpr size_t kKeep = size_t{1} << 30, kBlocks = 64;

struct Block {
    void* p;
    size_t bytes;
    hipEvent_t done;  // recorded after the last use
    hipStream_t st;   // stream of the last use
};

struct Device {
    std::deque<Block> free;  // oldest first
    size_t free_bytes = 0;
};

std::mutex g_mu;
std::unordered_map<int, Device> g_devices;
std::unordered_map<void*, Block> g_used;  // blocks a call holds

// Blocks come in sizes of 1/4 octave, so that calls of similar sizes share them.
size_t block_size(size_t bytes)
{
    size_t step = size_t{1} << 16;
    while (step * 8 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

// Another thread may be capturing a graph, which (in the global mode, PyTorch's
// default) calls like hipEventQuery and hipMallocAsync from any thread would
// invalidate; none of those made here touches a captured stream.  Waiting for an
// event and recording one need no such cover, so a call that finds its own stream's
// block pays nothing for it.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

hipError_t event_passed(hipEvent_t e)
{
    const RelaxedCapture relaxed;
    return hipEventQuery(e);
}

}  // namespace

bool ws_capturing(hipStream_t st)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &status) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return status != hipStreamCaptureStatusNone;
}

hipError_t ws_alloc(void** p, size_t bytes, hipStream_t st)
{
    // a captured allocation belongs to the graph, which has memory of its own (the
    // forward BPs make none: bp_stream.hpp)
    if (ws_capturing(st)) return hipMallocAsync(p, bytes, st);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const size_t want = block_size(bytes);
    try {
        std::lock_guard<std::mutex> lock(g_mu);
        Device& D = g_devices[dev];
        // newest first: its lines may still be in the caches
        for (size_t i = D.free.size(); i-- > 0;) {
            Block b = D.free[i];
            if (b.bytes < bytes || b.bytes > 2 * want) continue;
            if (b.st != st && event_passed(b.done) != hipSuccess) {
                (void)hipGetLastError();  // not ready
                continue;
            }
            // (a destroyed stream's handle may name a new stream: hence the wait)
            e = hipStreamWaitEvent(st, b.done, 0);
            if (e != hipSuccess) return e;
            g_used.emplace(b.p, b);
            D.free.erase(D.free.begin() + static_cast<std::ptrdiff_t>(i));
            D.free_bytes -= b.bytes;
            *p = b.p;
            return hipSuccess;
        }
        const RelaxedCapture relaxed;
        Block b{nullptr, want, nullptr, st};
        e = hipEventCreateWithFlags(&b.done, hipEventDisableTiming);
        if (e != hipSuccess) return e;
        e = hipMallocAsync(&b.p, want, st);
        if (e == hipErrorOutOfMemory && !D.free.empty()) {  // the kept blocks make room
            (void)hipGetLastError();
            for (const Block& old : D.free) {
                if (hipStreamWaitEvent(st, old.done, 0) == hipSuccess) (void)hipFreeAsync(old.p, st);
                (void)hipEventDestroy(old.done);
            }
            D.free.clear();
            D.free_bytes = 0;
            e = hipMallocAsync(&b.p, want, st);
        }
        if (e == hipSuccess) {
            g_used.emplace(b.p, b);
            *p = b.p;
        } else {
            (void)hipEventDestroy(b.done);
        }
        return e;
    } catch (const std::exception&) {
        return hipErrorOutOfMemory;
    }
}

hipError_t ws_free(void* p, hipStream_t st)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    try {
        std::lock_guard<std::mutex> lock(g_mu);
        const auto it = g_used.find(p);
        if (it == g_used.end()) return hipFreeAsync(p, st);  // a captured allocation
        Block b = it->second;
        g_used.erase(it);
        b.st = st;
        e = hipEventRecord(b.done, st);
        if (e != hipSuccess) {
            const RelaxedCapture relaxed;
            (void)hipEventDestroy(b.done);
            const hipError_t f = hipFreeAsync(p, st);
            return f != hipSuccess ? f : e;
        }
        Device& D = g_devices[dev];
        D.free.push_back(b);
        D.free_bytes += b.bytes;
        while (D.free_bytes > kKeep || D.free.size() > kBlocks) {
            const RelaxedCapture relaxed;
            const Block old = D.free.front();
            D.free.pop_front();
            D.free_bytes -= old.bytes;
            e = hipStreamWaitEvent(st, old.done, 0);
            if (e == hipSuccess) e = hipFreeAsync(old.p, st);
            (void)hipEventDestroy(old.done);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    } catch (const std::exception&) {
        return hipErrorOutOfMemory;
    }
}

}  // namespace ctr

extern "C" int ctr_release_workspace(void)
{
    using namespace ctr;
    try {
        std::lock_guard<std::mutex> lock(g_mu);
        int dev = 0;
        CTR_HIP(hipGetDevice(&dev));
        const RelaxedCapture relaxed;
        Device& D = g_devices[dev];
        while (!D.free.empty()) {
            const Block b = D.free.back();
            D.free.pop_back();
            D.free_bytes -= b.bytes;
            CTR_HIP(hipEventSynchronize(b.done));
            (void)hipEventDestroy(b.done);
            CTR_HIP(hipFree(b.p));
        }
        // the pool behind hipMallocAsync would hold on to them until the next
        // synchronisation
        hipMemPool_t pool = nullptr;
        CTR_HIP(hipDeviceGetDefaultMemPool(&pool, dev));
        CTR_HIP(hipMemPoolTrimTo(pool, 0));
        return CTR_OK;
    } catch (const std::exception& e) {
        set_error(std::string("ctr_release_workspace: ") + e.what());
        return CTR_ERR_ALLOC;
    }
}
