#include "readback.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <exception>
#include <thread>

#include "scene.h"

namespace vt {

ReadbackStage::~ReadbackStage() {
    for (hipEvent_t e : done_)
        if (e) (void)hipEventDestroy(e);
    if (pinned_) (void)hipHostFree(pinned_);
}

// False when something could not be had; what was stays for the next attempt.
bool ReadbackStage::prepare() {
    for (hipEvent_t &e : done_)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
    return pinned_ || hipHostMalloc(reinterpret_cast<void **>(&pinned_), kThreads * kChunk, hipHostMallocDefault) == hipSuccess;
}

// The bytes copied from the front.
size_t ReadbackStage::staged(int device, char *dst, const char *src, size_t bytes) {
    using Clock = std::chrono::steady_clock;
    const size_t chunk = bytes < kSmall ? kChunk / 2 : kChunk, chunks = (bytes + chunk - 1) / chunk;
    std::atomic<size_t> next{0};
    std::atomic<bool> ok{true}, busy{false};
    const auto work = [&](int t) {
        char *const buf = pinned_ + (size_t)t * kChunk;
        if (hipSetDevice(device) != hipSuccess) ok = false;
        while (ok && !busy) {
            const size_t c = next++;
            if (c >= chunks) return;
            const size_t at = c * chunk, n = std::min(chunk, bytes - at);
            const Clock::time_point start = Clock::now();
            if (launch_copy_out(src + at, buf, n, nullptr) != hipSuccess || hipEventRecord(done_[t], nullptr) != hipSuccess ||
                hipEventSynchronize(done_[t]) != hipSuccess) {
                ok = false;
                return;
            }
            if (Clock::now() - start > kBusy) busy = true;
            std::memcpy(dst + at, buf, n);
        }
    };
    std::thread pool[kThreads];
    for (int t = 1; t < kThreads && (size_t)t < chunks; ++t) {
        try {
            pool[t] = std::thread(work, t);
        } catch (const std::exception &) {
            break;  // the threads there are draw all chunks
        }
    }
    work(0);
    for (std::thread &t : pool)
        if (t.joinable()) t.join();
    if (ok) return std::min(bytes, next * chunk);
    (void)hipStreamSynchronize(nullptr);  // nothing is under way to the buffers any more
    return 0;
}

void ReadbackStage::copy(int device, void *dst, const void *src, size_t bytes) {
    size_t done = 0;
    if (bytes >= kStaged) {
        // Pinned and device destinations are copied to directly.
        hipPointerAttribute_t attr{};
        const bool known = hipPointerGetAttributes(&attr, dst) == hipSuccess && attr.type != hipMemoryTypeUnregistered;
        (void)hipGetLastError();  // an address that HIP does not know may be reported as an error
        std::unique_lock<std::mutex> lock(mutex_, std::try_to_lock);
        if (!known && lock.owns_lock() && prepare())
            done = staged(device, static_cast<char *>(dst), static_cast<const char *>(src), bytes);
        if (done == bytes) return;
        (void)hipGetLastError();
    }
    check(hipMemcpy(static_cast<char *>(dst) + done, static_cast<const char *>(src) + done, bytes - done, hipMemcpyDeviceToHost),
          "hipMemcpy");
}

}  // namespace vt
