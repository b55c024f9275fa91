#include "readback.h"

#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

#include "scene.h"

namespace vt {

ReadbackStage::~ReadbackStage() {
    for (auto &t : done_)
        for (hipEvent_t e : t)
            if (e) (void)hipEventDestroy(e);
    if (ready_) (void)hipEventDestroy(ready_);
    if (stream_) (void)hipStreamDestroy(stream_);
    if (pinned_) (void)hipHostFree(pinned_);
}

// False when something could not be had; what was stays for the next attempt.
bool ReadbackStage::prepare() {
    if (!stream_ && hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking) != hipSuccess) return false;
    if (!ready_ && hipEventCreateWithFlags(&ready_, hipEventDisableTiming) != hipSuccess) return false;
    for (auto &t : done_)
        for (hipEvent_t &e : t)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
    return pinned_ || hipHostMalloc(reinterpret_cast<void **>(&pinned_), kThreads * 2 * kChunk, hipHostMallocDefault) == hipSuccess;
}

bool ReadbackStage::staged(int device, char *dst, const char *src, size_t bytes) {
    if (hipEventRecord(ready_, nullptr) != hipSuccess || hipStreamWaitEvent(stream_, ready_, 0) != hipSuccess) return false;
    const size_t chunks = (bytes + kChunk - 1) / kChunk;
    std::atomic<size_t> next{0};
    std::atomic<bool> ok{true};
    const auto work = [&](int t) {
        char *const buf = pinned_ + (size_t)t * 2 * kChunk;
        const auto size = [&](size_t c) { return c + 1 < chunks ? kChunk : bytes - c * kChunk; };
        const auto start = [&](size_t c, int b) {
            if (hipMemcpyAsync(buf + b * kChunk, src + c * kChunk, size(c), hipMemcpyDeviceToHost, stream_) != hipSuccess ||
                hipEventRecord(done_[t][b], stream_) != hipSuccess)
                ok = false;
        };
        if (hipSetDevice(device) != hipSuccess) ok = false;
        size_t c = ok ? next++ : chunks;
        if (c < chunks) start(c, 0);
        for (int b = 0; c < chunks && ok; b ^= 1) {
            const size_t n = next++;
            if (n < chunks) start(n, b ^ 1);
            if (hipEventSynchronize(done_[t][b]) != hipSuccess) ok = false;
            if (ok) std::memcpy(dst + c * kChunk, buf + b * kChunk, size(c));
            c = n;
        }
    };
    std::thread pool[kThreads];
    for (int t = 1; t < kThreads && (size_t)t < chunks; ++t) {
        try {
            pool[t] = std::thread(work, t);
        } catch (const std::system_error &) {
            break;  // the threads there are draw all chunks
        }
    }
    work(0);
    for (std::thread &t : pool)
        if (t.joinable()) t.join();
    if (!ok) (void)hipStreamSynchronize(stream_);  // nothing is under way to the buffers any more
    return ok;
}

void ReadbackStage::copy(int device, void *dst, const void *src, size_t bytes) {
    if (bytes >= 4 * kChunk) {
        // Pinned and device destinations are copied to directly.
        hipPointerAttribute_t attr{};
        const bool known = hipPointerGetAttributes(&attr, dst) == hipSuccess && attr.type != hipMemoryTypeUnregistered;
        (void)hipGetLastError();  // an address that HIP does not know may be reported as an error
        std::unique_lock<std::mutex> lock(mutex_, std::try_to_lock);
        const bool done = !known && lock.owns_lock() && prepare() &&
                          staged(device, static_cast<char *>(dst), static_cast<const char *>(src), bytes);
        if (done) return;
        (void)hipGetLastError();
    }
    check(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost), "hipMemcpy");
}

}  // namespace vt
