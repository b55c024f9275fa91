// readback.h -- copies of whole images from the device to ordinary host memory.
#pragma once
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstddef>
#include <mutex>

namespace vt {

// Copies device memory to a caller's buffer, in the order hipMemcpy on the null stream would: after the work
// before it on blocking streams, complete on return.  src and bytes are multiples of 16.
//
// hipMemcpy to pageable memory stages through one buffer on one thread, where copying out of the staging
// buffer and the page faults of a fresh destination add up.  Here a few threads draw chunks of an image of 8 MB
// and more; for each a kernel writes the chunk to the thread's pinned buffer (50 GB/s, where the copy engine has
// 41) and the thread copies it out.  Milliseconds, hipMemcpy -> here:
//                memory in use   fresh memory   first of a process   first of a later context (in use)
//   9.0 MB       0.53 -> 0.36    2.5 -> 1.5     8.1 -> 0.8           0.53 -> 0.9
//   16.4 MB      0.98 -> 0.57    4.7 -> 2.7     8.6 -> 1.0           0.97 -> 0.9
//   33.2 MB      1.95 -> 0.88    9.3 -> 5.6     9.5 -> 1.6           1.95 -> 1.4
//   132.7 MB     7.8  -> 3.1     36  -> 21      15  -> 3.8           7.8  -> 3.6
// A first copy pays for what it sets up, so little is: no stream of its own (3 ms each for the first few of a
// process), no copy engine (6 ms for the first copy on each, and copies that change engine or stream were at
// times slower than hipMemcpy: 33.2 MB 2.8, 132.7 MB 10.3), and 4 MB of pinned memory (0.1 ms a MB when first
// touched; 32 MB in chunks of 2 MB took 0.85 and 2.8 later, 4.3 and 5.7 at first).  Chunks of 1 MB, below 16 MB
// of 512 KB (0.33 ms for 9.4 MB with either, but half the memory to touch); of 256 KB they take 1.35 ms for
// 33.2 MB.
// Other work on blocking streams may come between the chunks.  A chunk that takes longer than kBusy shows it,
// and hipMemcpy copies the rest in one piece.
class ReadbackStage {
public:
    ~ReadbackStage();
    void copy(int device, void *dst, const void *src, size_t bytes);

private:
    static constexpr int kThreads = 4;
    static constexpr size_t kChunk = (size_t)1 << 20;
    static constexpr size_t kStaged = (size_t)8 << 20;  // from here on (4.5 MB: hipMemcpy is as fast)
    static constexpr size_t kSmall = (size_t)16 << 20;  // half chunks below
    static constexpr std::chrono::milliseconds kBusy{2};
    bool prepare();
    size_t staged(int device, char *dst, const char *src, size_t bytes);
    std::mutex mutex_;  // held by the copy that uses the buffers; another meanwhile takes hipMemcpy
    char *pinned_ = nullptr;  // kThreads x kChunk, allocated by the first large copy
    hipEvent_t done_[kThreads] = {};
};

}  // namespace vt
