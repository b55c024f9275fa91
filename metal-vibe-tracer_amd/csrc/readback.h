// readback.h -- copies of whole images from the device to ordinary host memory.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace vt {

// Copies device memory to a caller's buffer, in the order hipMemcpy on the null stream would: after the work
// before it on blocking streams, complete on return.
//
// hipMemcpy to pageable memory stages through one buffer on one thread, where copying out of the staging
// buffer and the page faults of a fresh destination add up.  Here a few threads draw chunks of the image; each
// has two pinned buffers, so its next chunk is on the bus while it copies the last one out, and the threads
// take page faults side by side.  Images of four chunks and more go this way (milliseconds, hipMemcpy -> here):
//                 memory in use    fresh memory
//   8.3 MB        0.46 -> 0.37     1.14 -> 0.66
//   14.7 MB       0.86 -> 0.53     1.85 -> 1.09
//   33.2 MB       1.84 -> 0.94     3.69 -> 1.41
//   132.7 MB      7.6  -> 3.4      14.3 -> 4.0
// At half of that the threads cost what they save (4.5 MB to memory in use: 0.26 -> 0.23 to 0.28).  Chunks of 1 MB take 1.14 ms where 2 MB take 0.94
// (an event wait each), six threads on 0.5 MB 1.6.
class ReadbackStage {
public:
    ~ReadbackStage();
    void copy(int device, void *dst, const void *src, size_t bytes);

private:
    static constexpr int kThreads = 4;
    static constexpr size_t kChunk = (size_t)2 << 20;
    bool prepare();
    bool staged(int device, char *dst, const char *src, size_t bytes);
    std::mutex mutex_;  // held by the copy that uses the buffers; another meanwhile takes hipMemcpy
    char *pinned_ = nullptr;  // kThreads x 2 x kChunk, allocated by the first large copy
    hipStream_t stream_ = nullptr;
    hipEvent_t ready_ = nullptr, done_[kThreads][2] = {};
};

}  // namespace vt
