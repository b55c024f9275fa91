// csrc/readback.cpp over a HIP stub whose device memory is host memory, built and run by
// tests/test_readback_host.py: every size and every failure must leave the caller's buffer complete and its
// surroundings untouched.
#include <dlfcn.h>
#include <pthread.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

#include "readback.h"
#include "scene.h"

namespace {
// Which call fails (-1: none; 0: each; k: the k-th), and what was done.
struct Plan {
    int alloc = -1, event = -1, launch = -1, record = -1, sync = -1, memcpy = -1, thread = -1;
    bool known = false, slow = false;
} plan;
std::atomic<int> events{0}, launches{0}, records{0}, syncs{0}, streams{0};
std::atomic<size_t> staged{0}, direct{0}, pinned{0};
thread_local bool throw_new = false;
std::atomic<bool> arm_new{false};
bool fails(int want, std::atomic<int> &count) { const int k = ++count; return want == 0 || want == k; }
}  // namespace

void *operator new(size_t n) {
    if (throw_new && arm_new) throw std::bad_alloc();
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    if (plan.thread >= 0) return EAGAIN;
    using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    return reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, arg);
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    if (fails(plan.event, events)) return hipErrorOutOfMemory;
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *, unsigned) { ++streams; return hipErrorOutOfMemory; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (plan.alloc >= 0) return hipErrorOutOfMemory;
    pinned += n;
    return (*p = std::aligned_alloc(4096, n)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return fails(plan.record, records) ? hipErrorUnknown : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
    if (plan.slow) std::this_thread::sleep_for(std::chrono::milliseconds(5));
    return fails(plan.sync, syncs) ? hipErrorUnknown : hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) {
    throw_new = arm_new;  // from here on, on the thread that starts the others
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    throw_new = false;
    if (plan.memcpy >= 0) return hipErrorUnknown;
    std::memcpy(d, s, n);
    direct += n;
    return hipSuccess;
}
hipError_t hipMalloc(void **, size_t) { return hipErrorOutOfMemory; }
hipError_t hipFree(void *) { return hipSuccess; }
}
#undef hipPointerGetAttributes
extern "C" hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
    a->type = hipMemoryTypeHost;
    return plan.known ? hipSuccess : hipErrorInvalidValue;
}
namespace vt {
hipError_t launch_copy_out(const void *s, void *d, size_t n, hipStream_t) {
    if (n % 16 || fails(plan.launch, launches)) return hipErrorInvalidValue;
    std::memcpy(d, s, n);
    staged += n;
    return hipSuccess;
}
}  // namespace vt

static void run(const char *what, size_t bytes, int pad = 1) {
    events = launches = records = syncs = streams = 0;
    staged = direct = pinned = 0;
    std::vector<unsigned char> src(bytes), dst(bytes + 64, 0xA5);
    for (size_t i = 0; i < bytes; ++i) src[i] = (unsigned char)((i * 2654435761u) >> 13);
    bool threw = false;
    {
        vt::ReadbackStage stage;
        throw_new = arm_new;
        try {
            stage.copy(0, dst.data() + 32 + pad, src.data(), bytes);
        } catch (const vt::DeviceError &) {
            threw = true;
        }
        throw_new = false;
    }
    bool good = threw == (plan.memcpy >= 0 && direct == 0 && staged < bytes);
    if (!threw) good = good && std::memcmp(dst.data() + 32 + pad, src.data(), bytes) == 0;
    for (int i = 0; i < 32 + pad; ++i) good = good && dst[i] == 0xA5;
    for (size_t i = 32 + pad + bytes; i < dst.size(); ++i) good = good && dst[i] == 0xA5;
    std::printf("%s %zu: %s staged %zu direct %zu pinned %zu streams %d\n", what, bytes, good ? "ok" : "BAD", staged.load(),
                direct.load(), pinned.load(), streams.load());
    if (!good) std::exit(1);
}

int main(int, char **argv) {
    const std::string mode = argv[1];
    const size_t mb = (size_t)1 << 20;
    if (mode == "sizes")
        for (size_t n : {(size_t)0, (size_t)16, 8 * mb - 16, 8 * mb, 8 * mb + 16, 9 * mb + 512 * 1024, 16 * mb - 16, 16 * mb,
                         16 * mb + 16, 17 * mb - 16, 33 * mb + 48})
            run("size", n);
    else if (mode == "known") {
        plan.known = true;
        run("known", 20 * mb);
    } else if (mode == "failures") {
        const size_t n = 20 * mb + 32;
        for (int k : {0, 1, 2, 4}) {
            plan = Plan{}; plan.event = k; run("event", n);
            plan = Plan{}; plan.launch = k; run("launch", n);
            plan = Plan{}; plan.record = k; run("record", n);
            plan = Plan{}; plan.sync = k; run("sync", n);
        }
        plan = Plan{}; plan.alloc = 0; run("alloc", n);
        plan.memcpy = 0; run("alloc and copy", n);
    } else if (mode == "threads") {
        plan.thread = 0;
        run("no threads", 20 * mb);
    } else if (mode == "memory") {
        arm_new = true;
        run("no memory for threads", 20 * mb);
    } else if (mode == "busy") {
        plan.slow = true;
        run("busy", 40 * mb);
    }
    return 0;
}
