// trace.hip -- gfx950 closest-hit and any-hit traversal kernels over SoA ray buffers.
//
// Persistent grids: a ray belongs to one lane of a 64-lane wavefront, which takes the next ray when its own
// ends; the wave tests its lanes' triangles together.  Ray components are separate arrays, read a batch of 64
// consecutive rays at a time.  The per-ray traversal (traverse8.h) keeps its node-group stack in LDS, laid
// out [depth][lane] so every lane's push/pop touches its own bank.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "resolve.h"
#include "trace_kernels.h"
#include "traverse8.h"

namespace vt {
namespace {

constexpr int kBlock = 128;
constexpr int kRefillIdle = 12;

// A tree of depth D leaves at most D - 1 node groups pending; the launcher picks the smallest
// instantiated depth that covers the scene's tree (the builder bounds it by 24), so LDS per block,
// and with it the number of resident waves, follows the tree actually traced.
template <int kStack, int kBlk = kBlock>
struct LdsStack {
    uint32_t (*base)[kBlk];
    uint16_t (*bits)[kBlk];  // imask << 8 | slots still to visit
    int lane;
    int sp;
    int cap;  // groups the stack may hold: kStack, or less under TraceScene::stack_cap
    int floor = 0;  // groups below belong to an outer hierarchy
    __device__ __forceinline__ void push(uint32_t b, uint32_t m) {
        base[sp][lane] = b;
        bits[sp][lane] = (uint16_t)m;
        ++sp;
    }
    __device__ __forceinline__ bool full() const { return sp >= cap; }
    __device__ __forceinline__ void pop(uint32_t &b, uint32_t &m) {
        --sp;
        b = base[sp][lane];
        m = bits[sp][lane];
    }
    __device__ __forceinline__ bool empty() const { return sp == floor; }
};

// The counting traversal (node and triangle records a launch fetches): one ray per lane, one-lane triangle tests.
template <bool ANY, int kStack>
__global__ __launch_bounds__(kBlock) void count_kernel(const U4 *__restrict__ nodes, const F4 *__restrict__ tris,
                                                       RayArgs rays, HitArgs hits, uint8_t *__restrict__ occluded,
                                                       uint32_t n, const uint32_t *__restrict__ count,
                                                       float root_max, unsigned long long *__restrict__ counters,
                                                       uint32_t *__restrict__ fault, int cap) {
    __shared__ uint32_t stack_base[kStack][kBlock];
    __shared__ uint16_t stack_bits[kStack][kBlock];
    const int lane = threadIdx.x;
    const uint32_t i = blockIdx.x * kBlock + lane;
    if (count) n = min(n, *count);
    if (i >= n) return;
    TraceRay r{rays.ox[i], rays.oy[i], rays.oz[i], rays.dx[i], rays.dy[i], rays.dz[i], rays.tmin[i], rays.tmax[i]};
    LdsStack<kStack> st{stack_base, stack_bits, lane, 0, cap};
    TraceResult res = traverse<ANY, true>(nodes, tris, root_max, box_scale(root_max), r, st);
    if (res.overflow && fault) atomicOr(fault, 1u);
    if (ANY) {
        occluded[i] = res.occluded ? 1 : 0;
    } else {
        hits.t[i] = res.t;
        hits.b1[i] = res.b1;
        hits.b2[i] = res.b2;
        hits.face[i] = res.face;
        if (hits.instance) hits.instance[i] = 0u;
    }
    unsigned long long *c = counters + 2 * (blockIdx.x & 63u);
    atomicAdd(c, (unsigned long long)res.nodes);
    atomicAdd(c + 1, (unsigned long long)res.tris);
}

// Persistent traversal with lane refill.  The grid is sized to what the chip holds at once; the waves of a
// block draw batches of 64 ray indices, the block's share of the rays, from an LDS counter,
// and a lane whose ray finishes takes the next index at once, so a wave no longer idles until its
// slowest ray ends.  Node visits are per lane (trav_nodes); the triangles the wave's lanes reach in a
// step are tested by the whole wave together (wave_triangles).  Per ray the arithmetic, the nodes
// visited and the result are exactly a ray's alone (trav_step).
// Source: where a ray's scene comes from -- one scene for the launch (OneScene) or the ray's job
// (JobScenes, batched rendering).  kScaled: for hierarchies whose box scale (traverse8.h) is not 1; theirs is
// a kernel of its own, since the two multiplications a node visit takes for it cost 6 % on shadow rays.
template <bool kScaled>
struct OneScene {
    static constexpr bool kShared = true;  // every lane reads the same triangle array
    const U4 *nodes;
    const F4 *tris;
    float root_max;
    uint32_t *fault;
    int cap;
    struct Lane {};
    __device__ __forceinline__ bool begin(uint32_t, Lane &) const { return true; }
    __device__ __forceinline__ const U4 *node_ptr(const Lane &) const { return nodes; }
    __device__ __forceinline__ const F4 *tri_ptr(const Lane &) const { return tris; }
    __device__ __forceinline__ float root(const Lane &) const { return root_max; }
    __device__ __forceinline__ float scale(const Lane &) const { return kScaled ? box_scale(root_max) : 1.0f; }
    __device__ __forceinline__ uint32_t *fault_word(const Lane &) const { return fault; }
    __device__ __forceinline__ int stack_cap(const Lane &, int k) const { return cap < k ? cap : k; }
};
template <bool kScaled>
struct JobScenes {
    static constexpr bool kShared = false;
    const TraceScene *job_trace;
    const uint32_t *job;
    struct Lane {
        const U4 *nodes;
        const F4 *tris;
        float root_max;
        uint32_t *fault;
        uint32_t cap;
    };
    // False for a scene without geometry (the ray misses).
    __device__ __forceinline__ bool begin(uint32_t ray, Lane &l) const {
        const TraceScene &ts = job_trace[job[ray]];
        l.nodes = reinterpret_cast<const U4 *>(ts.nodes);
        l.tris = reinterpret_cast<const F4 *>(ts.tris);
        l.root_max = ts.root_max;
        l.fault = ts.fault;
        l.cap = ts.stack_cap;
        return ts.node_count != 0;
    }
    __device__ __forceinline__ const U4 *node_ptr(const Lane &l) const { return l.nodes; }
    __device__ __forceinline__ const F4 *tri_ptr(const Lane &l) const { return l.tris; }
    __device__ __forceinline__ float root(const Lane &l) const { return l.root_max; }
    __device__ __forceinline__ float scale(const Lane &l) const { return kScaled ? box_scale(l.root_max) : 1.0f; }
    __device__ __forceinline__ uint32_t *fault_word(const Lane &l) const { return l.fault; }
    __device__ __forceinline__ int stack_cap(const Lane &l, int k) const {
        return l.cap && (int)l.cap < k ? (int)l.cap : k;
    }
};

// Order-preserving map of a float's bits to an unsigned integer.  -0 maps with +0, since the closest-hit
// rule compares t numerically (a hit at t = -0 ties with one at +0 and the smaller face wins).
__device__ __forceinline__ uint32_t ord_bits(float f) {
    const uint32_t u = __float_as_uint(f == 0.0f ? 0.0f : f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
// Position of the k-th set bit (from 0) of m, for k < popcount(m) and m below 2^31.
__device__ __forceinline__ uint32_t nth_set_bit(uint32_t m, uint32_t k) {
    uint32_t pos = 0;
#pragma unroll
    for (uint32_t w = 16; w; w >>= 1) {
        const uint32_t low = __popc(m & ((1u << w) - 1u));
        const bool up = k >= low;
        k = up ? k - low : k;
        m = up ? m >> w : m;
        pos = up ? pos + w : pos;
    }
    return pos;
}
// Orders the wave's LDS accesses on either side (no instruction: a wave's LDS operations complete in
// issue order; this only keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Triangle half of a step for a whole wave.  After its node visit each lane holds up to 24 triangles
// (trimask over tri_base); tested one lane at a time the wave would loop as often as its fullest lane
// (5.6 times per step on incoherent bounce rays with 0.44 x 64 tests to do).  Here the wave's tests are
// numbered by a prefix sum over the lanes' counts and handed out 64 at a time: test j belongs to the
// lane whose range holds j (binary search over the prefixes) and is its k-th triangle; the worker reads
// that lane's ray through cross-lane permutes, runs the same Woop test, and folds a hit into the
// owner's LDS slot with an atomic minimum of (order-preserving t bits << 32 | face + 1) -- the nearest t,
// equal t going to the smaller face, as the one-lane rule.  The winner of each round stores its t and
// barycentrics; the key's identity picks it since a face is tested at most once per ray.  They stay in the
// owner's LDS slot until its ray ends, as do its triangle-test constants (woop, packed by pack_woop): both
// are read only around triangle tests, and the registers are worth a wave per SIMD.  Any-hit queries only
// raise the owner's flag.  Must be called by all 64 lanes together.
// Exclusive prefix over the wave of per-lane counts below 32 (pre) and their sum (total): one ballot per
// bit of the count.
__device__ __forceinline__ void wave_prefix(uint32_t cnt, unsigned long long below, uint32_t &pre, uint32_t &total) {
    pre = 0;
    total = 0;
#pragma unroll
    for (int b = 0; b < 5; ++b) {
        const unsigned long long m = __ballot((cnt >> b) & 1u);
        pre += (uint32_t)__popcll(m & below) << b;
        total += (uint32_t)__popcll(m) << b;
    }
}

__device__ __forceinline__ F4 pack_woop(const WoopRay &w) {
    return F4{w.sx, w.sy, w.sz, bits_to_float((uint32_t)(w.kx | (w.ky << 2) | (w.kz << 4)))};
}

template <bool ANY, int kBlk, class Source>
__device__ __forceinline__ void wave_triangles(const Source &src, const typename Source::Lane &sl, TravState &ts,
                                               uint32_t trimask, uint32_t tri_base, uint32_t tri_bits, uint32_t lane, uint32_t pre,
                                               uint32_t total, const F4 *woop, unsigned long long *key, float (*hit_tb)[kBlk]) {
    const uint32_t cnt = __popc(trimask);
    if (total == 0u) return;
    const uint32_t wave0 = threadIdx.x & ~63u;
    unsigned long long key0 = 0ull;
    if (cnt) {
        // The low word is face + 1: no hit yet counts as 0, below every face, so that a hit at exactly tmax
        // is not nearer and no test's key equals the starting one.
        if (!ANY) key0 = ((unsigned long long)ord_bits(ts.res.t) << 32) | ((uint32_t)ts.res.face + 1u);
        key[threadIdx.x] = key0;
    }
    wave_lds_order();
    const uint64_t tri_addr = reinterpret_cast<uint64_t>(src.tri_ptr(sl));
    for (uint32_t j0 = 0; j0 < total; j0 += 64u) {
        const uint32_t j = j0 + lane;
        uint32_t owner = 0;
#pragma unroll
        for (uint32_t step = 32; step; step >>= 1) {
            const uint32_t cand = owner + step;  // at most 63
            if ((uint32_t)__shfl((int)pre, (int)cand) <= j) owner = cand;
        }
        const int o = (int)owner;
        const uint32_t k = j - (uint32_t)__shfl((int)pre, o);
        const uint32_t omask = (uint32_t)__shfl((int)trimask, o), obase = (uint32_t)__shfl((int)tri_base, o);
        const uint32_t obits = (uint32_t)__shfl((int)tri_bits, o);
        const F4 wo = woop[wave0 + owner];
        const uint32_t kp = float_to_bits(wo.w);
        WoopRay w;
        w.kx = (int)(kp & 3u);
        w.ky = (int)((kp >> 2) & 3u);
        w.kz = (int)(kp >> 4);
        w.sx = wo.x;
        w.sy = wo.y;
        w.sz = wo.z;
        const float ox = __shfl(ts.ox, o), oy = __shfl(ts.oy, o), oz = __shfl(ts.oz, o);
        const float tmin = __shfl(ts.tmin, o);
        const float tmax = ANY ? __shfl(ts.res.t, o) : 0.0f;
        const F4 *tris;
        if constexpr (Source::kShared) {
            tris = src.tri_ptr(sl);
        } else {
            const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)tri_addr, o);
            const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(tri_addr >> 32), o);
            tris = reinterpret_cast<const F4 *>(((uint64_t)hi << 32) | lo);
        }
        bool hit = false;
        unsigned long long mine = 0ull;
        float t = 0.0f, b1 = 0.0f, b2 = 0.0f;
        if (j < total) {
            const F4 *tp = tris + 3 * (size_t)(obase + tri_rank(obits, nth_set_bit(omask, k)));
            const F4 p0 = tp[0], p1 = tp[1], p2 = tp[2];
            if (woop_triangle(w, ox, oy, oz, p0, p1, p2, t, b1, b2) && t >= tmin && (!ANY || t < tmax)) {
                hit = true;
                if (ANY) {
                    key[wave0 + owner] = 1ull;
                } else {
                    mine = ((unsigned long long)ord_bits(t) << 32) | (float_to_bits(p0.w) + 1u);
                    atomicMin(&key[wave0 + owner], mine);
                }
            }
        }
        if (!ANY) {
            wave_lds_order();
            if (hit && key[wave0 + owner] == mine) {
                hit_tb[0][wave0 + owner] = t;
                hit_tb[1][wave0 + owner] = b1;
                hit_tb[2][wave0 + owner] = b2;
            }
        }
        wave_lds_order();
    }
    if (cnt) {
        const unsigned long long got = key[threadIdx.x];
        if (ANY) {
            if (got) ts.res.occluded = true;
        } else if (got != key0) {
            ts.res.t = hit_tb[0][threadIdx.x];
            ts.res.face = (int32_t)((uint32_t)got - 1u);
        }
    }
    wave_lds_order();
}

// LDS of a block of the persistent kernels, kHits: with room for closest hits.  Each lane's part is its
// own wave's, but for `next`: the batches drawn so far from the block's share of each of two queues.
template <int kStack, int kBlk, bool kHits>
struct RefillLds {
    uint32_t stack_base[kStack][kBlk];
    uint16_t stack_bits[kStack][kBlk];
    unsigned long long tri_key[kBlk];
    float tri_hit[kHits ? 3 : 1][kBlk];
    F4 woop[kBlk];
    uint32_t next[2];
};
// The rays are dealt out in units of a few batches of 64, a unit to each block in turn, so cheap and dear
// regions of an image are spread over the blocks (against one contiguous range per block: 10 M terrain
// bounce rays 681 -> 640 us, field shadow rays 213 -> 189 us) and a launch of few rays over the CUs.
// (Renumbering the blocks so that each XCD's share is contiguous lost it all again: the XCDs' shares
// are uneven, and their L2s hold the same upper tree anyway.)
// Each round of units starts at another block (golden-ratio steps): in an image whose width is a multiple of
// the unit a block would otherwise stay in one column, and the columns' costs differ (2048 x 1024 camera rays:
// field 228 -> 178 us, 1024 instances 404 -> 246; 1920 x 1080 unchanged).  Units of a batch per wave take 181
// and 258 us there and 490 against 465 on the terrain's camera rays, units of one batch 162, 260 and 487.
struct Deal {
    uint32_t batches, shift;  // unit = 1 << shift: half the block's waves, fewer when the rays are few
    __device__ __forceinline__ Deal(uint32_t n, uint32_t waves) : batches(n / 64u + (n % 64u != 0u)), shift(0) {
        while ((4u << shift) <= waves && (2u << shift) <= batches / gridDim.x) ++shift;
    }
    // The block's draw-th batch; none from `batches` on.
    __device__ __forceinline__ uint32_t batch(uint32_t draw) const {
        const uint32_t round = draw >> shift, at = blockIdx.x + __umulhi(round * 0x9e3779b9u, gridDim.x);
        const uint32_t unit = round * gridDim.x + (at < gridDim.x ? at : at - gridDim.x);
        return (unit << shift) + (draw & ((1u << shift) - 1u));
    }
};

// Traces the block's share of n rays; `next` is zero when the block's first wave gets here.
template <bool ANY, int kStack, int kBlk, class Source, class Lds>
__device__ __forceinline__ void refill_trace(const Source &src, const RayArgs &rays, const HitArgs &hits,
                                             uint8_t *__restrict__ occluded, uint32_t n, Lds &lds, uint32_t &next) {
    constexpr uint32_t kNone = 0xffffffffu;
    const Deal deal(n, kBlk / 64);
    const uint32_t lane = threadIdx.x & 63u;
    const unsigned long long below = (1ull << lane) - 1ull;
    LdsStack<kStack, kBlk> st{lds.stack_base, lds.stack_bits, (int)threadIdx.x, 0, kStack};
    TravState ts;
    typename Source::Lane sl{};
    uint32_t ray = kNone;
    // The lane's pending triangles (from its last node visit, not yet tested) and whether its ray has
    // no node left to visit.
    uint32_t trimask = 0, tri_base = 0, tri_bits = 0;
    bool done = false;
    // Wave-uniform: the wave's current batch of 64 indices and how many of them are handed out.
    uint32_t batch = 0, used = 64;
    bool exhausted = false;
    for (;;) {
        const unsigned long long need = __ballot(ray == kNone);
        // Refilling costs the whole wave the ray set-up (loads, Woop constants, reciprocals), so idle
        // lanes wait until kRefillIdle of them can be served together (a CPU replay of the benchmark
        // rays put the best trade-off between 8 and 12; measured: bounce rays 4% faster).
        if (!exhausted && __popcll(need) >= kRefillIdle) {
            const uint32_t cnt = (uint32_t)__popcll(need), rank = (uint32_t)__popcll(need & below);
            const uint32_t avail = 64u - used;
            uint32_t idx = batch + used + rank;
            if (cnt > avail) {
                uint32_t draw = 0;
                if (lane == 0) draw = atomicAdd(&next, 1u);
                draw = __builtin_amdgcn_readfirstlane(draw);
                const uint32_t at = deal.batch(draw);
                exhausted = at >= deal.batches;
                const uint32_t fresh = exhausted ? n : at * 64u;
                if (rank >= avail) idx = fresh + (rank - avail);
                batch = fresh;
                used = cnt - avail;
            } else {
                used += cnt;
            }
            if (ray == kNone && idx < n) {
                const TraceRay r{rays.ox[idx], rays.oy[idx], rays.oz[idx], rays.dx[idx], rays.dy[idx], rays.dz[idx],
                                 rays.tmin[idx], rays.tmax[idx]};
                if (src.begin(idx, sl)) {
                    ray = idx;
                    trav_init(ts, r, src.root(sl), src.scale(sl));
                    lds.woop[threadIdx.x] = pack_woop(woop_ray(r.dx, r.dy, r.dz));
                    st.sp = 0;
                    st.cap = src.stack_cap(sl, kStack);
                    done = !(r.tmax == r.tmax);  // nothing is nearer than a NaN
                } else if (ANY) {
                    occluded[idx] = 0;
                } else {
                    hits.t[idx] = r.tmax;
                    hits.b1[idx] = 0.0f;
                    hits.b2[idx] = 0.0f;
                    hits.face[idx] = -1;
                    if (hits.instance) hits.instance[idx] = 0u;
                }
            }
        }
        const bool busy = ray != kNone;
        const unsigned long long live = __ballot(busy);
        if (!live && exhausted) break;
        // A lane holding untested triangles waits (its next node visit needs the hits they may give),
        // so triangles of several steps are tested together: the wave flushes once a quarter of its
        // live lanes wait (a CPU replay of the benchmark rays: 0.97 -> 0.62 rounds per step on bounce
        // rays, about 11% fewer issue cycles).  Nodes visited and results are unchanged.
        if (busy && !done && trimask == 0u) done = trav_nodes<false>(ts, src.node_ptr(sl), src.scale(sl), st, trimask, tri_base, tri_bits);
        const unsigned long long waiting = __ballot(busy && (done || trimask != 0u));
        if (4u * (uint32_t)__popcll(waiting) >= (uint32_t)__popcll(live)) {
            uint32_t pre, total;
            wave_prefix(__popc(trimask), below, pre, total);
            wave_triangles<ANY, kBlk>(src, sl, ts, trimask, tri_base, tri_bits, lane, pre, total, lds.woop, lds.tri_key, lds.tri_hit);
            trimask = 0u;
        }
        if (busy && ((done && trimask == 0u) || (ANY && ts.res.occluded))) {
            if (ts.res.overflow) {
                uint32_t *f = src.fault_word(sl);
                if (f) atomicOr(f, 1u);
            }
            if (ANY) {
                occluded[ray] = ts.res.occluded ? 1 : 0;
            } else {
                const bool hit = ts.res.face >= 0;
                hits.t[ray] = ts.res.t;
                hits.b1[ray] = hit ? lds.tri_hit[1][threadIdx.x] : 0.0f;
                hits.b2[ray] = hit ? lds.tri_hit[2][threadIdx.x] : 0.0f;
                hits.face[ray] = ts.res.face;
                if (hits.instance) hits.instance[ray] = 0u;
            }
            ray = kNone;
        }
    }
}

// Work-group of the persistent kernel: 512 lanes up to a stack of 10 groups, 256 for deeper ones, of which
// LDS holds too few otherwise.  Trees up to depth 11, which the 10 M triangle terrain has, get a stack of 10
// groups: with one of 12 their blocks were 256 lanes and 5 % slower on its camera rays, though 5 waves per
// SIMD are resident then and 4 (two blocks a CU) with 512.
template <int kStack>
constexpr int refill_block() {
    return kStack <= 10 ? 512 : 256;
}
// Waves per SIMD the registers are budgeted for (80 for six).  Six won for any-hit rays and for the
// shallow stacks of small scenes (Cornell image 9.49 against 9.83 ms), five for closest hits in deep
// trees, whose rays wait on memory and whose caches a sixth wave only divides (10 M terrain, 2 M rays:
// camera 480 -> 456 us, bounce 641 -> 630 us).
// At six, trace_vertex_kernel<8> spills two registers (12 bytes of scratch a lane); no other kernel here does.
template <bool ANY, int kStack>
constexpr int refill_waves() {
    return kStack > 12 ? 1 : ANY || kStack <= 8 ? 6 : 5;  // LDS bounds the deeper stacks
}

template <bool ANY, int kStack, bool kScaled = false>
__global__ __launch_bounds__(refill_block<kStack>(), (refill_waves<ANY, kStack>())) void trace_refill_kernel(
    const U4 *__restrict__ nodes, const F4 *__restrict__ tris, RayArgs rays, HitArgs hits, uint8_t *__restrict__ occluded,
    uint32_t n, const uint32_t *__restrict__ count, float root_max, uint32_t *__restrict__ fault, int cap) {
    constexpr int kBlk = refill_block<kStack>();
    __shared__ RefillLds<kStack, kBlk, !ANY> lds;
    if (threadIdx.x == 0) lds.next[0] = 0;
    __syncthreads();
    if (count) n = min(n, *count);
    refill_trace<ANY, kStack, kBlk>(OneScene<kScaled>{nodes, tris, root_max, fault, cap}, rays, hits, occluded, n, lds, lds.next[0]);
}

// One wavefront vertex in one launch: each wave traces its part of the continuation rays, goes on with its
// part of the shadow rays while the block's other waves still finish theirs, and once the block's
// shadow rays are known, the block adds the contributions of those that see their light -- the rays it
// traced, in queue order, so the reads are coalesced.  As three launches a vertex (closest, any,
// resolve) a 320 x 180 preview of 4 vertices took 233 us, as one 204, an OpenPBR frame of 8 vertices 3.41
// ms, now 2.98.
template <int kStack, int kBlk, class PathSource, class ShadowSource, class Lds>
__device__ __forceinline__ void trace_vertex(const PathSource &psrc, const RayArgs &rays, const HitArgs &hits, uint32_t paths,
                                             const ShadowSource &ssrc, const RayArgs &shadow, uint8_t *occluded,
                                             uint32_t shadows, const ResolveArgs &resolve, Lds &lds) {
    if (threadIdx.x < 2) lds.next[threadIdx.x] = 0;
    __syncthreads();
    refill_trace<false, kStack, kBlk>(psrc, rays, hits, nullptr, paths, lds, lds.next[0]);
    refill_trace<true, kStack, kBlk>(ssrc, shadow, HitArgs{}, occluded, shadows, lds, lds.next[1]);
    __syncthreads();
    const Deal deal(shadows, kBlk / 64);
    for (uint32_t draw = threadIdx.x / 64u;; draw += kBlk / 64) {
        const uint32_t at = deal.batch(draw);
        if (at >= deal.batches) break;
        const uint32_t i = at * 64u + (threadIdx.x & 63u);
        if (i < shadows && !occluded[i]) resolve_ray(resolve, i);
    }
}
template <int kStack>
__global__ __launch_bounds__(refill_block<kStack>(), (refill_waves<false, kStack>())) void trace_vertex_kernel(
    const U4 *__restrict__ nodes, const F4 *__restrict__ tris, RayArgs rays, HitArgs hits, const uint32_t *path_count,
    RayArgs shadow, uint8_t *occluded, const uint32_t *shadow_count, ResolveArgs resolve, uint32_t n, float root_max,
    uint32_t *__restrict__ fault, int cap) {
    constexpr int kBlk = refill_block<kStack>();
    __shared__ RefillLds<kStack, kBlk, true> lds;
    const OneScene<false> src{nodes, tris, root_max, fault, cap};
    trace_vertex<kStack, kBlk>(src, rays, hits, path_count ? min(n, *path_count) : 0u, src, shadow, occluded,
                               min(n, *shadow_count), resolve, lds);
}
__global__ __launch_bounds__(256) void resolve_kernel(ResolveArgs a, const uint8_t *occluded, const uint32_t *count, uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < min(n, *count) && !occluded[i]) resolve_ray(a, i);
}

// Two-level traversal (main.swift:1843-1900 mesh_closest, 1902-1983 mesh_occluded, software branch), on the
// persistent kernel's scheme: lanes refill as their rays end and the wave tests triangles together.  The
// instance hierarchy is walked as a one-level one whose leaves name instances, with the boxes grown by
// enlarge (|origin|max + reach); a leaf's instance traces its asset with the object-space ray, up to the
// closest hit so far.  A lane is on one level at a time and both visit nodes in the same instructions.
// Entering an instance (its record, the ray's transform, six divisions) costs the wave as much as a refill,
// so lanes wait for it in the same way; while a lane is inside, its place on the instance level rests in
// LDS: the ray's origin and reciprocals, the next node, the pending group and instances.
// Ties: the closest-hit rule compares (t, instance, face), so the result does not depend on the order
// instances are visited in.  At equal t a hit of this instance wins over the current one only if its index
// is smaller: the current hit's face then counts as the largest number, else as 0.
//
// Bound by the node test's instructions, a quarter of them at lanes' different levels, and by entering.
// 1024 instances of 1280 triangles, 2 M rays, against a ray per lane until its wave's slowest ends and
// one-lane triangle tests: camera rays 306 -> 243 us, random rays 870 -> 418, any-hit 806 -> 366.  Waiting to
// enter until half of the live lanes want it took 249 / 437 / 386 us; an eighth 245 / 426 / 377; making the
// instance level's ray anew on the way back, which fits a fifth wave per SIMD, 262 / 439 / 379.
constexpr int kTlasBlock = 256;
struct InstanceTris {
    static constexpr bool kShared = false;
    struct Lane {
        const F4 *tris;
    };
    __device__ __forceinline__ const F4 *tri_ptr(const Lane &l) const { return l.tris; }
};
// Where a lane left the instance level: next node (kNoTopNode: none), pending group, and the instances of
// the last leaf still to enter (bits as trav_nodes returns them).
enum : int { kTopNode, kTopBase, kTopBits, kItems, kItemBase, kItemBits, kTopWords };
constexpr uint32_t kNoTopNode = 0xffffffffu;

template <bool ANY, int kStack, bool kScaled = false>
__global__ __launch_bounds__(kTlasBlock, (kStack <= 10 ? 4 : 1)) void trace_tlas_kernel(TlasScene sc, RayArgs rays, HitArgs hits,
                                                                   uint8_t *__restrict__ occluded, uint32_t n) {
    __shared__ RefillLds<kStack, kTlasBlock, !ANY> lds;
    __shared__ float top_ray[6][kTlasBlock];
    __shared__ uint32_t top[kTopWords][kTlasBlock];
    if (threadIdx.x == 0) lds.next[0] = 0;
    __syncthreads();
    constexpr uint32_t kNone = 0xffffffffu;
    enum { kTop, kEnter, kMesh };
    const Deal deal(n, kTlasBlock / 64);
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const unsigned long long below = (1ull << lane) - 1ull;
    LdsStack<kStack, kTlasBlock> st{lds.stack_base, lds.stack_bits, (int)tid, 0, kStack};
    const InstanceTris src;
    InstanceTris::Lane sl{};
    TravState ts;
    uint32_t ray = kNone, trimask = 0, tri_base = 0, tri_bits = 0;
    uint32_t cur = 0, binst = 0xffffffffu;  // the instance the lane is in, and its closest hit's
    int32_t bface = -1, sentinel = -1;
    const U4 *nodes = nullptr;
    float scale = 1.0f;  // box scale of the lane's level: 1 but in an asset when kScaled (instances lie within 1e8)
    int mode = kTop;
    bool done = false, overflow = false;  // done: no node left on the lane's level
    uint32_t batch = 0, used = 64;
    bool exhausted = false;
    for (;;) {
        const unsigned long long need = __ballot(ray == kNone);
        if (!exhausted && __popcll(need) >= kRefillIdle) {
            const uint32_t cnt = (uint32_t)__popcll(need), rank = (uint32_t)__popcll(need & below);
            const uint32_t avail = 64u - used;
            uint32_t idx = batch + used + rank;
            if (cnt > avail) {
                uint32_t draw = 0;
                if (lane == 0) draw = atomicAdd(&lds.next[0], 1u);
                draw = __builtin_amdgcn_readfirstlane(draw);
                const uint32_t at = deal.batch(draw);
                exhausted = at >= deal.batches;
                const uint32_t fresh = exhausted ? n : at * 64u;
                if (rank >= avail) idx = fresh + (rank - avail);
                batch = fresh;
                used = cnt - avail;
            } else {
                used += cnt;
            }
            if (ray == kNone && idx < n) {
                const TraceRay r{rays.ox[idx], rays.oy[idx], rays.oz[idx], rays.dx[idx], rays.dy[idx], rays.dz[idx],
                                 rays.tmin[idx], rays.tmax[idx]};
                ray = idx;
                trav_init_e(ts, r, sc.enlarge * (max_abs3(r.ox, r.oy, r.oz) + sc.reach), 1.0f);
                top_ray[0][tid] = ts.ox;
                top_ray[1][tid] = ts.oy;
                top_ray[2][tid] = ts.oz;
                top_ray[3][tid] = ts.invx;
                top_ray[4][tid] = ts.invy;
                top_ray[5][tid] = ts.invz;
                st.sp = st.floor = 0;
                nodes = reinterpret_cast<const U4 *>(sc.nodes);
                scale = 1.0f;
                bface = -1;
                binst = 0xffffffffu;
                overflow = false;
                mode = kTop;
                done = !(r.tmax == r.tmax);  // nothing is nearer than a NaN
            }
        }
        const bool busy = ray != kNone;
        const unsigned long long live = __ballot(busy);
        if (!live && exhausted) break;
        const uint32_t lives = (uint32_t)__popcll(live);
        // Enter instances, enough lanes at a time, or as soon as no lane can do anything else.
        const unsigned long long enter = __ballot(busy && mode == kEnter);
        const unsigned long long steps = __ballot(busy && mode != kEnter && !done && trimask == 0u);
        if (enter && (__popcll(enter) >= kRefillIdle || 4u * (uint32_t)__popcll(enter) >= lives || !steps)) {
            if (busy && mode == kEnter) {
                uint32_t items = top[kItems][tid];
                const uint32_t b = __builtin_ctz(items);
                top[kItems][tid] = items & (items - 1u);
                const InstanceRecord &R = sc.instances[top[kItemBase][tid] + tri_rank(top[kItemBits][tid], b)];
                const TraceRay r{rays.ox[ray], rays.oy[ray], rays.oz[ray], rays.dx[ray], rays.dy[ray], rays.dz[ray],
                                 ts.tmin, 0.0f};
                const TraceRay l = instance_ray(R.local, r, ts.res.t);
                if (kScaled) scale = box_scale(R.root_max);
                trav_init(ts, l, R.root_max, scale);
                lds.woop[tid] = pack_woop(woop_ray(l.dx, l.dy, l.dz));
                cur = R.index;
                sentinel = (bface >= 0 && cur < binst) ? 0x7fffffff : -1;
                ts.res.face = sentinel;
                nodes = reinterpret_cast<const U4 *>(R.nodes);
                sl.tris = reinterpret_cast<const F4 *>(R.tris);
                mode = kMesh;
                done = R.faces == 0u;
            }
        }
        if (busy && mode != kEnter && !done && trimask == 0u) {
            uint32_t mask;
            done = trav_nodes<false>(ts, nodes, scale, st, mask, tri_base, tri_bits);
            if (mode == kMesh) {
                trimask = mask;
            } else if (mask) {
                top[kTopNode][tid] = done ? kNoTopNode : ts.node;
                top[kTopBase][tid] = ts.cur_base;
                top[kTopBits][tid] = ts.cur_bits;
                top[kItems][tid] = mask;
                top[kItemBase][tid] = tri_base;
                top[kItemBits][tid] = tri_bits;
                st.floor = st.sp;
                overflow |= ts.res.overflow;
                mode = kEnter;
                done = false;
            }
        }
        const unsigned long long waiting = __ballot(busy && (done || trimask != 0u));
        if (4u * (uint32_t)__popcll(waiting) >= lives || (!steps && waiting)) {
            uint32_t pre, total;
            wave_prefix(__popc(trimask), below, pre, total);
            wave_triangles<ANY, kTlasBlock>(src, sl, ts, trimask, tri_base, tri_bits, lane, pre, total, lds.woop, lds.tri_key,
                                            lds.tri_hit);
            trimask = 0u;
        }
        bool end = busy && done && trimask == 0u && mode == kTop;
        if (busy && mode == kMesh && ((done && trimask == 0u) || (ANY && ts.res.occluded))) {
            // The instance is done: the next of its leaf, or back to the instance level.
            if (!ANY && ts.res.face != sentinel) {
                bface = ts.res.face;
                binst = cur;
            }
            overflow |= ts.res.overflow;
            done = false;
            trimask = 0u;
            st.sp = st.floor;
            if (ANY && ts.res.occluded) {
                end = true;
            } else if (top[kItems][tid] != 0u) {
                mode = kEnter;
            } else if (top[kTopNode][tid] == kNoTopNode) {
                end = true;
            } else {
                mode = kTop;
                st.floor = 0;
                nodes = reinterpret_cast<const U4 *>(sc.nodes);
                ts.node = top[kTopNode][tid];
                ts.cur_base = top[kTopBase][tid];
                ts.cur_bits = top[kTopBits][tid];
                ts.ox = top_ray[0][tid];
                ts.oy = top_ray[1][tid];
                ts.oz = top_ray[2][tid];
                ts.invx = top_ray[3][tid];
                ts.invy = top_ray[4][tid];
                ts.invz = top_ray[5][tid];
                set_enlargement(ts, sc.enlarge * (max_abs3(ts.ox, ts.oy, ts.oz) + sc.reach));
                scale = 1.0f;
                ts.oct = (float_to_bits(ts.invx) >> 31) | (float_to_bits(ts.invy) >> 31 << 1) |
                         (float_to_bits(ts.invz) >> 31 << 2);
                ts.res.overflow = false;
            }
        }
        if (end) {
            if ((overflow || ts.res.overflow) && sc.fault) atomicOr(sc.fault, 1u);
            if (ANY) {
                occluded[ray] = ts.res.occluded ? 1 : 0;
            } else {
                const bool hit = bface >= 0;
                hits.t[ray] = ts.res.t;
                hits.b1[ray] = hit ? lds.tri_hit[1][tid] : 0.0f;
                hits.b2[ray] = hit ? lds.tri_hit[2][tid] : 0.0f;
                hits.face[ray] = bface;
                if (hits.instance) hits.instance[ray] = binst;
            }
            ray = kNone;
        }
    }
}

template <bool ANY>
__global__ __launch_bounds__(256) void miss_kernel(RayArgs rays, HitArgs hits, uint8_t *occluded, uint32_t n,
                                                   const uint32_t *count, uint32_t miss_instance) {
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (count) n = min(n, *count);
    if (i >= n) return;
    if (ANY) {
        occluded[i] = 0;
    } else {
        hits.t[i] = rays.tmax[i];
        hits.b1[i] = 0.0f;
        hits.b2[i] = 0.0f;
        hits.face[i] = -1;
        if (hits.instance) hits.instance[i] = miss_instance;
    }
}

// The reference's software traversal of its flat binary hierarchy (trace_scene's mesh branch,
// main.swift:2058-2080, with mesh_box_ray / mesh_node_hit / push_mesh_children :1511-1528): one ray per
// lane, a stack of node indices in LDS, the child on the ray's side of the node's split axis first.
// Boxes are the reference's: the slabs of [lo, hi] against the origin moved by -+e, e = 2^-23 (1 + ...)
// x (|origin|max + |root|max), a direction component below 1e-8 testing the origin against the
// enlarged slab.  Triangles are the same watertight test as the 8-wide traversal, and the closest-hit
// rule the same (t, then the smaller document face index at equal t), so hits do not depend on the
// hierarchy.  A ray whose stack would overflow (never, for the depths the host admits) raises *fault.
template <bool ANY>
__global__ __launch_bounds__(256) void trace_median_kernel(const F4 *__restrict__ nodes, const F4 *__restrict__ tris,
                                                           RayArgs rays, HitArgs hits, uint8_t *__restrict__ occluded,
                                                           uint32_t n, const uint32_t *__restrict__ count, float root_max,
                                                           uint32_t *__restrict__ fault) {
    __shared__ uint32_t stack[kMedianStack][256];
    const uint32_t lane = threadIdx.x, i = blockIdx.x * 256 + lane;
    if (count) n = min(n, *count);
    if (i >= n) return;
    const float o[3] = {rays.ox[i], rays.oy[i], rays.oz[i]}, d[3] = {rays.dx[i], rays.dy[i], rays.dz[i]};
    const float tmin = rays.tmin[i], tmax = rays.tmax[i];
    const WoopRay w = woop_ray(d[0], d[1], d[2]);
    const float e = 1.1920929e-6f * (fmaxf(fabsf(o[0]), fmaxf(fabsf(o[1]), fabsf(o[2]))) + root_max);
    const float low[3] = {o[0] + e, o[1] + e, o[2] + e}, high[3] = {o[0] - e, o[1] - e, o[2] - e};
    float best = tmax, bb1 = 0.0f, bb2 = 0.0f;
    int32_t bface = -1;
    bool hit = false, overflow = false;
    uint32_t top = 0;
    stack[top++][lane] = 0u;
    while (top > 0u) {
        const uint32_t ni = stack[--top][lane];
        const F4 lo = nodes[3 * (size_t)ni], hi = nodes[3 * (size_t)ni + 1], lk = nodes[3 * (size_t)ni + 2];
        const int32_t links[4] = {(int32_t)__float_as_uint(lk.x), (int32_t)__float_as_uint(lk.y),
                                  (int32_t)__float_as_uint(lk.z), (int32_t)__float_as_uint(lk.w)};
        // mesh_node_hit against [tmin, closest hit so far].
        float near_t = tmin, far_t = ANY ? tmax : best;
        const float nlo[3] = {lo.x, lo.y, lo.z}, nhi[3] = {hi.x, hi.y, hi.z};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (fabsf(d[a]) < 1e-8f) {
                if (low[a] < nlo[a] || high[a] > nhi[a]) far_t = -1.0f;
            } else {
                const float ta = (nlo[a] - low[a]) / d[a], tb = (nhi[a] - high[a]) / d[a];
                near_t = fmaxf(near_t, fminf(ta, tb));
                far_t = fminf(far_t, fmaxf(ta, tb));
            }
        }
        if (!(near_t <= far_t)) continue;
        if (links[3] == 0) {
            if (top + 2u > kMedianStack) {
                overflow = true;
                continue;
            }
            const int axis = min(max(links[2], 0), 2);
            const bool left_first = d[axis] >= 0.0f;
            stack[top++][lane] = (uint32_t)(left_first ? links[1] : links[0]);
            stack[top++][lane] = (uint32_t)(left_first ? links[0] : links[1]);
            continue;
        }
        for (int32_t k = 0; k < links[3]; ++k) {
            const size_t r = 3 * (size_t)(links[2] + k);
            const F4 p0 = tris[r], p1 = tris[r + 1], p2 = tris[r + 2];
            const int32_t face = (int32_t)__float_as_uint(p0.w);
            float t, b1, b2;
            if (!woop_triangle(w, o[0], o[1], o[2], p0, p1, p2, t, b1, b2)) continue;
            if (ANY) {
                if (t >= tmin && t < tmax) {
                    hit = true;
                    break;
                }
                continue;
            }
            if (t >= tmin && (t < best || (t == best && bface >= 0 && face < bface))) {
                best = t;
                bb1 = b1;
                bb2 = b2;
                bface = face;
            }
        }
        if (ANY && hit) break;
    }
    if (overflow && fault) atomicOr(fault, 1u);
    if (ANY) {
        occluded[i] = hit ? 1 : 0;
    } else {
        hits.t[i] = best;
        hits.b1[i] = bb1;
        hits.b2[i] = bb2;
        hits.face[i] = bface;
        if (hits.instance) hits.instance[i] = 0u;
    }
}

// Batched rendering: a vertex's rays of many scenes in one persistent launch.  Ray i of a queue belongs to
// job job[i], whose scene is job_trace[job[i]]; rays of one job are contiguous in the queues, so a wave
// rarely spans two scenes.
template <int kStack, int kBlk, bool kScaled = false>
__global__ __launch_bounds__(kBlk, (kStack <= 12 && kBlk <= 256 ? 5 : 1)) void batch_trace_kernel(
    const TraceScene *__restrict__ job_trace, const uint32_t *__restrict__ path_job, RayArgs rays, HitArgs hits,
    const uint32_t *path_count, const uint32_t *__restrict__ shadow_job, RayArgs shadow, uint8_t *occluded,
    const uint32_t *shadow_count, ResolveArgs resolve, uint32_t n) {
    __shared__ RefillLds<kStack, kBlk, true> lds;
    trace_vertex<kStack, kBlk>(JobScenes<kScaled>{job_trace, path_job}, rays, hits, path_count ? min(n, *path_count) : 0u,
                               JobScenes<kScaled>{job_trace, shadow_job}, shadow, occluded,
                               shadow_count ? min(n, *shadow_count) : 0u, resolve, lds);
}

}  // namespace

namespace {

// Blocks of the refill kernel that are resident at once on the current device (at least 1), at most one
// per batch of 64 rays (a launch of few rays leaves most waves of a block idle but reaches every CU); the
// occupancy query is made once per kernel.
uint32_t refill_grid(const void *kernel, uint32_t n, int block) {
    struct Entry {
        const void *k;
        uint32_t blocks;
    };
    static Entry cache[32] = {};
    static std::mutex lock;
    std::lock_guard<std::mutex> guard(lock);
    uint32_t resident = 0;
    for (auto &e : cache)
        if (e.k == kernel) resident = e.blocks;
    if (!resident) {
        int dev = 0, cus = 256, per = 1;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, block, 0) != hipSuccess || per < 1) per = 1;
        resident = (uint32_t)(cus * per);
        for (auto &e : cache)
            if (!e.k) {
                e = Entry{kernel, resident};
                break;
            }
    }
    const uint32_t need = n / 64u + (n % 64u != 0u);
    return need < resident ? (need > 0 ? need : 1) : resident;
}

}  // namespace

// ---------------------------------------------------------------- allocation-free work counters
// The counting traversal's 64 partial (node fetches, triangle tests) pairs live in this file-scope
// array: 1 KiB per device, whatever the number of rays.  Host code never passes the symbol itself
// (in host code it only names a stand-in); it passes the per-device address scratch_init found.
static __device__ __align__(256) unsigned long long scratch[kStatsScratchWords];

namespace {
constexpr int kMaxDevices = 64;
void *g_scratch[kMaxDevices] = {};
std::mutex g_scratch_lock;

__global__ void zero_scratch_kernel(unsigned long long *p) {
    if (threadIdx.x < kStatsScratchWords) p[threadIdx.x] = 0ull;
}
__global__ void sum_pairs_kernel(const unsigned long long *p, unsigned long long *out) {
    if (threadIdx.x != 0) return;
    unsigned long long nodes = 0, tris = 0;
    for (int k = 0; k < kStatsScratchWords / 2; ++k) {
        nodes += p[2 * k];
        tris += p[2 * k + 1];
    }
    out[0] = nodes;
    out[1] = tris;
}
}  // namespace

hipError_t scratch_init(int device) {
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> guard(g_scratch_lock);
    if (g_scratch[device]) return hipSuccess;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch[device] = p;
    return hipSuccess;
}

hipError_t launch_trace_stats_scratch(int device, const TraceScene &scene, const RayArgs &rays, const HitArgs &hits,
                                      uint8_t *occluded, uint32_t n, bool any, unsigned long long *out,
                                      hipStream_t stream) {
    if (device < 0 || device >= kMaxDevices || !g_scratch[device]) return hipErrorNotInitialized;
    unsigned long long *p = static_cast<unsigned long long *>(g_scratch[device]);
    hipLaunchKernelGGL(zero_scratch_kernel, dim3(1), dim3(kStatsScratchWords), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (n) {
        e = launch_trace(scene, rays, hits, occluded, n, any, p, stream);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(sum_pairs_kernel, dim3(1), dim3(64), 0, stream, p, out);
    return hipGetLastError();
}

// Node8 records (bvh8.h) re-encoded in place for the traversal (traverse8.h), a record a thread.
__global__ __launch_bounds__(256) void encode_nodes_kernel(U4 *nodes, uint32_t n, float scale) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    U4 in[5], out[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) in[k] = nodes[5 * (size_t)i + k];
    encode_node(in, out, scale);
#pragma unroll
    for (int k = 0; k < 5; ++k) nodes[5 * (size_t)i + k] = out[k];
}
hipError_t launch_encode_nodes(void *nodes, uint32_t n, float root_max, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(encode_nodes_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, static_cast<U4 *>(nodes), n,
                       box_scale(root_max));
    return hipGetLastError();
}

hipError_t launch_trace_vertex_batch(const TraceScene *job_trace, const uint32_t *path_job, const RayArgs &rays,
                                     const HitArgs &hits, const uint32_t *path_count, const uint32_t *shadow_job,
                                     const RayArgs &shadow, uint8_t *occluded, const uint32_t *shadow_count,
                                     const ResolveArgs &resolve, uint32_t n, uint32_t max_depth, float max_root, uint32_t block,
                                     uint32_t grid, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const int need = max_depth > 1 ? (int)max_depth - 1 : 1;
    if (need > 24 || (block != 64 && block != 128 && block != 256 && block != 512) || grid == 0) return hipErrorInvalidValue;
#define VT_BATCH(S, B, X)                                                                                              \
    hipLaunchKernelGGL((batch_trace_kernel<S, B, X>), dim3(grid), dim3(B), 0, stream, job_trace, path_job, rays, hits,  \
                       path_count, shadow_job, shadow, occluded, shadow_count, resolve, n)
#define VT_BATCH_STACK(S, X)                                                                                           \
    do {                                                                                                               \
        if (block == 64) VT_BATCH(S, 64, X);                                                                           \
        else if (block == 128) VT_BATCH(S, 128, X);                                                                    \
        else if (block == 256) VT_BATCH(S, 256, X);                                                                    \
        else VT_BATCH(S, 512, X);                                                                                      \
    } while (0)
    if (box_scale(max_root) != 1.0f) VT_BATCH_STACK(24, true);
    else if (need <= 8) VT_BATCH_STACK(8, false);
    else if (need <= 12) VT_BATCH_STACK(12, false);
    else if (need <= 16) VT_BATCH_STACK(16, false);
    else VT_BATCH_STACK(24, false);
#undef VT_BATCH_STACK
#undef VT_BATCH
    return hipGetLastError();
}

hipError_t launch_trace_vertex(const TraceScene &scene, const RayArgs &rays, const HitArgs &hits, const uint32_t *path_count,
                               const RayArgs &shadow, uint8_t *occluded, const uint32_t *shadow_count,
                               const ResolveArgs &resolve, uint32_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const int need = scene.depth > 1 ? (int)scene.depth - 1 : 1;
    if (scene.node_count == 0 || scene.kind != 0u || need > 24 || box_scale(scene.root_max) != 1.0f) {
        // No 8-wide hierarchy, or one with scaled boxes: a launch for each part.
        hipError_t e = path_count ? launch_trace(scene, rays, hits, nullptr, n, false, nullptr, stream, path_count) : hipSuccess;
        if (e != hipSuccess) return e;
        e = launch_trace(scene, shadow, HitArgs{}, occluded, n, true, nullptr, stream, shadow_count);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(resolve_kernel, dim3(n / 256u + (n % 256u != 0u)), dim3(256), 0, stream, resolve, occluded,
                           shadow_count, n);
        return hipGetLastError();
    }
    const U4 *nd = reinterpret_cast<const U4 *>(scene.nodes);
    const F4 *tr = reinterpret_cast<const F4 *>(scene.tris);
    const int cap = scene.stack_cap ? (int)scene.stack_cap : 24;
#define VT_VERTEX(S)                                                                                                   \
    hipLaunchKernelGGL((trace_vertex_kernel<S>), dim3(refill_grid((const void *)trace_vertex_kernel<S>, n, refill_block<S>())), \
                       dim3(refill_block<S>()), 0, stream, nd, tr, rays, hits, path_count, shadow, occluded, shadow_count,     \
                       resolve, n, scene.root_max, scene.fault, cap < S ? cap : S)
    if (need <= 8) VT_VERTEX(8);
    else if (need <= 10) VT_VERTEX(10);
    else if (need <= 12) VT_VERTEX(12);
    else if (need <= 16) VT_VERTEX(16);
    else VT_VERTEX(24);
#undef VT_VERTEX
    return hipGetLastError();
}

hipError_t launch_trace_tlas(const TlasScene &scene, const RayArgs &rays, const HitArgs &hits, uint8_t *occluded,
                             uint32_t n, bool any, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    if (scene.node_count == 0) {
        dim3 grid((n + 255) / 256);
        if (any) hipLaunchKernelGGL(miss_kernel<true>, grid, dim3(256), 0, stream, rays, hits, occluded, n, nullptr, 0u);
        else hipLaunchKernelGGL(miss_kernel<false>, grid, dim3(256), 0, stream, rays, hits, occluded, n, nullptr, 0xffffffffu);
        return hipGetLastError();
    }
    const int top = scene.depth > 1 ? (int)scene.depth - 1 : 1, bot = scene.blas_depth > 1 ? (int)scene.blas_depth - 1 : 1;
    if (top > 16 || bot > 24) return hipErrorInvalidValue;
    // One stack holds the instance level's pending groups and, above them, those of the mesh a ray is in.
#define VT_TLAS(S, X)                                                                                                  \
    do {                                                                                                               \
        const uint32_t g = refill_grid(any ? (const void *)trace_tlas_kernel<true, S, X> : (const void *)trace_tlas_kernel<false, S, X>, n, kTlasBlock); \
        if (any) hipLaunchKernelGGL((trace_tlas_kernel<true, S, X>), dim3(g), dim3(kTlasBlock), 0, stream, scene, rays, hits, occluded, n); \
        else hipLaunchKernelGGL((trace_tlas_kernel<false, S, X>), dim3(g), dim3(kTlasBlock), 0, stream, scene, rays, hits, occluded, n); \
    } while (0)
    if (box_scale(scene.blas_max) != 1.0f) VT_TLAS(40, true);
    else if (top + bot <= 10) VT_TLAS(10, false);
    else if (top + bot <= 16) VT_TLAS(16, false);
    else if (top + bot <= 24) VT_TLAS(24, false);
    else VT_TLAS(40, false);
#undef VT_TLAS
    return hipGetLastError();
}

hipError_t launch_trace(const TraceScene &scene, const RayArgs &rays, const HitArgs &hits, uint8_t *occluded,
                        uint32_t n, bool any, unsigned long long *counters, hipStream_t stream, const uint32_t *count) {
    if (n == 0) return hipSuccess;
    if (scene.node_count == 0) {
        dim3 grid((n + 255) / 256);
        if (any) hipLaunchKernelGGL(miss_kernel<true>, grid, dim3(256), 0, stream, rays, hits, occluded, n, count, 0u);
        else hipLaunchKernelGGL(miss_kernel<false>, grid, dim3(256), 0, stream, rays, hits, occluded, n, count, 0u);
        return hipGetLastError();
    }
    if (scene.kind == 1u) {
        // The reference's flat binary hierarchy: no counting variant.
        if (counters) return hipErrorInvalidValue;
        const dim3 grid((n + 255) / 256);
        const F4 *nd = reinterpret_cast<const F4 *>(scene.nodes), *tr = reinterpret_cast<const F4 *>(scene.tris);
        if (any)
            hipLaunchKernelGGL(trace_median_kernel<true>, grid, dim3(256), 0, stream, nd, tr, rays, hits, occluded, n,
                               count, scene.root_max, scene.fault);
        else
            hipLaunchKernelGGL(trace_median_kernel<false>, grid, dim3(256), 0, stream, nd, tr, rays, hits, occluded, n,
                               count, scene.root_max, scene.fault);
        return hipGetLastError();
    }
    dim3 grid((n + kBlock - 1) / kBlock), block(kBlock);
    const U4 *nd = reinterpret_cast<const U4 *>(scene.nodes);
    const F4 *tr = reinterpret_cast<const F4 *>(scene.tris);
    const int need = scene.depth > 1 ? (int)scene.depth - 1 : 1;
    if (need > 24) return hipErrorInvalidValue;
    const int cap = scene.stack_cap ? (int)scene.stack_cap : 24;
    if (!counters) {
        // Persistent refill kernel: as many blocks as the chip holds at once (never more than the rays
        // need), each drawing its share of the rays.
#define VT_REFILL(S, X)                                                                                                \
    do {                                                                                                               \
        constexpr int b = refill_block<S>();                                                                          \
        const uint32_t g = refill_grid(any ? (const void *)trace_refill_kernel<true, S, X> : (const void *)trace_refill_kernel<false, S, X>, n, b); \
        if (any) hipLaunchKernelGGL((trace_refill_kernel<true, S, X>), dim3(g), dim3(b), 0, stream, nd, tr, rays, hits, occluded, n, count, scene.root_max, scene.fault, cap < S ? cap : S); \
        else hipLaunchKernelGGL((trace_refill_kernel<false, S, X>), dim3(g), dim3(b), 0, stream, nd, tr, rays, hits, occluded, n, count, scene.root_max, scene.fault, cap < S ? cap : S); \
    } while (0)
        if (box_scale(scene.root_max) != 1.0f) VT_REFILL(24, true);
        else if (need <= 8) VT_REFILL(8, false);
        else if (need <= 10) VT_REFILL(10, false);
        else if (need <= 12) VT_REFILL(12, false);
        else if (need <= 16) VT_REFILL(16, false);
        else VT_REFILL(24, false);
#undef VT_REFILL
        return hipGetLastError();
    }
#define VT_LAUNCH(S)                                                                                                   \
    do {                                                                                                               \
        if (any) hipLaunchKernelGGL((count_kernel<true, S>), grid, block, 0, stream, nd, tr, rays, hits, occluded, n, count, scene.root_max, counters, scene.fault, cap < S ? cap : S); \
        else hipLaunchKernelGGL((count_kernel<false, S>), grid, block, 0, stream, nd, tr, rays, hits, occluded, n, count, scene.root_max, counters, scene.fault, cap < S ? cap : S); \
    } while (0)
    if (need <= 8) VT_LAUNCH(8);
    else if (need <= 12) VT_LAUNCH(12);
    else if (need <= 16) VT_LAUNCH(16);
    else VT_LAUNCH(24);
#undef VT_LAUNCH
    return hipGetLastError();
}

}  // namespace vt
