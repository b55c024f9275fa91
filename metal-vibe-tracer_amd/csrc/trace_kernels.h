// trace_kernels.h -- launch interface between the host runtime and the traversal kernels.
#pragma once
#include <hip/hip_runtime_api.h>
#include <stdint.h>

namespace vt {

struct RayArgs {
    const float *ox, *oy, *oz, *dx, *dy, *dz, *tmin, *tmax;
};
struct HitArgs {
    float *t, *b1, *b2;
    int32_t *face;
    uint32_t *instance;
};
struct TraceScene {
    const void *nodes;  // the 8-wide nodes, encoded for the traversal (launch_encode_nodes), or MeshNode records
    const void *tris;   // TriRecord records
    uint32_t node_count;
    uint32_t depth;  // tree depth (root = 1); the traversal stack holds depth - 1 groups
    float root_max;
    // Device word raised (bit 0) by a ray whose node-group stack filled: the ray ends early with the
    // hit found so far.  The launcher sizes the stack to depth - 1 groups, which a traversal never
    // exceeds (one pending group per level), so only a stack capped below that (stack_cap, a test
    // hook; 0 = no cap) can raise it.
    uint32_t *fault;
    uint32_t stack_cap;
    // 0: the 8-wide tree; 1: MeshNode records (the reference's flat binary median
    // hierarchy, bvh8.h), walked by trace_median_kernel with a stack of kMedianStack entries.
    uint32_t kind = 0;
};
constexpr uint32_t kMedianStack = 32;

// Two-level scenes (the reference's MeshSceneLayout, Sources/Acceleration.swift:356-573): an 8-wide
// hierarchy over the instances' world bounds whose leaf slots name InstanceRecords (in leaf order),
// each tracing its asset's hierarchy with the object-space ray.
struct alignas(16) InstanceRecord {
    float local[3][4];  // rows of the world-to-object matrix: x = row.xyz . p + row.w
    const void *nodes;  // the asset's encoded nodes
    const void *tris;   // the asset's TriRecord records
    float root_max;     // the asset's max |local coordinate| (its box enlargement term)
    uint32_t index;     // the instance's position in the caller's list
    uint32_t faces;     // the asset's face count (0: nothing to trace)
    uint32_t pad;
};
static_assert(sizeof(InstanceRecord) == 80, "InstanceRecord is five 16-byte words");
struct TlasScene {
    const void *nodes;                  // encoded nodes over instance bounds
    const InstanceRecord *instances;    // leaf order
    uint32_t node_count, depth;         // of the instance hierarchy
    uint32_t blas_depth;                // deepest asset hierarchy
    float blas_max;                     // largest root_max of the assets
    float enlarge, reach;               // per-ray growth of the instance boxes: enlarge (|origin|max + reach)
    uint32_t *fault;                    // raised (bit 0) by a ray whose node-group stack filled
};
// Re-encodes n Node8 records (bvh8.h) of a hierarchy with max |coordinate| root_max in place, in device
// memory, as the traversal reads them (traverse8.h).
hipError_t launch_encode_nodes(void *nodes, uint32_t n, float root_max, hipStream_t stream);

// Closest hit (hits.instance = the instance's index, 0xffffffff on a miss) or any hit over a
// two-level scene.  Among hits at exactly equal t the smaller instance index wins, then the smaller
// face index.
hipError_t launch_trace_tlas(const TlasScene &scene, const RayArgs &rays, const HitArgs &hits, uint8_t *occluded,
                             uint32_t n, bool any, hipStream_t stream);

// Closest hit (any = false) into `hits`, or any hit into `occluded`.  `counters` (device, 128
// u64, zeroed by the caller) selects the counting variant: 64 pairs (node fetches, triangle tests).
// `count` (device, optional) caps n at launch time: the wavefront integrator's queue length.
hipError_t launch_trace(const TraceScene &scene, const RayArgs &rays, const HitArgs &hits, uint8_t *occluded,
                        uint32_t n, bool any, unsigned long long *counters, hipStream_t stream,
                        const uint32_t *count = nullptr);

// The contributions of a wavefront's shadow rays (ray i's to path id[i], resolve.h).  sacc is null unless
// a radiance cache trains on the paths.
struct ResolveArgs {
    const uint32_t *id;
    const float *r, *g, *b;
    const float4 *s;
    float *radiance;
    float4 *sacc;
    uint32_t npix, sample_index0, train_period;
};
// One wavefront vertex's rays in one launch: the closest hits of min(n, *path_count) continuation rays into
// `hits`, the any hits of min(n, *shadow_count) shadow rays into `occluded`, and the contributions of the
// shadow rays that see their light (resolve).  path_count null: no continuation rays.
hipError_t launch_trace_vertex(const TraceScene &scene, const RayArgs &rays, const HitArgs &hits, const uint32_t *path_count,
                               const RayArgs &shadow, uint8_t *occluded, const uint32_t *shadow_count,
                               const ResolveArgs &resolve, uint32_t n, hipStream_t stream);

// The counting traversal of launch_trace (counters variant) with its partial counters in the
// library's static device scratch (kStatsScratchWords u64, 64 pairs) instead of an allocation:
// zeroes the scratch with a kernel, traces into the caller's hits / occluded, and sums the pairs into
// out[0] (node fetches) and out[1] (triangle tests), device memory.  Asynchronous; allocates nothing.
// scratch_init(device) must have run once with `device` current.  Calls that overlap on one device
// race on the scratch.
constexpr int kStatsScratchWords = 128;
hipError_t scratch_init(int device);
hipError_t launch_trace_stats_scratch(int device, const TraceScene &scene, const RayArgs &rays, const HitArgs &hits,
                                      uint8_t *occluded, uint32_t n, bool any, unsigned long long *out,
                                      hipStream_t stream);

// launch_trace_vertex of batched rendering: ray i of a queue traces the scene job_trace[job[i]], on a
// persistent grid of `grid` blocks of `block` (64, 128, 256 or 512) lanes; max_depth is the deepest tree, max_root
// the largest root_max.
// path_count or shadow_count null: none of those rays.
hipError_t launch_trace_vertex_batch(const TraceScene *job_trace, const uint32_t *path_job, const RayArgs &rays,
                                     const HitArgs &hits, const uint32_t *path_count, const uint32_t *shadow_job,
                                     const RayArgs &shadow, uint8_t *occluded, const uint32_t *shadow_count,
                                     const ResolveArgs &resolve, uint32_t n, uint32_t max_depth, float max_root, uint32_t block,
                                     uint32_t grid, hipStream_t stream);

}  // namespace vt
