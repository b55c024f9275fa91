// resolve.h -- what happens to a shadow ray's contribution once its visibility is known, shared by the
// traversal kernels that trace a wavefront's shadow rays and the shading kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "trace_kernels.h"

namespace vt {

// pcg_hash (main.swift:91-95).
__device__ __forceinline__ uint32_t pcg_hash(uint32_t input) {
    uint32_t state = input * 747796405u + 2891336453u;
    uint32_t word = ((state >> ((state >> 28u) + 4u)) ^ state) * 277803737u;
    return (word >> 22u) ^ word;
}

// Training paths of the radiance cache: 1 in `period`, by a hash of pixel and sample index.
__device__ __forceinline__ bool nrc_training_path(uint32_t npix, uint32_t sample_index0, uint32_t period, uint32_t id) {
    const uint32_t smp = id / npix, pix = id - smp * npix;
    return pcg_hash((pix * 0x9E3779B9u) ^ ((sample_index0 + smp) * 0x85EBCA6Bu)) % period == 0u;
}

// Adds shadow ray i's contribution to its path's radiance (and, for a training path, to the spectral
// radiance it has gathered).  A path casts at most one shadow ray per vertex, so no two rays of a
// launch share one.
__device__ __forceinline__ void resolve_ray(const ResolveArgs &a, uint32_t i) {
    const uint32_t id = a.id[i];
    a.radiance[3 * (size_t)id] += a.r[i];
    a.radiance[3 * (size_t)id + 1] += a.g[i];
    a.radiance[3 * (size_t)id + 2] += a.b[i];
    if (a.sacc && nrc_training_path(a.npix, a.sample_index0, a.train_period, id)) {
        const float4 v = a.s[i], s = a.sacc[id];
        a.sacc[id] = make_float4(s.x + v.x, s.y + v.y, s.z + v.z, s.w + v.w);
    }
}

}  // namespace vt
