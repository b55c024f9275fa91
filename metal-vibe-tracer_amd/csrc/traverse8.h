// traverse8.h -- per-ray traversal of the 8-wide compressed BVH, shared by every kernel that traces
// (closest-hit, any-hit, and the integrator's extend/shadow stages).
//
// The builder's Node8 records (bvh8.h) are re-encoded on the device when a hierarchy is published
// (encode_node) into the form the node test reads with the fewest instructions, 80 bytes as before, five
// 16-byte words:
//   w0   grid origin px, py, pz; the high halves of the x and y steps (low and high 16 bits)
//   w1   first child, first triangle; the high half of the z step (high 16 bits); the triangles of the
//        leaf children, three bits per slot (bit 3 s + q: slot s has a q-th triangle), and the inner
//        children (bits 24 + s)
//   w2-4 per axis, word k: low and high plane of slot 2 k, low and high plane of slot 2 k + 1
// A step is a power of two, so its high 16 bits are all of it; it is stored times 2^24, because the node
// test reads a plane byte as the fp16 number with those bits, q 2^-24.  Origin and steps are further stored
// times the hierarchy's box scale (box_scale), 1 for all but scenes of astronomical size.
//
// The node-group stack is abstracted (Stack::push/pop/size) so a kernel keeps it in LDS.
// Arithmetic follows the reference exactly where results depend on it:
//   * boxes: conservative slab test of wide_node_hit (main.swift:1766-1779) on the exactly
//     dequantised child boxes, grown by e = 1.1920929e-6 (|o|max + root max) (main.swift:1792);
//   * triangles: watertight Woop test (main.swift:1537-1582), products rounded separately,
//     correctly rounded divisions, FMA tie-break of equal rounded edge products.
// Among hits at exactly equal t the smaller document face index wins.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define VT_HD __host__ __device__ __forceinline__
#else
#include <cmath>
#include <cstring>
#define VT_HD inline
#endif

namespace vt {

struct U4 {
    uint32_t x, y, z, w;
};
struct F4 {
    float x, y, z, w;
};

VT_HD float bits_to_float(uint32_t u) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __uint_as_float(u);
#else
    float f;
    __builtin_memcpy(&f, &u, 4);
    return f;
#endif
}
VT_HD uint32_t float_to_bits(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __float_as_uint(f);
#else
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    return u;
#endif
}

struct WoopRay {
    int kx, ky, kz;
    float sx, sy, sz;
};

VT_HD float sel3(float x, float y, float z, int k) { return k == 0 ? x : (k == 1 ? y : z); }

// main.swift:1537-1550 watertight_ray.
VT_HD WoopRay woop_ray(float dx, float dy, float dz) {
    float ax = fabsf(dx), ay = fabsf(dy), az = fabsf(dz);
    int kz = ax > ay ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int kx = kz == 2 ? 0 : kz + 1, ky = kx == 2 ? 0 : kx + 1;
    float dkz = sel3(dx, dy, dz, kz);
    if (dkz < 0.0f) {
        int s = kx;
        kx = ky;
        ky = s;
    }
    WoopRay w;
    w.kx = kx;
    w.ky = ky;
    w.kz = kz;
    w.sx = sel3(dx, dy, dz, kx) / dkz;
    w.sy = sel3(dx, dy, dz, ky) / dkz;
    w.sz = 1.0f / dkz;
    return w;
}

// main.swift:1557-1562 watertight_edge.
VT_HD float watertight_edge(float px, float py, float qx, float qy) {
#pragma clang fp contract(off)
    float x = px * qy, y = py * qx, e = x - y;
    if (e == 0.0f) e = __builtin_fmaf(px, qy, -x) - __builtin_fmaf(py, qx, -y);
    return e;
}

// main.swift:1564-1578 without the [tmin, tmax) check (the caller applies it).
VT_HD bool woop_triangle(const WoopRay &w, float ox, float oy, float oz, F4 p0, F4 p1, F4 p2, float &t, float &b1,
                         float &b2) {
#pragma clang fp contract(off)
    float Ax = p0.x - ox, Ay = p0.y - oy, Az = p0.z - oz;
    float Bx = p1.x - ox, By = p1.y - oy, Bz = p1.z - oz;
    float Cx = p2.x - ox, Cy = p2.y - oy, Cz = p2.z - oz;
    float akz = sel3(Ax, Ay, Az, w.kz), bkz = sel3(Bx, By, Bz, w.kz), ckz = sel3(Cx, Cy, Cz, w.kz);
    float ax = sel3(Ax, Ay, Az, w.kx) - w.sx * akz, ay = sel3(Ax, Ay, Az, w.ky) - w.sy * akz;
    float bx = sel3(Bx, By, Bz, w.kx) - w.sx * bkz, by = sel3(Bx, By, Bz, w.ky) - w.sy * bkz;
    float cx = sel3(Cx, Cy, Cz, w.kx) - w.sx * ckz, cy = sel3(Cx, Cy, Cz, w.ky) - w.sy * ckz;
    float U = watertight_edge(cx, cy, bx, by);
    float V = watertight_edge(ax, ay, cx, cy);
    float W = watertight_edge(bx, by, ax, ay);
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    float det = U + V + W;
    if (det == 0.0f) return false;
    float T = U * (w.sz * akz) + V * (w.sz * bkz) + W * (w.sz * ckz);
    float inv = 1.0f / det;
    t = T * inv;
    b1 = V * inv;
    b2 = W * inv;
    return true;
}

struct TraceRay {
    float ox, oy, oz, dx, dy, dz, tmin, tmax;
};

struct TraceResult {
    float t, b1, b2;
    int32_t face;    // -1: miss
    bool occluded;   // any-hit result
    bool overflow;   // the node-group stack filled: the ray ended before its traversal did
    uint32_t nodes;  // node records fetched
    uint32_t tris;   // triangle records tested
};

// Per-ray traversal state, so a ray can be advanced one node visit at a time (the persistent
// kernels refill a lane with a new ray as soon as its ray finishes).  The ray's triangle-test constants
// (WoopRay) are kept apart: the wave-cooperative kernels hold them in LDS.
struct TravState {
    float ox, oy, oz, tmin;
    float invx, invy, invz, ex, ey, ez;  // 1 / direction; e / |direction|, e the reference's box enlargement
    uint32_t oct;  // direction sign bits (x 1, y 2, z 4); the closest hit so far is res.t
    // Current node group: first child index and (imask << 8 | visit-order bits still to visit).
    uint32_t cur_base, cur_bits, node;
    TraceResult res;
};

// Sets the axes' box enlargements in units of the ray, e / |direction|.  Where one overflows (box scale 1 and
// an origin beyond 1e36) the infinity would take every box into that axis' slab, and a ray that enters
// nothing would visit the whole tree.  From an origin farther out on the axis than e (the scene, below 2^82,
// is nothing beside it) the slab is infinitely far ahead or behind instead, as without enlargement; within e
// of the scene it is indeed unbounded.
VT_HD void set_enlargement(TravState &st, float e) {
    st.ex = e * fabsf(st.invx);
    st.ey = e * fabsf(st.invy);
    st.ez = e * fabsf(st.invz);
    if (__builtin_expect(e > 3.4e30f, 0)) {  // 1 / direction is at most 1e8
        if (st.ex > 3.4028234664e38f && fabsf(st.ox) > 2.0f * e) st.ex = 0.0f;
        if (st.ey > 3.4028234664e38f && fabsf(st.oy) > 2.0f * e) st.ey = 0.0f;
        if (st.ez > 3.4028234664e38f && fabsf(st.oz) > 2.0f * e) st.ez = 0.0f;
    }
}

// The power of two by which a hierarchy's node boxes are scaled, and with them the ray's origin and its
// distances in the node test, given its max |coordinate|: 1 below 2^82.  The steps times 2^24 times
// 1 / direction, at most 1e8, must stay finite: unscaled they do up to steps of 2^76, and extents below 2^83
// have no larger ones.
// Above, 2^-64 keeps every product finite up to the largest extent a float holds; what it rounds away is
// below 2^-62, and the boxes are enlarged by at least 2^62 there.
VT_HD float box_scale(float root_max) { return root_max < 0x1p82f ? 1.0f : 0x1p-64f; }

// Starts a ray with box enlargement e (trav_init: the reference's e for a one-level hierarchy) in a
// hierarchy of box scale `scale`.
VT_HD void trav_init_e(TravState &st, const TraceRay &r, float e, float scale) {
    st.res.t = r.tmax;
    st.res.b1 = st.res.b2 = 0.0f;
    st.res.face = -1;
    st.res.occluded = false;
    st.res.overflow = false;
    st.res.nodes = st.res.tris = 0;
    st.ox = r.ox;
    st.oy = r.oy;
    st.oz = r.oz;
    st.tmin = r.tmin;
    // A component below 1e-8 in magnitude (the reference's parallel threshold) is taken as +-1e-8 with
    // its sign: the slab of a parallel axis then spans about -+1e8 x the origin's distance to its
    // planes -- the whole ray when the origin lies inside the (e-enlarged) slab, nothing reachable
    // when it lies at least e outside -- so no separate parallel test is needed.
    const uint32_t sx = float_to_bits(r.dx) >> 31, sy = float_to_bits(r.dy) >> 31, sz = float_to_bits(r.dz) >> 31;
    st.invx = 1.0f / (fabsf(r.dx) < 1e-8f ? (sx ? -1e-8f : 1e-8f) : r.dx);
    st.invy = 1.0f / (fabsf(r.dy) < 1e-8f ? (sy ? -1e-8f : 1e-8f) : r.dy);
    st.invz = 1.0f / (fabsf(r.dz) < 1e-8f ? (sz ? -1e-8f : 1e-8f) : r.dz);
    set_enlargement(st, e * scale);
    st.oct = sx | (sy << 1) | (sz << 2);
    st.cur_base = 0;
    st.cur_bits = 0;
    st.node = 0;
}

VT_HD float max_abs3(float x, float y, float z) { return fmaxf(fabsf(x), fmaxf(fabsf(y), fabsf(z))); }

// main.swift:1790-1792: e = 1.1920929e-6 (|origin|max + root max).
VT_HD void trav_init(TravState &st, const TraceRay &r, float root_max, float scale) {
    trav_init_e(st, r, 1.1920929e-6f * (max_abs3(r.ox, r.oy, r.oz) + root_max), scale);
}

// The object-space ray of an instance (main.swift:1634-1637 instance_ray): origin and direction by
// the rows of the world-to-object matrix, the direction not renormalised, so t keeps its meaning.
// Each dot product is evaluated as ((r0 x + r1 y) + r2 z) (+ r3), every operation rounded.
VT_HD TraceRay instance_ray(const float (&local)[3][4], const TraceRay &r, float tmax) {
#pragma clang fp contract(off)
    TraceRay l;
    l.ox = ((local[0][0] * r.ox + local[0][1] * r.oy) + local[0][2] * r.oz) + local[0][3];
    l.oy = ((local[1][0] * r.ox + local[1][1] * r.oy) + local[1][2] * r.oz) + local[1][3];
    l.oz = ((local[2][0] * r.ox + local[2][1] * r.oy) + local[2][2] * r.oz) + local[2][3];
    l.dx = (local[0][0] * r.dx + local[0][1] * r.dy) + local[0][2] * r.dz;
    l.dy = (local[1][0] * r.dx + local[1][1] * r.dy) + local[1][2] * r.dz;
    l.dz = (local[2][0] * r.dx + local[2][1] * r.dy) + local[2][2] * r.dz;
    l.tmin = r.tmin;
    l.tmax = tmax;
    return l;
}

// The traversal's node (see the head of this file) of a builder's Node8, both as five 16-byte words, in a
// hierarchy of box scale `scale`.
VT_HD void encode_node(const U4 (&n)[5], U4 (&o)[5], float scale) {
    const uint32_t imask = n[0].w >> 24;
    uint32_t half[3];
    for (int a = 0; a < 3; ++a) {
        // 2^(e - 127) as the builder's grid has it (0 for e = 0), times 2^24 and the box scale; 0 where
        // that is below the normal floats (a step below 2^-86 of a scene of 2^82).
        const int e = (int)((n[0].w >> (8 * a)) & 0xffu), x = e + 24 + (int)(float_to_bits(scale) >> 23) - 127;
        half[a] = e == 0 || x < 1 ? 0u : (uint32_t)(x < 255 ? x : 255) << 7;
    }
    uint32_t tri = 0;
    for (int s = 0; s < 8; ++s) {
        const uint32_t meta = ((s < 4 ? n[1].z : n[1].w) >> (8 * (s & 3))) & 0xffu;
        if (meta & 0x80u) continue;
        tri |= ((1u << (meta & 3u)) - 1u) << (3 * s);
    }
    o[0] = U4{float_to_bits(bits_to_float(n[0].x) * scale), float_to_bits(bits_to_float(n[0].y) * scale),
              float_to_bits(bits_to_float(n[0].z) * scale), half[0] | (half[1] << 16)};
    o[1] = U4{n[1].x, n[1].y, half[2] << 16, tri | (imask << 24)};
    const uint32_t lo[3][2] = {{n[2].x, n[2].y}, {n[2].z, n[2].w}, {n[3].x, n[3].y}};
    const uint32_t hi[3][2] = {{n[3].z, n[3].w}, {n[4].x, n[4].y}, {n[4].z, n[4].w}};
    for (int a = 0; a < 3; ++a) {
        uint32_t w[4];
        for (int k = 0; k < 4; ++k) {
            const int sh = 16 * (k & 1);
            const uint32_t l = lo[a][k >> 1] >> sh, h = hi[a][k >> 1] >> sh;
            w[k] = (l & 0xffu) | ((h & 0xffu) << 8) | ((l & 0xff00u) << 8) | ((h & 0xff00u) << 16);
        }
        o[2 + a] = U4{w[0], w[1], w[2], w[3]};
    }
}

// Two bytes of w as two fp16 numbers q 2^-24: bytes 0 and 2 (sel kPlaneLo) or 1 and 3 (kPlaneHi).
constexpr uint32_t kPlaneLo = 0x0c020c00u, kPlaneHi = 0x0c030c01u;
#if defined(__HIP_DEVICE_COMPILE__)
typedef _Float16 PlanePair __attribute__((ext_vector_type(2)));
__device__ __forceinline__ PlanePair plane_pair(uint32_t w, uint32_t sel) {
    return __builtin_bit_cast(PlanePair, __builtin_amdgcn_perm(w, w, sel));
}
__device__ __forceinline__ float plane(PlanePair p, int c) { return (float)p[c]; }
#else
typedef uint32_t PlanePair;
VT_HD PlanePair plane_pair(uint32_t w, uint32_t sel) { return (sel == kPlaneLo ? w : w >> 8) & 0x00ff00ffu; }
VT_HD float plane(PlanePair p, int c) { return (float)((p >> (16 * c)) & 0xffu) * 0x1p-24f; }
#endif

// Position of triangle bit p of a node with triangle bits tv (24 bits, tv's high byte ignored): the
// triangles below it.
VT_HD uint32_t tri_rank(uint32_t tv, uint32_t p) { return __builtin_popcount(tv & ((1u << p) - 1u)); }

// Node half of a step in a hierarchy of box scale `scale`: tests st.node's 8 child boxes, pushes the current
// group if inner children were hit, and moves st.node to the next node near to far.  Returns the triangles of the leaf children hit
// (trimask: bits of the node's triangle word tri_bits, whose first triangle is tri_base; triangle p of
// trimask is record tri_base + tri_rank(tri_bits, p)) and true when no node is left to visit (the
// triangles returned must still be tested).  The next node does not depend on those triangles, so
// testing them after the move gives the same result as testing them first.
//
// The kernels are bound by the instructions of this test.  Per child: six fused multiply-adds that read
// their plane as fp16 in place (v_fma_mix_f32), four min / max, a compare and a select, with half an or, for
// its bit of the hit mask (left to the compiler, which keeps two wait states between the compare and the
// instruction that reads its mask, as this hardware wants); per node: 24 byte permutes that pick the near and
// far planes by the ray's direction signs, and a few words' worth of bit arithmetic for the leaves' triangles
// and the visiting order.  Converting each byte (48 v_cvt_f32_ubyte), choosing near and far words per axis and
// handling each child's leaf or inner kind in a branch took about 290 vector and 140 scalar instructions
// a visit where this takes 200 and 40 (camera rays of the icosphere field 209 -> 168 us with the dealing
// of rays in trace.hip, bounce rays of the 10 M terrain 775 -> 630 us, 2 M rays each).
template <bool STATS, class Stack>
VT_HD bool trav_nodes(TravState &st, const U4 *__restrict__ nodes, float scale, Stack &stack, uint32_t &trimask,
                      uint32_t &tri_base, uint32_t &tri_bits) {
    const U4 *np = nodes + 5 * (size_t)st.node;
    const U4 w0 = np[0], w1 = np[1], w2 = np[2], w3 = np[3], w4 = np[4];
    if (STATS) ++st.res.nodes;
    // Slab distances of plane q of an axis: ((q s + p) - o -+ e) / d = q (s / d) + (p - o) / d -+ e / |d|,
    // one fma per plane, all in units of the box scale.  The near plane of an axis is its low plane for a
    // positive direction, its high plane otherwise.  The boxes are the reference's e-enlarged ones; the rounding
    // differs from the reference's (plane - o -+ e) / d by a few ulps of terms no larger than the scene, far inside the
    // enlargement, so no box the reference enters is culled.
    const float bx = bits_to_float(w0.w << 16) * st.invx, by = bits_to_float(w0.w & 0xffff0000u) * st.invy;
    const float bz = bits_to_float(w1.z) * st.invz;
    const float dx = __builtin_fmaf(-st.ox, scale, bits_to_float(w0.x)), dy = __builtin_fmaf(-st.oy, scale, bits_to_float(w0.y));
    const float dz = __builtin_fmaf(-st.oz, scale, bits_to_float(w0.z));
    const float tmin = st.tmin * scale, tmax = st.res.t * scale;
    const float nx = __builtin_fmaf(dx, st.invx, -st.ex), fx = __builtin_fmaf(dx, st.invx, st.ex);
    const float ny = __builtin_fmaf(dy, st.invy, -st.ey), fy = __builtin_fmaf(dy, st.invy, st.ey);
    const float nz = __builtin_fmaf(dz, st.invz, -st.ez), fz = __builtin_fmaf(dz, st.invz, st.ez);
    const uint32_t selx = (st.oct & 1u) ? kPlaneHi : kPlaneLo, sely = (st.oct & 2u) ? kPlaneHi : kPlaneLo;
    const uint32_t selz = (st.oct & 4u) ? kPlaneHi : kPlaneLo;
    constexpr uint32_t kOther = kPlaneLo ^ kPlaneHi;
    const uint32_t wx[4] = {w2.x, w2.y, w2.z, w2.w}, wy[4] = {w3.x, w3.y, w3.z, w3.w}, wz[4] = {w4.x, w4.y, w4.z, w4.w};
    uint32_t hit = 0;  // bit s: the box of slot s is hit (slots without a child are masked below)
#pragma unroll
    for (int k = 3; k >= 0; --k) {
        const PlanePair pnx = plane_pair(wx[k], selx), pfx = plane_pair(wx[k], selx ^ kOther);
        const PlanePair pny = plane_pair(wy[k], sely), pfy = plane_pair(wy[k], sely ^ kOther);
        const PlanePair pnz = plane_pair(wz[k], selz), pfz = plane_pair(wz[k], selz ^ kOther);
#pragma unroll
        for (int c = 1; c >= 0; --c) {
            const float tnx = __builtin_fmaf(plane(pnx, c), bx, nx), tfx = __builtin_fmaf(plane(pfx, c), bx, fx);
            const float tny = __builtin_fmaf(plane(pny, c), by, ny), tfy = __builtin_fmaf(plane(pfy, c), by, fy);
            const float tnz = __builtin_fmaf(plane(pnz, c), bz, nz), tfz = __builtin_fmaf(plane(pfz, c), bz, fz);
            const float tn = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, tmin));
            const float tf = fminf(fminf(tfx, tfy), fminf(tfz, tmax));
            hit |= tn <= tf ? 1u << (2 * k + c) : 0u;
        }
#if defined(__HIP_DEVICE_COMPILE__)
        __builtin_amdgcn_sched_barrier(0);  // a pair of slots at a time: fewer registers, one wave more per SIMD
#endif
    }
    // Each slot's bit spread to its three triangle bits.
    uint32_t spread = (hit | (hit << 8)) & 0x00f00fu;
    spread = (spread | (spread << 4)) & 0x0c30c3u;
    spread = (spread | (spread << 2)) & 0x249249u;
    tri_bits = w1.w;
    tri_base = w1.y;
    trimask = (spread * 7u) & w1.w;
    // Visiting order: slot s at bit s ^ oct, i.e. neighbours of 1, 2 and 4 swapped where the octant says.
    uint32_t order = hit & (w1.w >> 24);
    if (order) {
        if (st.cur_bits & 0xffu) {
            // The launcher sizes the stack to the tree's depth, so a full stack never occurs; if it did,
            // the ray stops (never an out-of-bounds access) and the kernel reports it.
            if (stack.full()) {
                st.res.overflow = true;
                trimask = 0;
                return true;
            }
            stack.push(st.cur_base, st.cur_bits);
        }
        const uint32_t s1 = st.oct & 1u, s2 = st.oct & 2u, s4 = st.oct & 4u;
        order = ((order & 0x55u) << s1) | ((order & 0xaau) >> s1);
        order = ((order & 0x33u) << s2) | ((order & 0xccu) >> s2);
        order = ((order & 0x0fu) << s4) | ((order & 0xf0u) >> s4);
        st.cur_base = w1.x;
        st.cur_bits = ((w1.w >> 16) & 0xff00u) | order;
    }
    if ((st.cur_bits & 0xffu) == 0u) {
        if (stack.empty()) return true;
        stack.pop(st.cur_base, st.cur_bits);
    }
    const uint32_t v = __builtin_ctz(st.cur_bits & 0xffu);
    st.cur_bits &= ~(1u << v);
    const uint32_t slot = v ^ st.oct;
    st.node = st.cur_base + __builtin_popcount((st.cur_bits >> 8) & ((1u << slot) - 1u));
    return false;
}

// A hit of the ray at t on face: the closest-hit rule (nearest t in [tmin, current t), equal t going
// to the smaller face index).  For the any-hit query any t in [tmin, tmax) ends the ray.
template <bool ANY>
VT_HD bool trav_accept(const TravState &st, float t, int32_t face) {
    if (ANY) return t >= st.tmin && t < st.res.t;  // still tmax: an any-hit query ends at its first hit
    return t >= st.tmin && (t < st.res.t || (t == st.res.t && st.res.face >= 0 && face < st.res.face));
}

// Triangle half of a step, one lane alone: tests the triangles trav_nodes returned.  Returns true
// when an any-hit query found a hit.
template <bool ANY, bool STATS>
VT_HD bool trav_tris(TravState &st, const WoopRay &w, const F4 *__restrict__ tris, uint32_t trimask, uint32_t tri_base,
                     uint32_t tri_bits) {
    while (trimask) {
        const uint32_t b = __builtin_ctz(trimask);
        trimask &= trimask - 1u;
        const F4 *tp = tris + 3 * (size_t)(tri_base + tri_rank(tri_bits, b));
        const F4 p0 = tp[0], p1 = tp[1], p2 = tp[2];
        if (STATS) ++st.res.tris;
        float t, b1, b2;
        if (!woop_triangle(w, st.ox, st.oy, st.oz, p0, p1, p2, t, b1, b2)) continue;
        const int32_t face = (int32_t)float_to_bits(p0.w);
        if (!trav_accept<ANY>(st, t, face)) continue;
        if (ANY) {
            st.res.occluded = true;
            return true;
        }
        st.res.t = t;
        st.res.b1 = b1;
        st.res.b2 = b2;
        st.res.face = face;
    }
    return false;
}

// One step of one ray: a node visit and the triangles of the leaves it hits.  Returns true when the
// ray is finished (result in st.res).
template <bool ANY, bool STATS, class Stack>
VT_HD bool trav_step(TravState &st, const WoopRay &w, const U4 *__restrict__ nodes, float scale,
                     const F4 *__restrict__ tris, Stack &stack) {
    uint32_t trimask, tri_base, tri_bits;
    const bool done = trav_nodes<STATS>(st, nodes, scale, stack, trimask, tri_base, tri_bits);
    if (trav_tris<ANY, STATS>(st, w, tris, trimask, tri_base, tri_bits)) return true;
    return done;
}

// Traverses one ray.  nodes: encoded nodes as 5 U4 each; tris: TriRecord as 3 F4 each.
template <bool ANY, bool STATS, class Stack>
VT_HD TraceResult traverse(const U4 *__restrict__ nodes, const F4 *__restrict__ tris, float root_max, float scale,
                           const TraceRay &r, Stack &stack) {
    TravState st;
    trav_init(st, r, root_max, scale);
    const WoopRay w = woop_ray(r.dx, r.dy, r.dz);
    while (!trav_step<ANY, STATS>(st, w, nodes, scale, tris, stack)) {
    }
    return st.res;
}

}  // namespace vt
