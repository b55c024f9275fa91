// The traversal of csrc/traverse8.h, one ray at a time, compiled for the host by tests/test_traversal_host.py.
#include <cstdint>
#include <vector>

#include "traverse8.h"

namespace {
struct Stack {
    std::vector<uint32_t> base, bits;
    bool full() const { return base.size() >= 24; }
    bool empty() const { return base.empty(); }
    void push(uint32_t b, uint32_t m) {
        base.push_back(b);
        bits.push_back(m);
    }
    void pop(uint32_t &b, uint32_t &m) {
        b = base.back();
        m = bits.back();
        base.pop_back();
        bits.pop_back();
    }
};
}  // namespace

// nodes: the builder's Node8 records, encoded here; rays: [8][n].  visits: node records read, triangles tested.
extern "C" void closest(const void *nodes, uint32_t node_count, const void *tris, float root_max, const float *rays, uint32_t n,
                        float *t, float *b1, float *b2, int32_t *face, uint8_t *occluded, uint64_t *visits) {
    const float scale = vt::box_scale(root_max);
    std::vector<vt::U4> encoded(5 * (size_t)node_count);
    for (uint32_t i = 0; i < node_count; ++i) {
        vt::U4 in[5], out[5];
        for (int k = 0; k < 5; ++k) in[k] = static_cast<const vt::U4 *>(nodes)[5 * (size_t)i + k];
        vt::encode_node(in, out, scale);
        for (int k = 0; k < 5; ++k) encoded[5 * (size_t)i + k] = out[k];
    }
    const vt::F4 *records = static_cast<const vt::F4 *>(tris);
    visits[0] = visits[1] = 0;
    for (uint32_t i = 0; i < n; ++i) {
        const vt::TraceRay r{rays[i], rays[n + i], rays[2 * (size_t)n + i], rays[3 * (size_t)n + i], rays[4 * (size_t)n + i],
                             rays[5 * (size_t)n + i], rays[6 * (size_t)n + i], rays[7 * (size_t)n + i]};
        Stack s;
        const vt::TraceResult c = vt::traverse<false, true>(encoded.data(), records, root_max, scale, r, s);
        t[i] = c.t;
        b1[i] = c.b1;
        b2[i] = c.b2;
        face[i] = c.face;
        visits[0] += c.nodes;
        visits[1] += c.tris;
        Stack any;
        occluded[i] = vt::traverse<true, false>(encoded.data(), records, root_max, scale, r, any).occluded ? 1 : 0;
    }
}
