// nrc.hip -- gfx950 kernels of the learned radiance cache (nrc.h): fused encode + MLP inference,
// fused forward + backward with gradient accumulation, Adam with a moving average of the weights.
//
// All matrix products run on the matrix cores (v_mfma_f32_16x16x32_bf16: bf16 operands, fp32
// accumulation).  The weights are the A operand and the activations the B operand, so a layer's output
// tile is already the next layer's operand and activations stay in registers, forward and backward; for
// the weight gradients, products over the samples, training also keeps the activations and their
// gradients of a block's 128 samples in LDS, transposed.  The bf16 network (60 KB) sits in LDS for the
// life of a block.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nrc.h"

namespace vt {
namespace {

typedef short s4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kOffW2 = kNrcW1, kOffW3 = kOffW2 + kNrcWh, kOffW4 = kOffW3 + kNrcWh, kOffW5 = kOffW4 + kNrcWh;

__device__ __forceinline__ uint16_t to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float from_bf16(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ __forceinline__ f4v mfma(s4v a, s4v b, f4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
// Input k of query q: inputs are [q][11] (stride 0) or [11][stride].
__device__ __forceinline__ float query_input(const float *inputs, uint32_t stride, uint32_t q, int k) {
    return stride ? inputs[(size_t)k * stride + q] : inputs[(size_t)q * kNrcInputs + k];
}

// ---------------------------------------------------------------- inference
// v_mfma_f32_16x16x32_bf16 (gfx950: twice the K of the 16x16x16 form for the same issue cost).  The
// weights are the A operand and the activations the B operand (D^T = W . X^T).  Lane l = r + 16 g
// holds A row r / B column r and the eight k of group g; the sum over k does not depend on which
// hardware k a (group, element) pair stands for, as long as A and B agree, so each layer's inputs are
// numbered for the convenience of the data:
//   layer 1: k-step ks, group g carries feature quad Q = 9 g + ks, element e feature 8 Q + e of the
//            network's order (24 per input: sin and cos of bands 0..11), i.e. bands 4 (ks % 3) ..
//            4 (ks % 3) + 3 of input 3 g + ks / 3.  A lane thus needs three inputs of its query, and
//            the band group of every step is a compile-time constant.  Quads 33 .. 35 (lanes of
//            group 3 in steps 6 .. 8) have zero weights: the constant feature 264 is the bias,
//            which starts the accumulation instead (fp32 copy of its bf16 weights);
//   layers 2-5: k-step ks, group g, element e is input neuron 32 ks + 16 (e / 4) + 4 g + e % 4, the
//            neurons the lane already holds in its output tiles 2 ks and 2 ks + 1 (D layout: lane l
//            holds rows 4 g + j of a tile), so activations never leave registers.
// The LDS copy of each weight row is stored in that k order.  A wave handles 16 T queries per pass
// and loads the next pass's inputs while it computes the current one.
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef short s8v __attribute__((ext_vector_type(8)));

constexpr int kK1 = 288;                           // layer-1 k: 272 features padded to 9 steps of 32
constexpr int kW1Pitch = kK1 + 8, kWhPitch = 64 + 8;  // bf16; rows 592 / 144 bytes apart: the 16 rows
                                                      // a quarter-wave reads fall in distinct banks
constexpr int kLdsW1 = 0, kLdsW2 = kLdsW1 + kNrcHidden * kW1Pitch, kLdsW3 = kLdsW2 + kNrcHidden * kWhPitch,
              kLdsW4 = kLdsW3 + kNrcHidden * kWhPitch, kLdsW5 = kLdsW4 + kNrcHidden * kWhPitch;
constexpr int kLdsBias = kLdsW5 + kNrcOutPad * kWhPitch;          // 64 floats
constexpr int kInferLds = kLdsBias * 2 + kNrcHidden * 4;          // 68,096 bytes
constexpr int kInferTiles = 2;

// Input neuron of position p (0..63) of a permuted hidden-layer row.
__host__ __device__ constexpr int hidden_input(int p) {
    return 32 * (p >> 5) + 16 * ((p & 7) >> 2) + 4 * ((p >> 3) & 3) + (p & 3);
}
// The weight copy moves positions 8 k .. 8 k + 7 as two runs of four inputs.
constexpr bool hidden_runs_agree() {
    for (int p = 0; p < 64; ++p)
        if (hidden_input(p) != 32 * (p >> 5) + 4 * ((p >> 3) & 3) + 16 * ((p & 7) >> 2) + (p & 3)) return false;
    return true;
}
static_assert(hidden_runs_agree(), "hidden-layer weight permutation");

// A thread's share of the network on its way into LDS in the permuted orders: all its loads are issued
// before its stores.  Layer 1: position 32 ks + 8 g + e of a row holds feature 8 (9 g + ks) + e (below
// 264), else 0; the weights of feature 264 (the constant 1) are the bias, as floats.  Hidden layers:
// positions 8 k .. 8 k + 7 of a row hold inputs b .. b + 3 and b + 16 .. b + 19, b = 32 (k / 4) + 4 (k % 4).
template <int kThreads>
struct FirstLayerCopy {
    static constexpr int kChunks = kNrcHidden * (kK1 / 8), kSteps = (kChunks + kThreads - 1) / kThreads;
    uint4 v[kSteps];
    __device__ __forceinline__ void load(const uint16_t *src) {
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const int c = threadIdx.x + i * kThreads, row = c / (kK1 / 8), chunk = c - row * (kK1 / 8);
            const int q = 9 * (chunk & 3) + (chunk >> 2);
            v[i] = make_uint4(0u, 0u, 0u, 0u);
            if (c < kChunks && q < 33) v[i] = *reinterpret_cast<const uint4 *>(src + row * kNrcFeatures + 8 * q);
        }
    }
    __device__ __forceinline__ void store(uint16_t *w) const {
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const int c = threadIdx.x + i * kThreads, row = c / (kK1 / 8), chunk = c - row * (kK1 / 8);
            if (c < kChunks) *reinterpret_cast<uint4 *>(w + kLdsW1 + row * kW1Pitch + 8 * chunk) = v[i];
        }
    }
};
template <int kThreads>
struct HiddenCopy {
    static constexpr int kChunks = (3 * kNrcHidden + kNrcOutPad) * 8, kSteps = (kChunks + kThreads - 1) / kThreads;
    uint4 v[kSteps];
    float bias;
    __device__ __forceinline__ void load(const uint16_t *src) {
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const int c = threadIdx.x + i * kThreads, row = c >> 3, k = c & 7;
            if (c < kChunks) {
                const uint16_t *r = src + kNrcW1 + row * 64 + 32 * (k >> 2) + 4 * (k & 3);
                const uint2 lo = *reinterpret_cast<const uint2 *>(r), hi = *reinterpret_cast<const uint2 *>(r + 16);
                v[i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
            }
        }
        bias = threadIdx.x < kNrcHidden ? from_bf16(src[threadIdx.x * kNrcFeatures + 264]) : 0.0f;
    }
    __device__ __forceinline__ void store(uint16_t *w) const {
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const int c = threadIdx.x + i * kThreads;
            if (c < kChunks) *reinterpret_cast<uint4 *>(w + kLdsW2 + (c >> 3) * kWhPitch + 8 * (c & 7)) = v[i];
        }
        if (threadIdx.x < kNrcHidden) reinterpret_cast<float *>(w + kLdsBias)[threadIdx.x] = bias;
    }
    // W2..W4 transposed into wt: row `in` of layer l holds W[hidden_input(p)][in] at position p.
    __device__ __forceinline__ void store_transposed(uint16_t *wt) const {
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const int c = threadIdx.x + i * kThreads, row = c >> 3, k = c & 7, layer = row >> 6, out = row & 63;
            if (c >= 3 * kNrcHidden * 8) break;
            const int p = 32 * (out >> 5) + 8 * ((out >> 2) & 3) + 4 * ((out >> 4) & 1) + (out & 3);
            uint16_t *t = wt + (layer * kNrcHidden + 32 * (k >> 2) + 4 * (k & 3)) * kWhPitch + p;
            const uint32_t u[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) t[(16 * (e >> 2) + (e & 3)) * kWhPitch] = (uint16_t)(u[e >> 1] >> (16 * (e & 1)));
        }
    }
};

__device__ __forceinline__ f4v mfma32(bf8v a, bf8v b, f4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ bf8v lds8(const uint16_t *p) { return *reinterpret_cast<const bf8v *>(p); }

// Features of bands b0 .. b0 + 3 of input value x: sin and cos of pi 2^b x per band, as bf16.
// 2^(b-1) x is exact in fp32 and so is its fractional part, so the hardware sine and cosine
// (argument in turns) work on the exactly reduced angle.
template <int B0>
__device__ __forceinline__ bf8v band_quad(float x) {
    bf8v r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float t = __builtin_amdgcn_fractf(x * __builtin_ldexpf(1.0f, B0 + k - 1));
        r[2 * k] = (__bf16)__builtin_amdgcn_sinf(t);
        r[2 * k + 1] = (__bf16)__builtin_amdgcn_cosf(t);
    }
    return r;
}

// relu and bf16 of output tiles 2 ks and 2 ks + 1: the B operand of the next layer's k-step ks.
// Rounded first, then the relu as a signed 16-bit max with 0 (a bf16 with its sign bit set is a
// negative short): the same bits as rounding the relu.
typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
typedef short s2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t relu_bf16x2(float a, float b) {
    const s2v v = __builtin_bit_cast(s2v, __builtin_convertvector(f2v{a, b}, bf2v));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(v, s2v{0, 0}));
}
__device__ __forceinline__ bf8v relu_pair(f4v lo, f4v hi) {
    const uint4 u = {relu_bf16x2(lo[0], lo[1]), relu_bf16x2(lo[2], lo[3]), relu_bf16x2(hi[0], hi[1]), relu_bf16x2(hi[2], hi[3])};
    return __builtin_bit_cast(bf8v, u);
}

// One hidden layer: 64 neurons x 16 T queries in (acc, D layout) -> W . relu(acc) in acc.
template <int T>
__device__ __forceinline__ void hidden_layer(const uint16_t *w, f4v (&acc)[4][T], int r, int g) {
    bf8v h[2][T];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int t = 0; t < T; ++t) h[ks][t] = relu_pair(acc[2 * ks][t], acc[2 * ks + 1][t]);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const bf8v a = lds8(w + (16 * m + r) * kWhPitch + 32 * ks + 8 * g);
#pragma unroll
            for (int t = 0; t < T; ++t) acc[m][t] = mfma32(a, h[ks][t], ks ? acc[m][t] : f4v{0.0f, 0.0f, 0.0f, 0.0f});
        }
}

// Inputs 3 g .. 3 g + 2 (capped at the last) of query 16 T p + 16 t + r, zeros past n.
template <int T>
__device__ __forceinline__ void load_inputs(float (&x)[T][3], const float *inputs, uint32_t stride, uint32_t n, uint32_t p,
                                            int r, int g) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint64_t q = (uint64_t)p * (16 * T) + 16 * t + r;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int i = min(3 * g + c, kNrcInputs - 1);
            const float v = query_input(inputs, stride, (uint32_t)min(q, (uint64_t)n - 1), i);
            x[t][c] = q < n ? v : 0.0f;
        }
    }
}

// Layer-1 steps 3 c .. 3 c + 2 (input slot c of each query, band groups 0, 1, 2); the first
// accumulates onto the bias.
template <int T, bool kFirst>
__device__ __forceinline__ void layer1_steps(const uint16_t *lds, f4v (&acc)[4][T], const f4v (&bias)[4],
                                             const float (&x)[T][3], int c, int r, int g) {
    float xc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) xc[t] = kFirst ? x[t][0] : c == 1 ? x[t][1] : x[t][2];
#pragma unroll
    for (int bg = 0; bg < 3; ++bg) {
        const int ks = 3 * c + bg;
        bf8v a[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = lds8(lds + kLdsW1 + (16 * m + r) * kW1Pitch + 32 * ks + 8 * g);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const bf8v bv = bg == 0 ? band_quad<0>(xc[t]) : bg == 1 ? band_quad<4>(xc[t]) : band_quad<8>(xc[t]);
#pragma unroll
            for (int m = 0; m < 4; ++m) acc[m][t] = mfma32(a[m], bv, kFirst && bg == 0 ? bias[m] : acc[m][t]);
        }
    }
}

// Blocks of kInferBlock lanes share one LDS copy of the network.
constexpr int kInferBlock = 512, kInferWaves = kInferBlock / 64;
template <int T>
__global__ __launch_bounds__(kInferBlock) void nrc_infer_kernel(const uint16_t *wsrc, const float *inputs, uint32_t stride,
                                                                uint32_t n, float *out, const uint32_t *count) {
    extern __shared__ __align__(16) uint16_t lds[];
    if (count) n = min(n, *count);
    if (n == 0) return;
    {
        FirstLayerCopy<kInferBlock> first;
        HiddenCopy<kInferBlock> hidden;
        first.load(wsrc);
        hidden.load(wsrc);
        first.store(lds);
        hidden.store(lds);
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const uint32_t passes = (n + 16 * T - 1) / (16 * T), step = gridDim.x * kInferWaves;
    float xn[T][3];
    uint32_t p = blockIdx.x * kInferWaves + wave;
    load_inputs<T>(xn, inputs, stride, n, p, r, g);
    for (; p < passes; p += step) {
        float x[T][3];
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int c = 0; c < 3; ++c) x[t][c] = xn[t][c];
        load_inputs<T>(xn, inputs, stride, n, p + step, r, g);
        // Layer 1: steps ks = 3 c + bg take input slot c, bands 4 bg .. 4 bg + 3, from the bias.
        f4v acc[4][T], bias[4];
        {
            // Read each pass (an opaque zero offset keeps the compiler from holding the bias in
            // registers across the loop, which it needs for the hidden layers' weights).
            int zero = 0;
            asm volatile("" : "+v"(zero));
            const float *bl = reinterpret_cast<const float *>(lds + kLdsBias) + zero;
#pragma unroll
            for (int m = 0; m < 4; ++m) bias[m] = *reinterpret_cast<const f4v *>(bl + 16 * m + 4 * g);
        }
        layer1_steps<T, true>(lds, acc, bias, x, 0, r, g);
#pragma unroll 1
        for (int c = 1; c < 3; ++c) layer1_steps<T, false>(lds, acc, bias, x, c, r, g);
        hidden_layer<T>(lds + kLdsW2, acc, r, g);
        hidden_layer<T>(lds + kLdsW3, acc, r, g);
        hidden_layer<T>(lds + kLdsW4, acc, r, g);
        f4v y[T];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const bf8v a = lds8(lds + kLdsW5 + r * kWhPitch + 32 * ks + 8 * g);
#pragma unroll
            for (int t = 0; t < T; ++t)
                y[t] = mfma32(a, relu_pair(acc[2 * ks][t], acc[2 * ks + 1][t]), ks ? y[t] : f4v{0.0f, 0.0f, 0.0f, 0.0f});
        }
        // Lanes 0..15 hold outputs 0..3 of query 16 t + l.
        if (g == 0) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const uint64_t q = (uint64_t)p * (16 * T) + 16 * t + r;
                if (q < n) *reinterpret_cast<float4 *>(out + 4 * q) = make_float4(y[t][0], y[t][1], y[t][2], y[t][3]);
            }
        }
    }
}

// ---------------------------------------------------------------- training (forward + backward)
// A block of 8 waves takes 128 samples at a time, 16 a wave.  Forward and backward chains are the
// inference kernel's: each layer's D tile (rows: neurons, columns: the wave's samples) is rounded to bf16
// and is the next product's B operand, forward with the rows of W as A, backward with the rows of its
// transpose.  Only the weight gradients cross waves: dW = d^T a sums over all samples of the block, so
// activations a and their gradients d are also stored transposed in LDS ([neuron][sample], the k index of
// that product contiguous), and the 120 16 x 16 gradient tiles are dealt out 15 to a wave, accumulated
// in registers over all the block's samples and written once, as the block's partial sums.  The first
// layer's a (264 encodings) is evaluated again where its tiles are needed instead of stored: its tile's
// columns are all sines or all cosines (column r of tile t < 16 is feature 32 (t / 2) + 2 r + t % 2).
// nrc_adam_kernel adds the blocks' partial sums in a fixed order, so a step's result does not depend on
// how the blocks were scheduled.
//
// Bound by LDS traffic and the encodings' sines at the sizes a frame trains on (16384 records: 128 blocks
// on half the CUs, two waves a SIMD): a step takes 22.5 us, a quarter of it reading the weights the last
// step's Adam wrote; the kernel stands at its 256 registers and spills 11 (48 bytes of scratch a lane).  With
// one fp32 atomic per weight and block (7.9M a step), 64 samples a block of 4 waves and 2-byte strided LDS
// reads for the weight gradients it took 57.6 us.
constexpr int kTrainBlock = 512, kTrainWaves = kTrainBlock / 64, kTrainSamples = 16 * kTrainWaves;
constexpr int kTileSlots = 15;                        // gradient tiles per wave
constexpr int kTPitch = kTrainSamples + 8;            // bf16 per transposed row: 272 bytes, 16 rows of
                                                      // 16-byte reads fall in distinct banks
constexpr int kTBuf = kNrcHidden * kTPitch;           // one transposed 64 x 128 matrix
constexpr int kXPitch = kTrainSamples + 4;            // floats per input row
// LDS (bf16 units): the inference kernel's weight copy, whose first-layer part the transposed
// activations 3 and 4 take over once every wave is past layer 1; the transposed W2..W4; activations 1
// and 2 and the last layer's gradients, transposed; the output gradients; features 256 .. 263; the inputs
// (floats).
constexpr int kTrWt = kInferLds / 2, kTrA1 = kTrWt + 3 * kNrcHidden * kWhPitch, kTrA2 = kTrA1 + kTBuf,
              kTrD4 = kTrA2 + kTBuf, kTrDy = kTrD4 + kTBuf, kTrF = kTrDy + kNrcOut * kTPitch, kTrX = kTrF + 8 * kTPitch;
constexpr int kTrainLds = kTrX * 2 + kNrcInputs * kXPitch * 4;
static_assert(2 * kTBuf <= kNrcHidden * kW1Pitch, "activations 3 and 4 fit the first layer's weights");
static_assert(kTrainLds <= 160 * 1024 && kTrX % 8 == 0 && kTrWt % 8 == 0, "LDS layout");
static_assert(kTileSlots * kTrainWaves * 256 == kNrcParams, "every gradient tile has an owner");

// The parameter that element j of lane l of gradient tile `slot` of wave w is the gradient of.
__device__ __forceinline__ int tile_param(int w, int slot, int l, int j) {
    const int r = l & 15, row = 4 * (l >> 4) + j;
    if (slot < 8) return (16 * (slot & 3) + row) * kNrcFeatures + 32 * ((w + 2 * (slot & 4)) >> 1) + 2 * r + (w & 1);
    if (slot < 14) {
        const int layer = (slot - 8) >> 1, it = 2 * (w & 1) + (slot & 1);
        return kOffW2 + layer * kNrcWh + (16 * (w >> 1) + row) * kNrcHidden + 16 * it + r;
    }
    return w < 4 ? (16 * w + row) * kNrcFeatures + 256 + r : kOffW5 + row * kNrcHidden + 16 * (w - 4) + r;
}

// relu, rounded to bf16, of output tiles 2 ks and 2 ks + 1 (a NaN becomes 0, as fmaxf makes it).
__device__ __forceinline__ bf8v relu_frag(f4v lo, f4v hi) {
    bf8v h;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        h[j] = (__bf16)fmaxf(lo[j], 0.0f);
        h[4 + j] = (__bf16)fmaxf(hi[j], 0.0f);
    }
    return h;
}
// The gradients in tiles 2 ks and 2 ks + 1 where the activation they belong to is positive, else 0.
__device__ __forceinline__ bf8v mask_frag(f4v lo, f4v hi, bf8v act) {
    bf8v d;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        d[j] = (__bf16)((float)act[j] > 0.0f ? lo[j] : 0.0f);
        d[4 + j] = (__bf16)((float)act[4 + j] > 0.0f ? hi[j] : 0.0f);
    }
    return d;
}
// Column `col` of a transposed matrix from a wave's operand fragments (neuron order of hidden_input).
__device__ __forceinline__ void store_transposed(uint16_t *t, const bf8v (&f)[2], int col, int g) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const s8v bits = __builtin_bit_cast(s8v, f[ks]);
#pragma unroll
        for (int e = 0; e < 8; ++e) t[(32 * ks + 16 * (e >> 2) + 4 * g + (e & 3)) * kTPitch + col] = (uint16_t)bits[e];
    }
}
// acc[m] = rows 16 m .. 16 m + 15 of w (pitch kWhPitch, k in hidden_input order) times the fragments.
__device__ __forceinline__ void dense64(const uint16_t *w, const bf8v (&in)[2], f4v (&acc)[4], int r, int g) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int m = 0; m < 4; ++m)
            acc[m] = mfma32(lds8(w + (16 * m + r) * kWhPitch + 32 * ks + 8 * g), in[ks],
                            ks ? acc[m] : f4v{0.0f, 0.0f, 0.0f, 0.0f});
}
// acc += the product of 16 rows of each transposed matrix over the block's samples.
__device__ __forceinline__ void grad_tile(f4v &acc, const uint16_t *d_rows, const uint16_t *a_rows, int r, int g) {
#pragma unroll
    for (int ks = 0; ks < kTrainSamples / 32; ++ks)
        acc = mfma32(lds8(d_rows + r * kTPitch + 32 * ks + 8 * g), lds8(a_rows + r * kTPitch + 32 * ks + 8 * g), acc);
}

// The samples [offset, offset + n) of a slice (NrcSlice), n capped by the launch's n.
__device__ __forceinline__ uint32_t slice_bounds(const NrcSlice &sl, uint32_t n, uint32_t &offset) {
    offset = 0;
    if (!sl.count) return n;
    const uint32_t c = min(*sl.count, sl.limit);
    const uint32_t per = min((c + sl.parts - 1) / sl.parts, n);
    offset = sl.part * per;
    return offset < c ? min(per, c - offset) : 0u;
}

// Partial gradients of block b: partials[b][wave][slot][lane][4].
__global__ __launch_bounds__(kTrainBlock) void nrc_backward_kernel(const uint16_t *wsrc, const float *inputs, uint32_t stride,
                                                                   const float *targets, uint32_t n, float norm,
                                                                   float4 *partials, float *loss_sum, NrcSlice slice) {
    extern __shared__ __align__(16) uint16_t lds[];
    uint32_t offset;
    n = slice_bounds(slice, n, offset);
    const uint32_t groups = (n + kTrainSamples - 1) / kTrainSamples;
    if (blockIdx.x >= groups) return;
    inputs += stride ? (size_t)offset : (size_t)offset * kNrcInputs;
    targets += (size_t)offset * kNrcOut;
    if (!(norm > 0.0f)) norm = (float)n * kNrcOut;
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), col = 16 * w + r;  // w: a scalar
    uint16_t *a3 = lds + kLdsW1, *a4 = a3 + kTBuf, *a1 = lds + kTrA1, *a2 = lds + kTrA2, *d4t = lds + kTrD4;
    uint16_t *dyt = lds + kTrDy, *ft = lds + kTrF;
    float *xs = reinterpret_cast<float *>(lds + kTrX);
    f4v grad[kTileSlots] = {};
    float lsum = 0.0f;
    for (uint32_t group = blockIdx.x; group < groups; group += gridDim.x) {
        const uint32_t q0 = group * kTrainSamples, q = q0 + (uint32_t)col;
        constexpr int kXSteps = (kNrcInputs * kTrainSamples + kTrainBlock - 1) / kTrainBlock;
        float xv[kXSteps];
#pragma unroll
        for (int k = 0; k < kXSteps; ++k) {
            const int idx = threadIdx.x + k * kTrainBlock;
            const uint32_t qc = q0 + (uint32_t)(stride ? idx % kTrainSamples : idx / kNrcInputs);
            const int i = stride ? idx / kTrainSamples : idx % kNrcInputs;
            xv[k] = idx < kNrcInputs * kTrainSamples && qc < n ? query_input(inputs, stride, qc, i) : 0.0f;
        }
        float target[kNrcOut] = {};
        if (g == 0 && q < n) {
#pragma unroll
            for (int j = 0; j < kNrcOut; ++j) target[j] = targets[(size_t)q * kNrcOut + j];
        }
        {
            // The first layer's weights each time: the last group's activations overwrote them.
            FirstLayerCopy<kTrainBlock> first;
            first.load(wsrc);
            if (group == blockIdx.x) {
                HiddenCopy<kTrainBlock> hidden;
                hidden.load(wsrc);
                hidden.store(lds);
                hidden.store_transposed(lds + kTrWt);
            }
            first.store(lds);
        }
#pragma unroll
        for (int k = 0; k < kXSteps; ++k) {
            const int idx = threadIdx.x + k * kTrainBlock;
            const int i = stride ? idx / kTrainSamples : idx % kNrcInputs, c = stride ? idx % kTrainSamples : idx / kNrcInputs;
            if (idx < kNrcInputs * kTrainSamples) xs[i * kXPitch + c] = xv[k];
        }
        __syncthreads();
        // Forward: h[k] is the wave's operand fragment of activations k + 1.
        bf8v h[4][2];
        f4v acc[4];
        {
            const float *bl = reinterpret_cast<const float *>(lds + kLdsBias);
#pragma unroll
            for (int m = 0; m < 4; ++m) acc[m] = *reinterpret_cast<const f4v *>(bl + 16 * m + 4 * g);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float x = xs[min(3 * g + c, kNrcInputs - 1) * kXPitch + col];
#pragma unroll
                for (int bg = 0; bg < 3; ++bg) {
                    const bf8v bv = bg == 0 ? band_quad<0>(x) : bg == 1 ? band_quad<4>(x) : band_quad<8>(x);
                    if (c == 1 && bg == 2 && g == 3) {  // bands 8 .. 11 of input 10
                        const s8v bits = __builtin_bit_cast(s8v, bv);
#pragma unroll
                        for (int e = 0; e < 8; ++e) ft[e * kTPitch + col] = (uint16_t)bits[e];
                    }
#pragma unroll
                    for (int m = 0; m < 4; ++m)
                        acc[m] = mfma32(lds8(lds + kLdsW1 + (16 * m + r) * kW1Pitch + 32 * (3 * c + bg) + 8 * g), bv, acc[m]);
                }
            }
        }
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            h[l][0] = relu_frag(acc[0], acc[1]);
            h[l][1] = relu_frag(acc[2], acc[3]);
            if (l == 0) __syncthreads();  // every wave is past the first layer's weights
            if (l < 3) dense64(lds + kLdsW2 + l * kNrcHidden * kWhPitch, h[l], acc, r, g);
            store_transposed(l == 0 ? a1 : l == 1 ? a2 : l == 2 ? a3 : a4, h[l], col, g);
        }
        f4v y = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) y = mfma32(lds8(lds + kLdsW5 + r * kWhPitch + 32 * ks + 8 * g), h[3][ks], y);
        // d loss / d y (relative L2, y constant in the denominator): lanes 0..15 hold outputs 0..3 of
        // their sample, the other lanes the unused outputs.
        s4v dy = {0, 0, 0, 0};
        if (g == 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float d = 0.0f;
                if (q < n) {
                    const float den = y[j] * y[j] + 0.01f;
                    d = 2.0f * (y[j] - target[j]) / den / norm;
                    lsum += (y[j] - target[j]) * (y[j] - target[j]) / den;
                }
                dy[j] = (short)to_bf16(d);
                dyt[j * kTPitch + col] = to_bf16(d);
            }
        }
        // Backward: d[k] is the operand fragment of the gradients of activations k + 1.  The output layer
        // has four live rows: its transpose is the A operand of one 16-k product.
        bf8v d[4][2];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            s4v a = {0, 0, 0, 0};
            if (g == 0) {
                const uint16_t *w5 = lds + kLdsW5 + 32 * (m >> 1) + 8 * (r >> 2) + 4 * (m & 1) + (r & 3);
#pragma unroll
                for (int j = 0; j < 4; ++j) a[j] = (short)w5[j * kWhPitch];
            }
            acc[m] = mfma(a, dy, f4v{0.0f, 0.0f, 0.0f, 0.0f});
        }
        d[3][0] = mask_frag(acc[0], acc[1], h[3][0]);
        d[3][1] = mask_frag(acc[2], acc[3], h[3][1]);
        store_transposed(d4t, d[3], col, g);
#pragma unroll
        for (int l = 2; l >= 0; --l) {
            dense64(lds + kTrWt + l * kNrcHidden * kWhPitch, d[l + 1], acc, r, g);
            d[l][0] = mask_frag(acc[0], acc[1], h[l][0]);
            d[l][1] = mask_frag(acc[2], acc[3], h[l][1]);
        }
        __syncthreads();
        // Output layer (rows 4..15 of dy are 0), then layer 4.
        if (w >= 4) {
#pragma unroll
            for (int ks = 0; ks < kTrainSamples / 32; ++ks) {
                const bf8v zero = {};
                const bf8v a = r < kNrcOut ? lds8(dyt + r * kTPitch + 32 * ks + 8 * g) : zero;
                grad[14] = mfma32(a, lds8(a4 + (16 * (w - 4) + r) * kTPitch + 32 * ks + 8 * g), grad[14]);
            }
        }
        const int ot = 16 * (w >> 1) * kTPitch, it = 32 * (w & 1) * kTPitch;
        grad_tile(grad[12], d4t + ot, a3 + it, r, g);
        grad_tile(grad[13], d4t + ot, a3 + it + 16 * kTPitch, r, g);
        __syncthreads();
        // Activations 4 and 3 and d4 are spent: their rooms take d3, d1 and d2.
        store_transposed(a4, d[2], col, g);
        store_transposed(d4t, d[1], col, g);
        store_transposed(a3, d[0], col, g);
        __syncthreads();
        grad_tile(grad[10], a4 + ot, a2 + it, r, g);
        grad_tile(grad[11], a4 + ot, a2 + it + 16 * kTPitch, r, g);
        grad_tile(grad[8], d4t + ot, a1 + it, r, g);
        grad_tile(grad[9], d4t + ot, a1 + it + 16 * kTPitch, r, g);
        // First layer: feature tiles w and w + 8 (sines for even w, cosines for odd) against all four
        // output tiles; waves 0..3 also one output tile each of features 256 .. 271.
#pragma unroll
        for (int ks = 0; ks < kTrainSamples / 32; ++ks) {
            const uint16_t *dk = a3 + r * kTPitch + 32 * ks + 8 * g;
            bf8v da[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) da[m] = lds8(dk + 16 * m * kTPitch);
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int f = 32 * ((w + 8 * half) >> 1) + 2 * r, i = f / 24, b = (f - 24 * i) >> 1;
                const float *x = xs + i * kXPitch + 32 * ks + 8 * g;
                const float s = __builtin_ldexpf(1.0f, b - 1);
                bf8v e;
                if (w & 1) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) e[k] = (__bf16)__builtin_amdgcn_cosf(__builtin_amdgcn_fractf(x[k] * s));
                } else {
#pragma unroll
                    for (int k = 0; k < 8; ++k) e[k] = (__bf16)__builtin_amdgcn_sinf(__builtin_amdgcn_fractf(x[k] * s));
                }
#pragma unroll
                for (int m = 0; m < 4; ++m) grad[4 * half + m] = mfma32(da[m], e, grad[4 * half + m]);
            }
            if (w < 4) {
                // Features 256 .. 263, the constant 264, zeros.
                const bf8v zero = {};
                bf8v e = r < 8 ? lds8(ft + r * kTPitch + 32 * ks + 8 * g) : zero;
                if (r == 8) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) e[k] = (__bf16)(q0 + 32u * ks + 8u * g + k < n ? 1.0f : 0.0f);
                }
                grad[14] = mfma32(w == 0 ? da[0] : w == 1 ? da[1] : w == 2 ? da[2] : da[3], e, grad[14]);
            }
        }
        __syncthreads();
    }
    if (loss_sum) {
        for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off);
        if (lane == 0) atomicAdd(loss_sum, lsum);
    }
    float4 *out = partials + ((size_t)blockIdx.x * kTrainWaves + w) * kTileSlots * 64 + lane;
#pragma unroll
    for (int k = 0; k < kTileSlots; ++k) out[64 * k] = make_float4(grad[k][0], grad[k][1], grad[k][2], grad[k][3]);
}

// Sums the partial gradients of one tile (blockIdx.x = wave * kTileSlots + slot) over the blocks that
// wrote any and hands each of its 256 parameters and its sum to f, one per thread below 256.  Eight slices
// of the blocks are summed side by side, then added in order.
template <class F>
__device__ __forceinline__ void reduce_tile(const float4 *partials, uint32_t blocks, const F &f) {
    __shared__ float4 part[8][64];
    const int lane = threadIdx.x & 63, s = threadIdx.x >> 6;
    const float4 *p = partials + (size_t)blockIdx.x * 64 + lane;
    float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 8
    for (uint32_t b = (uint32_t)s; b < blocks; b += 8u) {
        const float4 v = p[(size_t)b * (kTrainWaves * kTileSlots * 64)];
        sum.x += v.x;
        sum.y += v.y;
        sum.z += v.z;
        sum.w += v.w;
    }
    part[s][lane] = sum;
    __syncthreads();
    if (threadIdx.x >= 256) return;
    const int l = threadIdx.x & 63, j = threadIdx.x >> 6;
    float g = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) g += reinterpret_cast<const float *>(&part[k][l])[j];
    f(tile_param((int)blockIdx.x / kTileSlots, (int)blockIdx.x % kTileSlots, l, j), g);
}
// Blocks of a backward launch of `grid` blocks that had samples.
__device__ __forceinline__ uint32_t blocks_used(uint32_t n, uint32_t grid) {
    return min((n + kTrainSamples - 1) / kTrainSamples, grid);
}

__global__ __launch_bounds__(512) void nrc_reduce_kernel(const float4 *partials, uint32_t n, uint32_t grid, float *grads) {
    reduce_tile(partials, blocks_used(n, grid), [&](int i, float g) { grads[i] = g; });
}

// One Adam step from a backward launch's partial gradients: 15.7 MB of them for 16384 samples, read at
// once by 120 blocks (one per tile).
__global__ __launch_bounds__(512) void nrc_adam_kernel(const float4 *partials, uint32_t grid, float *params, float *m, float *v,
                                                       uint16_t *wbf16, float *ema, uint16_t *wema, float lr, float c1,
                                                       float c2, uint32_t n, NrcSlice slice) {
    uint32_t offset;
    n = slice_bounds(slice, n, offset);
    if (n == 0) return;
    reduce_tile(partials, blocks_used(n, grid), [&](int i, float g) {
        const float mi = 0.9f * m[i] + 0.1f * g;
        const float vi = 0.99f * v[i] + 0.01f * g * g;
        m[i] = mi;
        v[i] = vi;
        const float p = params[i] - lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
        params[i] = p;
        wbf16[i] = to_bf16(p);
        const float e = kNrcEmaDecay * ema[i] + (1.0f - kNrcEmaDecay) * p;
        ema[i] = e;
        wema[i] = to_bf16(e);
    });
}

__global__ __launch_bounds__(256) void nrc_sync_kernel(const float *params, uint16_t *wbf16, float *ema, uint16_t *wema) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= kNrcParams) return;
    const float p = params[i];
    wbf16[i] = to_bf16(p);
    ema[i] = p;
    wema[i] = to_bf16(p);
}

__global__ __launch_bounds__(256) void nrc_zero_kernel(float *p, uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// Blocks for `work` items at `per_block` a block, at most `per_cu` blocks per compute unit.
int grid_for(uint32_t work, int per_block, int per_cu = 1) {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    const uint32_t blocks = (work + per_block - 1) / per_block, cap = (uint32_t)(cus * per_cu);
    return (int)(blocks < cap ? (blocks > 0 ? blocks : 1) : cap);
}

}  // namespace

hipError_t launch_nrc_infer(const NrcDevice &d, const float *inputs, uint32_t n, float *out, hipStream_t s,
                            const uint32_t *count, uint32_t stride) {
    if (n == 0) return hipSuccess;
    static bool configured = false;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute((const void *)nrc_infer_kernel<kInferTiles>, hipFuncAttributeMaxDynamicSharedMemorySize, kInferLds);
        if (e != hipSuccess) return e;
        configured = true;
    }
    hipLaunchKernelGGL(nrc_infer_kernel<kInferTiles>, dim3(grid_for(n, 16 * kInferTiles * kInferWaves, 2)), dim3(kInferBlock),
                       kInferLds, s, d.wema, inputs, stride, n, out, count);
    return hipGetLastError();
}

// Blocks of a backward launch over at most n samples.
static uint32_t train_grid(uint32_t n) {
    const uint32_t need = (n + kTrainSamples - 1) / kTrainSamples;
    return need < kNrcTrainBlocks ? need : kNrcTrainBlocks;
}

hipError_t launch_nrc_backward(const NrcDevice &d, const float *inputs, const float *targets, uint32_t n, float norm,
                               float *loss_sum, hipStream_t s, const NrcSlice &slice, uint32_t stride) {
    if (n == 0) return hipSuccess;
    static bool configured = false;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute((const void *)nrc_backward_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kTrainLds);
        if (e != hipSuccess) return e;
        configured = true;
    }
    hipLaunchKernelGGL(nrc_backward_kernel, dim3(train_grid(n)), dim3(kTrainBlock), kTrainLds, s, d.wbf16, inputs, stride, targets,
                       n, norm, reinterpret_cast<float4 *>(d.partials), loss_sum, slice);
    return hipGetLastError();
}

hipError_t launch_nrc_reduce(const NrcDevice &d, uint32_t n, float *grads, hipStream_t s) {
    hipLaunchKernelGGL(nrc_reduce_kernel, dim3(kNrcParams / 256), dim3(512), 0, s, reinterpret_cast<const float4 *>(d.partials), n,
                       train_grid(n), grads);
    return hipGetLastError();
}

hipError_t launch_nrc_adam(const NrcDevice &d, uint32_t step, float lr, hipStream_t s, uint32_t n, const NrcSlice &slice) {
    const float c1 = 1.0f - powf(0.9f, (float)step), c2 = 1.0f - powf(0.99f, (float)step);
    hipLaunchKernelGGL(nrc_adam_kernel, dim3(kNrcParams / 256), dim3(512), 0, s, reinterpret_cast<const float4 *>(d.partials),
                       train_grid(n), d.params, d.m, d.v, d.wbf16, d.ema, d.wema, lr, c1, c2, n, slice);
    return hipGetLastError();
}

hipError_t launch_nrc_sync(const NrcDevice &d, hipStream_t s) {
    hipLaunchKernelGGL(nrc_sync_kernel, dim3((kNrcParams + 255) / 256), dim3(256), 0, s, d.params, d.wbf16, d.ema, d.wema);
    return hipGetLastError();
}

hipError_t launch_nrc_zero(float *p, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(nrc_zero_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

}  // namespace vt
