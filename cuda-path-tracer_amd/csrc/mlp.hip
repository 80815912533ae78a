// Radiance-cache MLP on MFMA (no reference counterpart: the reference has no
// learned component).  96 inputs -> 4 x (64, ReLU) -> 3 outputs with exp;
// fp16 weights and activations as MFMA operands, fp32 accumulation, fp32
// master weights, Adam.
//
// Layout trick: every layer computes Z^T = W^T X^T with
// v_mfma_f32_16x16x16f16, activations as the B operand.  A 16x16 D fragment
// (lane l: rows 4(l/16)+e, column l%16) is then exactly the B fragment of the
// next layer's k-block (lane l: k = 4(l/16)+e, column l%16), so a sample
// block's activations stay in registers from the encoding to the output.
// Weights are pre-packed in A-fragment order (8 bytes per lane per 16x16
// block) and staged in LDS.
//
// Inference uses gfx950's doubled-K v_mfma_f32_16x16x32_f16 with its own
// fragment packing (below, kperm) and four 16-sample blocks per wave.
//
// Training step (deterministic: no floating-point atomics), two launches:
//   k_mlp_train      per workgroup, 64-sample rounds (one 16-sample block per
//                    wave): forward, relative-L2 loss, backward deltas, then
//                    the layer inputs and deltas go to LDS, a row per sample,
//                    and the four waves accumulate dW = act^T delta (MFMA,
//                    K = samples, operands through the transposing LDS read)
//                    and db = sum delta over the workgroup's samples; one fp32
//                    partial per workgroup
//   k_mlp_adam_pack  sums the partials in workgroup order, Adam on the fp32
//                    masters, and writes each updated weight into its fp16
//                    fragments (forward, backward and inference layouts)
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "context.hpp"
#include "sampling.hpp"

namespace pt {
namespace {

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kIn = 96, kHid = 64, kOut = 3, kLayers = 5;
__host__ __device__ constexpr int dim(int l) { return l == 0 ? kIn : (l == kLayers ? kOut : kHid); }
__host__ __device__ constexpr int w_off(int l) {
    return l == 0 ? 0 : w_off(l - 1) + dim(l - 1) * dim(l) + dim(l);
}
__host__ __device__ constexpr int b_off(int l) { return w_off(l) + dim(l) * dim(l + 1); }
constexpr int kParams = w_off(kLayers);  // 18,883
static_assert(kParams == 18883, "parameter count");
constexpr float kRelEps = 0.01f;

// 16-row/col blocks per layer: rows = output features (forward A), k = inputs.
__host__ __device__ constexpr int rb(int l) { return (dim(l + 1) + 15) / 16; }
__host__ __device__ constexpr int fb(int l) { return (dim(l) + 15) / 16; }
__host__ __device__ constexpr int fwd_base(int l) { return l == 0 ? 0 : fwd_base(l - 1) + rb(l - 1) * fb(l - 1); }
constexpr int kFwdFrags = fwd_base(kLayers);  // 76
// Backward A fragments (delta_{l-1} = W_l delta_l) for l = 1..4: rows = inputs, k = outputs.
__host__ __device__ constexpr int bwd_base(int l) { return l <= 1 ? 0 : bwd_base(l - 1) + fb(l - 1) * rb(l - 1); }
constexpr int kBwdFrags = bwd_base(kLayers);  // 52
constexpr int kFragHalves = 64 * 4;

// Inference fragments for gfx950's v_mfma_f32_16x16x32_f16 (A: lane L holds
// row L%16, k-elements 8(L/16)+j).  Two 16x16 D fragments of one layer --
// output rows 32q..32q+15 and 32q+16..32q+31 -- concatenated lane by lane
// (lane L: rows 4(L/16)+e of each) are the next layer's B operand for k-block
// q when the k index is permuted: element j of lane group g is feature
// kperm(q, g, j).  The weights are packed with the same permutation, so
// activations still never leave the registers.
__host__ __device__ constexpr int kperm(int q, int g, int j) { return 32 * q + (j < 4 ? 4 * g + j : 16 + 4 * g + (j - 4)); }
__host__ __device__ constexpr int kb32(int l) { return (dim(l) + 31) / 32; }
__host__ __device__ constexpr int f32_base(int l) { return l == 0 ? 0 : f32_base(l - 1) + rb(l - 1) * kb32(l - 1); }
constexpr int kF32Frags = f32_base(kLayers);  // 12 + 3 * 8 + 2 = 38
static_assert(kF32Frags == 38, "16x16x32 fragment count");
constexpr int kF32Halves = 64 * 8;

constexpr int kThreads = 256;

__device__ __forceinline__ floatx4 mfma(half4 a, half4 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ floatx4 mfma32(half8 a, half8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Masters -> 16x16x32 forward fragment (l, r, q), lane L, element j:
// W_l[kperm(q, L/16, j)][16r + L%16], zero outside the layer's shape.
__device__ __forceinline__ void pack32_frag(const float* __restrict__ master, _Float16* __restrict__ f32,
                                            int frag, int lane) {
    int l = 0;
    while (l + 1 < kLayers && frag >= f32_base(l + 1)) ++l;
    const int k = frag - f32_base(l);
    const int r = k / kb32(l), q = k % kb32(l);
    const int ni = dim(l), no = dim(l + 1);
    const float* W = master + w_off(l);
    const int o = 16 * r + lane % 16;
    _Float16* out = f32 + static_cast<size_t>(frag) * kF32Halves + lane * 8;
    for (int j = 0; j < 8; ++j) {
        const int i = kperm(q, lane / 16, j);
        out[j] = (i < ni && o < no) ? static_cast<_Float16>(W[i * no + o]) : static_cast<_Float16>(0.0f);
    }
}

// Masters -> fp16 fragments.  Forward fragment (l, r, f), lane L, element e:
// W_l[16f + 4(L/16) + e][16r + L%16]; backward fragment (l, r, f):
// W_l[16r + L%16][16f + 4(L/16) + e]; zero outside the layer's shape; then
// the 16x16x32 inference fragments (pack32_frag).  Also advances the
// device-side Adam step counter by `advance` (one thread).
__global__ __launch_bounds__(kThreads) void k_mlp_pack(const float* __restrict__ master,
                                                       _Float16* __restrict__ fwd,
                                                       _Float16* __restrict__ bwd,
                                                       _Float16* __restrict__ f32,
                                                       uint32_t* __restrict__ step, uint32_t advance) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0 && advance) step[0] += advance;
    const int frag = t / 64, lane = t % 64;
    if (frag >= kFwdFrags + kBwdFrags + kF32Frags) return;
    if (frag >= kFwdFrags + kBwdFrags) {
        pack32_frag(master, f32, frag - kFwdFrags - kBwdFrags, lane);
        return;
    }
    int l = 0, r = 0, f = 0;
    bool forward = frag < kFwdFrags;
    if (forward) {
        while (l + 1 < kLayers && frag >= fwd_base(l + 1)) ++l;
        const int k = frag - fwd_base(l);
        r = k / fb(l);
        f = k % fb(l);
    } else {
        const int fr = frag - kFwdFrags;
        l = 1;
        while (l + 1 < kLayers && fr >= bwd_base(l + 1)) ++l;
        const int k = fr - bwd_base(l);
        r = k / rb(l);
        f = k % rb(l);
    }
    const int ni = dim(l), no = dim(l + 1);
    const float* W = master + w_off(l);
    _Float16* out = (forward ? fwd + frag * kFragHalves : bwd + (frag - kFwdFrags) * kFragHalves) + lane * 4;
    for (int e = 0; e < 4; ++e) {
        int i, o;
        if (forward) {
            i = 16 * f + 4 * (lane / 16) + e;
            o = 16 * r + lane % 16;
        } else {
            i = 16 * r + lane % 16;
            o = 16 * f + 4 * (lane / 16) + e;
        }
        out[e] = (i < ni && o < no) ? static_cast<_Float16>(W[i * no + o]) : static_cast<_Float16>(0.0f);
    }
}

__device__ __forceinline__ half4 to_half4(floatx4 v) {
    return __builtin_convertvector(v, half4);
}

// ReLU of the rounded values: max(x, 0) commutes with rounding to fp16, and
// on halves it takes one instruction per pair.
__device__ __forceinline__ half4 relu_half4(floatx4 v) {
    return __builtin_elementwise_max(to_half4(v), half4{0, 0, 0, 0});
}

struct SceneBox {
    float mn[3], inv_ext[3];
};

// Input features 16 F + 4 g + {0, 1, 2, 3} of one sample (g: the lane's group
// of 16).  Features below 72 are (sin, cos) pairs of 2^k pi p, 12 frequencies
// for each axis -- sin/cos(2^k pi p) = sin/cos(2 pi frac(2^(k-1) p)), the
// hardware sine and cosine taking revolutions -- then come the normal, incoming
// direction and albedo (raw[3..11]), then zero padding.  F fixes the axis (in
// F = 1 up to the group) and what else a lane may hold, so nothing is indexed
// at run time: with arrays indexed by feature the 12 raw floats and positions
// lived in scratch memory.
template <int F>
__device__ __forceinline__ floatx4 features(int g, const float* p01, floatx4 rest) {
    floatx4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (F < 5) {
        float p;
        int k;  // frequency of the first pair
        if constexpr (F == 0) { p = p01[0]; k = 2 * g; }
        if constexpr (F == 1) { p = g >= 2 ? p01[1] : p01[0]; k = 2 * g + (g >= 2 ? -4 : 8); }
        if constexpr (F == 2) { p = p01[1]; k = 2 * g + 4; }
        if constexpr (F == 3) { p = p01[2]; k = 2 * g; }
        if constexpr (F == 4) { p = p01[2]; k = 2 * g + 8; }
        // Powers of two: exact, and a lane's factor is the same for every sample.
        const float r0 = p * __uint_as_float(static_cast<uint32_t>(126 + k) << 23), r1 = r0 + r0;
        const float f0 = r0 - floorf(r0), f1 = r1 - floorf(r1);
        v.x = __builtin_amdgcn_sinf(f0);
        v.y = __builtin_amdgcn_cosf(f0);
        v.z = __builtin_amdgcn_sinf(f1);
        v.w = __builtin_amdgcn_cosf(f1);
        if constexpr (F == 4) {
            v.x = g < 2 ? v.x : rest.x;
            v.y = g < 2 ? v.y : rest.y;
            v.z = g < 2 ? v.z : rest.z;
            v.w = g < 2 ? v.w : rest.w;
        }
    } else {
        v.x = g == 0 ? rest.w : 0.0f;
    }
    return v;
}

// What a lane reads of one sample (zeros past the batch): the position, and of
// the other nine floats the four that its group's features hold -- raw[3..6]
// (group 2), raw[7..10] (group 3) or, as the last, raw[11] (group 0).  Two
// loads that need no more than the floats' own alignment.
struct Sample {
    float x, y, z;
    floatx4 rest;
};
__device__ __forceinline__ Sample load_sample(const float* __restrict__ raw, uint32_t n, uint32_t s) {
    typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));
    const int g = (threadIdx.x & 63) / 16;
    Sample v = {0.0f, 0.0f, 0.0f, {0.0f, 0.0f, 0.0f, 0.0f}};
    if (s < n) {
        const float* p = raw + 12 * static_cast<size_t>(s);
        v.rest = *reinterpret_cast<const floatx4u*>(p + (g == 2 ? 3 : (g == 3 ? 7 : 8)));
        v.x = p[0];
        v.y = p[1];
        v.z = p[2];
    }
    return v;
}
__device__ __forceinline__ void in_box(const Sample& v, const SceneBox& box, float* p01) {
    p01[0] = (v.x - box.mn[0]) * box.inv_ext[0];
    p01[1] = (v.y - box.mn[1]) * box.inv_ext[1];
    p01[2] = (v.z - box.mn[2]) * box.inv_ext[2];
}

// Lane's view of one 16-sample block: the input fragments X[f] (k-block f).
__device__ __forceinline__ void encode_block(const Sample& v, const SceneBox& box, half4* X) {
    const int g = (threadIdx.x & 63) / 16;
    float p01[3];
    in_box(v, box, p01);
    X[0] = to_half4(features<0>(g, p01, v.rest));
    X[1] = to_half4(features<1>(g, p01, v.rest));
    X[2] = to_half4(features<2>(g, p01, v.rest));
    X[3] = to_half4(features<3>(g, p01, v.rest));
    X[4] = to_half4(features<4>(g, p01, v.rest));
    X[5] = to_half4(features<5>(g, p01, v.rest));
}

__device__ __forceinline__ half4 lds_frag(const uint2* __restrict__ frags, int idx) {
    const uint2 u = frags[idx * 64 + (threadIdx.x & 63)];
    half4 h;
    __builtin_memcpy(&h, &u, sizeof h);
    return h;
}

// Biases of a lane's four rows of row block r, from LDS (zeros past the layer).
__device__ __forceinline__ floatx4 bias4(const float* b, int r) {
    const int o = 16 * r + 4 * ((threadIdx.x & 63) / 16);
    return floatx4{b[o + 0], b[o + 1], b[o + 2], b[o + 3]};
}

// Global -> LDS copy of BYTES bytes (a multiple of 1,024; both 16-byte aligned)
// by the workgroup's waves, 1,024 bytes an instruction straight into LDS, all
// in flight at once.  Barrier-ready once stage_wait has returned.
template <uint32_t BYTES>
__device__ __forceinline__ void stage(void* dst, const void* __restrict__ src) {
    static_assert(BYTES % 1024u == 0u, "whole wave copies");
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64u), lane = threadIdx.x & 63u;
    const char* s = static_cast<const char*>(src) + lane * 16u;
    char* d = static_cast<char*>(dst);
#pragma unroll
    for (uint32_t k = 0; k < (BYTES / 1024u + kThreads / 64u - 1u) / (kThreads / 64u); ++k) {
        const uint32_t piece = k * (kThreads / 64u) + wave;
        if (piece < BYTES / 1024u) {
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(s + piece * 1024u),
                (__attribute__((address_space(3))) void*)(d + piece * 1024u), 16, 0, 0);
        }
    }
}
__device__ __forceinline__ void stage_wait() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

__device__ __forceinline__ half8 lds_frag32(const uint4* __restrict__ frags, int idx) {
    const uint4 u = frags[idx * 64 + (threadIdx.x & 63)];
    half8 h;
    __builtin_memcpy(&h, &u, sizeof h);
    return h;
}

__device__ __forceinline__ half8 join(half4 a, half4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

// Next layer's B operand for k-block q from the D fragments of row blocks
// 2q and 2q + 1 (ReLU, fp16).
__device__ __forceinline__ half8 join_relu(floatx4 a, floatx4 b) { return join(relu_half4(a), relu_half4(b)); }

// Inference: out[3s + c] = exp(z_c).  A wave runs kInferBlocks 16-sample
// blocks at a time so each weight fragment read from LDS feeds kInferBlocks
// MFMAs.  2,073,600 samples take 81 us (152 with inputs indexed through
// scratch, MFMA results in accumulation registers and 16 lanes finishing one
// block's outputs): of a SIMD's 181,000 cycles its matrix core is busy 77,000,
// its vector instructions issue for 95,000, and 34,000 of these coincide.
// Prefetching the next samples (142 registers, three waves) changed nothing;
// what memory and staging alone take is 31 us.
constexpr int kInferBlocks = 4;

__global__ __launch_bounds__(kThreads) void k_mlp_infer(const uint4* __restrict__ f32,
                                                        const float* __restrict__ master,
                                                        const float* __restrict__ raw, uint32_t n,
                                                        SceneBox box, float* __restrict__ out) {
    __shared__ __align__(16) uint4 s_frag[kF32Frags * 64];
    __shared__ float s_bias[kLayers][kHid];
    stage<kF32Frags * 1024u>(s_frag, f32);
    for (int k = threadIdx.x; k < kLayers * kHid; k += blockDim.x) {
        const int l = k / kHid, o = k % kHid;
        s_bias[l][o] = o < dim(l + 1) ? master[b_off(l) + o] : 0.0f;
    }
    stage_wait();
    const int lane = threadIdx.x & 63, g = lane / 16;
    const uint32_t wave = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
    const uint32_t nwaves = gridDim.x * (blockDim.x / 64);
    auto bias = [&](int l, int r) { return bias4(s_bias[l], r); };
    constexpr uint32_t kSpan = 16 * kInferBlocks;
    for (uint32_t base = wave * kSpan; base < n; base += nwaves * kSpan) {
        // Weight fragments are read from LDS where used: kept from one
        // iteration to the next they would take 152 VGPRs (one wave per SIMD).
        asm volatile("" ::: "memory");
        half8 X[kInferBlocks][3];
#pragma unroll
        for (int b = 0; b < kInferBlocks; ++b) {
            half4 x[fb(0)];
            encode_block(load_sample(raw, n, base + 16 * b + lane % 16), box, x);
            X[b][0] = join(x[0], x[1]);
            X[b][1] = join(x[2], x[3]);
            X[b][2] = join(x[4], x[5]);
        }
        // Layer 0: 96 -> 64.  Waves in their layers issue before waves that
        // encode, whose vector instructions fill the matrix cores' cycles
        // (77.2 us against 78.4).
        __builtin_amdgcn_s_setprio(1);
        half8 H[kInferBlocks][2];
#pragma unroll
        for (int rp = 0; rp < 2; ++rp) {
            floatx4 acc[kInferBlocks][2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const floatx4 bv = bias(0, 2 * rp + h);
#pragma unroll
                for (int b = 0; b < kInferBlocks; ++b) acc[b][h] = bv;
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const half8 a = lds_frag32(s_frag, f32_base(0) + (2 * rp + h) * 3 + q);
#pragma unroll
                    for (int b = 0; b < kInferBlocks; ++b) acc[b][h] = mfma32(a, X[b][q], acc[b][h]);
                }
            }
#pragma unroll
            for (int b = 0; b < kInferBlocks; ++b) H[b][rp] = join_relu(acc[b][0], acc[b][1]);
        }
        // Layers 1..3: 64 -> 64.
#pragma unroll
        for (int l = 1; l < 4; ++l) {
            half8 Hn[kInferBlocks][2];
#pragma unroll
            for (int rp = 0; rp < 2; ++rp) {
                floatx4 acc[kInferBlocks][2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const floatx4 bv = bias(l, 2 * rp + h);
#pragma unroll
                    for (int b = 0; b < kInferBlocks; ++b) acc[b][h] = bv;
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const half8 a = lds_frag32(s_frag, f32_base(l) + (2 * rp + h) * 2 + q);
#pragma unroll
                        for (int b = 0; b < kInferBlocks; ++b) acc[b][h] = mfma32(a, H[b][q], acc[b][h]);
                    }
                }
#pragma unroll
                for (int b = 0; b < kInferBlocks; ++b) Hn[b][rp] = join_relu(acc[b][0], acc[b][1]);
            }
#pragma unroll
            for (int b = 0; b < kInferBlocks; ++b) {
                H[b][0] = Hn[b][0];
                H[b][1] = Hn[b][1];
            }
        }
        // Layer 4: 64 -> 3, exp.  Every fourth row takes the weights of rows
        // 0..3, so each lane group holds the three outputs of every block and
        // finishes one block: 64 samples' exponentials and stores at once.
        floatx4 z[kInferBlocks];
        const floatx4 b4 = {s_bias[4][0], s_bias[4][1], s_bias[4][2], 0.0f};
#pragma unroll
        for (int b = 0; b < kInferBlocks; ++b) z[b] = b4;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            half8 a;
            __builtin_memcpy(&a, &s_frag[(f32_base(4) + q) * 64 + (lane & ~12)], sizeof a);
#pragma unroll
            for (int b = 0; b < kInferBlocks; ++b) z[b] = mfma32(a, H[b][q], z[b]);
        }
        __builtin_amdgcn_s_setprio(0);
        static_assert(kInferBlocks == 4, "one lane group for each block's outputs");
        const floatx4 zl = g < 2 ? (g == 0 ? z[0] : z[1]) : (g == 2 ? z[2] : z[3]);
        const uint32_t s = base + lane;
        if (s < n) {
            out[3 * static_cast<size_t>(s) + 0] = expf(zl.x);
            out[3 * static_cast<size_t>(s) + 1] = expf(zl.y);
            out[3 * static_cast<size_t>(s) + 2] = expf(zl.z);
        }
    }
}

// Training rounds: 64 samples per workgroup round, one 16-sample block per
// wave.  A sample's layer inputs act_l (96 + 4 x 64 halves) and deltas delta_l
// = dL/dz_l scaled by n (4 x 64, then 16 of which 3 are used) are a row each of
// two LDS arrays: a lane stores the four features of its fragment in one
// 8-byte write, and gfx950's transposing LDS read returns them feature by
// feature, four samples to a lane, as the operands of the weight gradients.
// Row strides of 8 x an odd number of banks: the transposing read's eight rows
// of 32 bytes fall in different banks.
constexpr int kTrainChunk = 64;
constexpr int kActLd = 8 * 46;             // 352 halves used
constexpr int kDelLd = 8 * 34;             // 272 halves
static_assert(kActLd >= kIn + 4 * kHid && kActLd / 2 % 16 == 8, "activation rows");
static_assert(kDelLd >= 4 * kHid + 16 && kDelLd / 2 % 16 == 8, "delta rows");
__host__ __device__ constexpr int act_col(int l) { return l == 0 ? 0 : kIn + kHid * (l - 1); }
__host__ __device__ constexpr int del_col(int l) { return kHid * l; }
constexpr int kTilesPerWave = fwd_base(kLayers) / 4;  // 76 weight tiles (16 x 16)
static_assert(kTilesPerWave == 19, "weight tiles of a wave: 6 + 3 x 4 + 1");
constexpr uint32_t kMaxTrainBlocks = 256;  // workgroups (gradient partials) of one step

// Deltas are gradients of n * loss (a static loss scale of n keeps them well
// inside fp16's normal range); they are clamped to fp16's finite range so an
// outlier sample cannot turn a whole step into inf/NaN.
constexpr float kHalfMax = 65504.0f;
__device__ __forceinline__ float sat(float x) {
    return x > kHalfMax ? kHalfMax : (x < -kHalfMax ? -kHalfMax : x);
}

// Deltas d through the ReLU whose outputs are h (never negative): clamped as
// halves (rounding first gives the same: what rounds past the largest half
// becomes infinite and is clamped; NaN stays NaN), zero where h is zero.
__device__ __forceinline__ half4 mask4(floatx4 d, half4 h) {
    typedef short short4v __attribute__((ext_vector_type(4)));
    const half4 hi = static_cast<half4>(static_cast<_Float16>(kHalfMax));
    const half4 x = __builtin_elementwise_minimum(__builtin_elementwise_maximum(to_half4(d), -hi), hi);
    const short4v on = (static_cast<short4v>(0) - __builtin_bit_cast(short4v, h)) >> 15;
    return __builtin_bit_cast(half4, static_cast<short4v>(__builtin_bit_cast(short4v, x) & on));
}

// A lane's four features (row0 + 4(l/16) + e) of its sample (column l%16 of
// the wave's block): its place in the sample's LDS row.
__device__ __forceinline__ half4* lds_cell(_Float16* sample, int row0) {
    return reinterpret_cast<half4*>(sample + row0 + 4 * ((threadIdx.x & 63) / 16));
}

// MFMA operand: lane l gets feature l%16 of the 16 at `tile` (+ the lane's own
// offset tr_off, see there) for samples 4(l/16) .. +3 of the tile's 16.
__device__ __forceinline__ half4 lds_get(const _Float16* tile) {
    typedef short short4v __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                         (__attribute__((address_space(3))) short4v*)(tile)));
}
// Where lane l reads for lds_get: 8 bytes of sample 4(l/16) + (l%16)/4.
__device__ __forceinline__ int tr_off(int ld) {
    const int l = threadIdx.x & 63;
    return (4 * (l / 16) + l % 16 / 4) * ld + 4 * (l % 4);
}

// One training step's gradient partials.  Workgroup b handles rounds b,
// b + gridDim.x, ... and writes part[b][param] (weights and biases, fp32).
// loss[s] = the sample's relative-L2 loss summed over channels.  A sample
// whose first target channel is NaN is masked: zero loss, zero deltas (it
// still counts in the mean's n).  Thread 0 of workgroup 0 advances the Adam
// step counter by `advance` (read by k_mlp_adam_pack after this launch).
//
// Up to 16,384 samples a workgroup has one round and a SIMD one wave, so the
// kernel lasts as long as one round's chain of dependent steps, and code that
// runs once comes from memory as it is needed: the middle layers are loops
// (11 KB of code; unrolled, with the tiles' places worked out one by one, it
// was 25 KB), the samples and targets are loaded before the weights are
// staged.  A wave's tiles share operands: layer 0's six have one block of
// deltas, a middle layer's four one block of inputs.  A gradient of
// 16,384 samples takes 22.7 us of which this is 17; it took 42.5.
__global__ __launch_bounds__(kThreads) void k_mlp_train(
    const uint2* __restrict__ fwd, const uint2* __restrict__ bwd, const float* __restrict__ master,
    const float* __restrict__ raw, const float* __restrict__ target, uint32_t n, SceneBox box,
    float* __restrict__ part, float* __restrict__ loss, uint32_t* __restrict__ step, uint32_t advance) {
    __shared__ __align__(16) uint2 s_fwd[kFwdFrags * 64];
    __shared__ __align__(16) uint2 s_bwd[kBwdFrags * 64];
    __shared__ __align__(16) _Float16 s_act[kTrainChunk][kActLd];
    __shared__ __align__(16) _Float16 s_del[kTrainChunk][kDelLd];
    __shared__ __align__(16) float s_bias[kLayers][kHid];
    const int lane = threadIdx.x & 63, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int col = 16 * wave + lane % 16;  // the lane's sample of a round
    // Lane groups 0..2 hold a sample's three target channels, `first` the
    // first (NaN: masked) in all of them.
    float t = 0.0f, first = 0.0f;
    Sample in;
    auto load = [&](uint32_t round) {
        const uint32_t s = round * kTrainChunk + col;
        in = load_sample(raw, n, s);
        if (s < n) {
            first = target[3 * static_cast<size_t>(s)];
            t = target[3 * static_cast<size_t>(s) + (g < kOut ? g : 0)];
        }
    };
    load(blockIdx.x);
    stage<kFwdFrags * 512u>(s_fwd, fwd);
    stage<kBwdFrags * 512u>(s_bwd, bwd);
    for (int k = threadIdx.x; k < kLayers * kHid; k += kThreads) {
        const int l = k / kHid, o = k % kHid;
        s_bias[l][o] = o < dim(l + 1) ? master[b_off(l) + o] : 0.0f;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && advance) step[0] += advance;
    stage_wait();
    floatx4 acc[kTilesPerWave];
#pragma unroll
    for (int k = 0; k < kTilesPerWave; ++k) acc[k] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    // Bias sums: thread t owns delta column t (layers 0..3) and, for t < 3,
    // output bias t (delta 4's column t).
    float bsum = 0.0f, bsum4 = 0.0f;
    for (uint32_t round = blockIdx.x; round * kTrainChunk < n; round += gridDim.x) {
        if (round != blockIdx.x) load(round);
        const uint32_t s = round * kTrainChunk + col;
        _Float16* act = s_act[col];
        _Float16* del = s_del[col];
        // Forward.
        half4 H[4];
        {
            half4 X[fb(0)];
            encode_block(in, box, X);
            floatx4 z[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) z[r] = bias4(s_bias[0], r);
#pragma unroll
            for (int f = 0; f < fb(0); ++f) {
                *lds_cell(act, 16 * f) = X[f];
#pragma unroll
                for (int r = 0; r < 4; ++r) z[r] = mfma(lds_frag(s_fwd, r * fb(0) + f), X[f], z[r]);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                H[r] = relu_half4(z[r]);
                *lds_cell(act, act_col(1) + 16 * r) = H[r];
            }
        }
#pragma unroll 1
        for (int l = 1; l < 4; ++l) {
            const uint2* frags = s_fwd + (fwd_base(1) + 16 * (l - 1)) * 64;
            floatx4 z[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) z[r] = bias4(s_bias[l], r);
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int r = 0; r < 4; ++r) z[r] = mfma(lds_frag(frags, 4 * r + f), H[f], z[r]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                H[r] = relu_half4(z[r]);
                *lds_cell(act, act_col(1) + kHid * l + 16 * r) = H[r];
            }
        }
        // Outputs: as in inference, every lane group gets all three.
        floatx4 z = {s_bias[4][0], s_bias[4][1], s_bias[4][2], 0.0f};
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            half4 a;
            __builtin_memcpy(&a, &s_fwd[(fwd_base(4) + f) * 64 + (lane & ~12)], sizeof a);
            z = mfma(a, H[f], z);
        }
        // Output delta: d/dz of (e^z - t)^2 / (sg(e^z)^2 + eps), lane group c
        // computing channel c of its samples.
        const bool live = s < n && first == first;
        const float y = expf(g == 0 ? z.x : (g == 1 ? z.y : z.z));
        const float den = y * y + kRelEps;
        const float lc = (y - t) * (y - t) / den;
        const float gr = 2.0f * (y - t) / den * y;
        const float dd = live && gr == gr ? sat(gr) : 0.0f;  // NaN (inf/inf) -> no update
        const int c0 = lane % 16;
        const float l1 = __shfl(lc, c0 + 16), l2 = __shfl(lc, c0 + 32);
        const float d1 = __shfl(dd, c0 + 16), d2 = __shfl(dd, c0 + 32);
        if (lane < 16 && s < n && loss) loss[s] = live ? (lc + l1) + l2 : 0.0f;
        const floatx4 d4 = {dd, d1, d2, 0.0f};
        const half4 D4 = lane < 16 ? to_half4(d4) : half4{0, 0, 0, 0};
        *lds_cell(del, del_col(4)) = D4;
        // delta_3 = W4 delta_4 (masked by ReLU of layer 3's output).
        half4 D[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            floatx4 a = {0.0f, 0.0f, 0.0f, 0.0f};
            a = mfma(lds_frag(s_bwd, bwd_base(4) + r), D4, a);
            D[r] = mask4(a, H[r]);
            *lds_cell(del, del_col(3) + 16 * r) = D[r];
        }
#pragma unroll 1
        for (int l = 3; l >= 1; --l) {
            const uint2* frags = s_bwd + 16 * (l - 1) * 64;
            half4 h[4];  // layer l's inputs, as this lane stored them
            floatx4 a[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                h[r] = *lds_cell(act, act_col(1) + kHid * (l - 1) + 16 * r);
                a[r] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int r = 0; r < 4; ++r) a[r] = mfma(lds_frag(frags, 4 * r + f), D[f], a[r]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                D[r] = mask4(a[r], h[r]);
                *lds_cell(del, kHid * (l - 1) + 16 * r) = D[r];
            }
        }
        __syncthreads();
        // dW tiles of this wave over the round's 64 samples (K = 4 x 16):
        // layer 0 inputs 16 f .. by outputs 16 wave .., layers 1..3 inputs
        // 16 wave .. by outputs 16 r .., layer 4 inputs 16 wave ...
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            const _Float16* a0 = s_act[16 * kb] + tr_off(kActLd);
            const _Float16* d0 = s_del[16 * kb] + tr_off(kDelLd);
            {
                const half4 d = lds_get(d0 + 16 * wave);
#pragma unroll
                for (int f = 0; f < fb(0); ++f) acc[f] = mfma(lds_get(a0 + 16 * f), d, acc[f]);
            }
#pragma unroll
            for (int l = 1; l < 4; ++l) {
                const half4 a = lds_get(a0 + act_col(l) + 16 * wave);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[2 + 4 * l + r] = mfma(a, lds_get(d0 + del_col(l) + 16 * r), acc[2 + 4 * l + r]);
            }
            acc[18] = mfma(lds_get(a0 + act_col(4) + 16 * wave), lds_get(d0 + del_col(4)), acc[18]);
        }
        {
            const int c = threadIdx.x;
            float a = 0.0f;
#pragma unroll 16
            for (int j = 0; j < kTrainChunk; ++j) a += static_cast<float>(s_del[j][c]);
            bsum += a;
            if (c < kOut) {
                float a4 = 0.0f;
#pragma unroll 16
                for (int j = 0; j < kTrainChunk; ++j) a4 += static_cast<float>(s_del[j][del_col(4) + c]);
                bsum4 += a4;
            }
        }
        __syncthreads();  // the next round rewrites the LDS rows
    }
    // D lane: column (output) lane%16 of the tile, rows (inputs) 4(lane/16) + e.
    float* out = part + static_cast<size_t>(blockIdx.x) * kParams;
    const int in0 = 4 * g, o = lane % 16;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int f = 0; f < fb(0); ++f) out[(16 * f + in0 + e) * kHid + 16 * wave + o] = acc[f][e];
#pragma unroll
        for (int l = 1; l < 4; ++l)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                out[w_off(l) + (16 * wave + in0 + e) * kHid + 16 * r + o] = acc[2 + 4 * l + r][e];
        if (o < kOut) out[w_off(4) + (16 * wave + in0 + e) * kOut + o] = acc[18][e];
    }
    const int c = threadIdx.x;
    out[b_off(c / kHid) + c % kHid] = bsum;
    if (c < kOut) out[b_off(4) + c] = bsum4;
}

// Adam (Kingma & Ba 2015) on the fp32 masters, one thread per parameter; the
// gradient is the sum of the workgroup partials in workgroup order divided
// by n (the loss is a mean over n).  The bias corrections use step t =
// step[0] (k_mlp_train advanced it), read on the device so a captured frame
// replays with the right t.  The updated weight is written into its fp16
// fragments: forward (16x16x16, layer input as k), backward (16x16x16, layer
// output as k) and inference (16x16x32, permuted k).  grad_out: only the
// gradient, no update.
// One workgroup per 64 parameters: the four waves sum the partials
// s = w, w + 4, w + 8, ... of their parameter (coalesced rows), then the
// first wave adds the four sums in wave order -- a fixed order, so the
// gradient is the same bits on every call.
constexpr int kAdamParams = 64;

__global__ __launch_bounds__(kThreads) void k_mlp_adam_pack(float* __restrict__ master, float* __restrict__ m,
                                                            float* __restrict__ v, const float* __restrict__ part,
                                                            uint32_t nparts, float inv_n, float lr, float b1,
                                                            float b2, float eps, const uint32_t* __restrict__ step,
                                                            float* __restrict__ grad_out, _Float16* __restrict__ fwd,
                                                            _Float16* __restrict__ bwd, _Float16* __restrict__ f32) {
    __shared__ float s_sum[kThreads / kAdamParams][kAdamParams];
    const int lane = threadIdx.x % kAdamParams, wave = threadIdx.x / kAdamParams;
    const int p = blockIdx.x * kAdamParams + lane;
    constexpr int kWaves = kThreads / kAdamParams;
    float acc = 0.0f;
    if (p < kParams) {
        uint32_t s = static_cast<uint32_t>(wave);
#pragma unroll 16
        for (; s < nparts; s += kWaves) acc += part[static_cast<size_t>(s) * kParams + p];
    }
    s_sum[wave][lane] = acc;
    __syncthreads();
    if (wave != 0 || p >= kParams) return;
    float g = ((s_sum[0][lane] + s_sum[1][lane]) + s_sum[2][lane]) + s_sum[3][lane];
    static_assert(kWaves == 4, "four partial sums per parameter");
    g *= inv_n;
    if (grad_out) {
        grad_out[p] = g;
        return;
    }
    const float t = static_cast<float>(step[0]);
    const float c1 = 1.0f - powf(b1, t);
    const float c2 = 1.0f - powf(b2, t);
    const float mk = b1 * m[p] + (1.0f - b1) * g;
    const float vk = b2 * v[p] + (1.0f - b2) * g * g;
    m[p] = mk;
    v[p] = vk;
    const float w = master[p] - lr * (mk / c1) / (sqrtf(vk / c2) + eps);
    master[p] = w;
    int l = 0;
    while (l + 1 < kLayers && p >= w_off(l + 1)) ++l;
    if (p >= b_off(l)) return;  // a bias: no fragment
    const int no = dim(l + 1);
    const int i = (p - w_off(l)) / no, o = (p - w_off(l)) % no;
    const _Float16 h = static_cast<_Float16>(w);
    // Forward fragment (l, o/16, i/16): lane 16((i%16)/4) + o%16, element i%4.
    fwd[(fwd_base(l) + (o / 16) * fb(l) + i / 16) * kFragHalves + (16 * ((i % 16) / 4) + o % 16) * 4 + i % 4] = h;
    // Backward fragment (l, i/16, o/16), l >= 1: lane 16((o%16)/4) + i%16, element o%4.
    if (l >= 1)
        bwd[(bwd_base(l) + (i / 16) * rb(l) + o / 16) * kFragHalves + (16 * ((o % 16) / 4) + i % 16) * 4 + o % 4] = h;
    // Inference fragment (l, o/16, i/32): k index i - 32q = kperm's position.
    const int q = i / 32, ip = i - 32 * q;
    const int g4 = ip < 16 ? ip / 4 : (ip - 16) / 4;
    const int j = ip < 16 ? ip % 4 : 4 + (ip - 16) % 4;
    f32[(f32_base(l) + (o / 16) * kb32(l) + q) * kF32Halves + (16 * g4 + o % 16) * 8 + j] = h;
}

uint32_t blocks_for(uint64_t work, uint32_t per) { return static_cast<uint32_t>((work + per - 1) / per); }


}  // namespace

int RadianceCache::param_count() { return kParams; }

void RadianceCache::set_box(const float* bmin, const float* bmax) {
    for (int k = 0; k < 3; ++k) {
        box_min[k] = bmin[k];
        box_inv[k] = 1.0f / (bmax[k] - bmin[k]);
    }
}

void RadianceCache::init(uint64_t seed, hipStream_t st) {
    // He-uniform weights for the ReLU layers, a small output layer, zero
    // biases; drawn on the host from SplitMix64.
    std::vector<float> h(kParams, 0.0f);
    uint64_t s = seed;
    auto u01 = [&]() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return static_cast<float>(z >> 40) * (1.0f / 16777216.0f);
    };
    for (int l = 0; l < kLayers; ++l) {
        const int ni = dim(l), no = dim(l + 1);
        const float a = (l + 1 < kLayers ? std::sqrt(6.0f / ni) : 0.1f * std::sqrt(6.0f / ni));
        for (int k = 0; k < ni * no; ++k) h[w_off(l) + k] = (2.0f * u01() - 1.0f) * a;
    }
    set_params(h.data(), st);
}

void RadianceCache::set_params(const float* host, hipStream_t st) {
    master.reserve(kParams * sizeof(float));
    m.reserve(kParams * sizeof(float));
    v.reserve(kParams * sizeof(float));
    fwd.reserve(static_cast<size_t>(kFwdFrags) * kFragHalves * 2);
    f32.reserve(static_cast<size_t>(kF32Frags) * kF32Halves * 2);
    bwd.reserve(static_cast<size_t>(kBwdFrags) * kFragHalves * 2);
    dstep.reserve(sizeof(uint32_t));
    PT_HIP(hipMemcpyAsync(master.as<void>(), host, kParams * sizeof(float), hipMemcpyHostToDevice, st));
    PT_HIP(hipMemsetAsync(m.as<void>(), 0, kParams * sizeof(float), st));
    PT_HIP(hipMemsetAsync(v.as<void>(), 0, kParams * sizeof(float), st));
    PT_HIP(hipMemsetAsync(dstep.as<void>(), 0, sizeof(uint32_t), st));
    PT_HIP(hipStreamSynchronize(st));
    ready = true;
    pack(st, 0);
}

void RadianceCache::get_params(float* host, hipStream_t st) {
    if (!ready) throw Error(PT_E_INVALID_ARG, "radiance cache not initialised");
    PT_HIP(hipMemcpyAsync(host, master.as<void>(), kParams * sizeof(float), hipMemcpyDeviceToHost, st));
    PT_HIP(hipStreamSynchronize(st));
}

void RadianceCache::pack(hipStream_t st, uint32_t advance) {
    hipLaunchKernelGGL(k_mlp_pack, dim3(blocks_for((kFwdFrags + kBwdFrags + kF32Frags) * 64, kThreads)),
                       dim3(kThreads), 0, st, master.as<float>(), fwd.as<_Float16>(), bwd.as<_Float16>(),
                       f32.as<_Float16>(), dstep.as<uint32_t>(), advance);
    PT_HIP(hipGetLastError());
}

void RadianceCache::infer(const float* d_raw, uint32_t n, float* d_out, hipStream_t st) {
    if (!ready) throw Error(PT_E_INVALID_ARG, "radiance cache not initialised");
    if (n == 0) return;
    SceneBox b;
    for (int k = 0; k < 3; ++k) {
        b.mn[k] = box_min[k];
        b.inv_ext[k] = box_inv[k];
    }
    // At most what is resident at once (four workgroups a CU by LDS and
    // registers): the weights are staged once (2,048 blocks: a single call of
    // 2,073,600 samples 91.1 us, 89.6 with 1,024).
    const uint32_t blocks = std::min<uint32_t>(blocks_for(n, 4 * 16 * kInferBlocks), 1024);
    hipLaunchKernelGGL(k_mlp_infer, dim3(blocks), dim3(kThreads), 0, st, f32.as<uint4>(), master.as<float>(),
                       d_raw, n, b, d_out);
    PT_HIP(hipGetLastError());
}

// Workgroups (gradient partials) of a training step over n samples.
uint32_t train_blocks(uint32_t n) {
    return std::max<uint32_t>(1u, std::min<uint32_t>(kMaxTrainBlocks, blocks_for(n, kTrainChunk)));
}

void RadianceCache::prepare_train(uint32_t n) {
    part.reserve(static_cast<size_t>(train_blocks(n)) * kParams * sizeof(float));
    loss.reserve((static_cast<size_t>(n) + 16) * sizeof(float));
}

void RadianceCache::launch_train(const float* d_raw, const float* d_target, uint32_t n, float* d_loss,
                                 float* d_grad_out, hipStream_t st) {
    const uint32_t nb = train_blocks(n);
    SceneBox b;
    for (int k = 0; k < 3; ++k) {
        b.mn[k] = box_min[k];
        b.inv_ext[k] = box_inv[k];
    }
    hipLaunchKernelGGL(k_mlp_train, dim3(nb), dim3(kThreads), 0, st, fwd.as<uint2>(), bwd.as<uint2>(),
                       master.as<float>(), d_raw, d_target, n, b, part.as<float>(),
                       d_loss ? d_loss : loss.as<float>(), dstep.as<uint32_t>(), d_grad_out ? 0u : 1u);
    hipLaunchKernelGGL(k_mlp_adam_pack, dim3(blocks_for(kParams, kAdamParams)), dim3(kThreads), 0, st,
                       master.as<float>(), m.as<float>(), v.as<float>(), part.as<float>(), nb,
                       1.0f / static_cast<float>(n), lr, beta1, beta2, eps, dstep.as<uint32_t>(), d_grad_out,
                       fwd.as<_Float16>(), bwd.as<_Float16>(), f32.as<_Float16>());
    PT_HIP(hipGetLastError());
}

void RadianceCache::train(const float* d_raw, const float* d_target, uint32_t n, float* d_loss,
                          float* d_grad_out, hipStream_t st) {
    if (!ready) throw Error(PT_E_INVALID_ARG, "radiance cache not initialised");
    if (n == 0) return;
    prepare_train(n);
    launch_train(d_raw, d_target, n, d_loss, d_grad_out, st);
}

}  // namespace pt
