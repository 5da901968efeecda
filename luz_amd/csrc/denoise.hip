// denoise.hip — learned per-pixel denoiser of 1-spp ambient occlusion and
// soft shadows on gfx950, inference and training with BF16 MFMA.
//
// Network (per (pixel, light) sample): 150 features = a 5x5 neighbourhood
// (clamped to the image) x 6 channels {AO, visibility of the light, relative
// depth, normal.xyz}; 4 hidden layers of 64 with ReLU; 2 outputs {AO,
// visibility} added to the 5x5 mean of the noisy AO and visibility inputs over
// the window's foreground pixels (FP32), so the network learns a correction to
// that box filter and BF16 precision bounds only the correction.  A pixel's AO
// is the mean of the AO outputs of its L samples.  Weights are BF16,
// accumulation FP32, biases FP32.
//
// MFMA mapping (v_mfma_f32_16x16x32_bf16, 64 lanes): weights are the A
// operand (16 output features x 32 inputs), samples the B operand (32 inputs
// x 16 samples).  The 16x16 FP32 result leaves lane (j, g) = (lane % 16,
// lane / 16) holding features 4g..4g+3 of sample j, which is exactly the B
// operand lane layout of the next layer when its input index k of element e
// of K-step s is  k = 16 * (2s + e/4) + 4g + e%4.  Weight fragments are
// packed in that order, so activations stay in registers through all five
// layers, forward and backward (the transposed weights W^T are packed the
// same way for the backward pass).  The features of layer 1 go in the order of
// infer_feature.  Any K order works as long as A and B agree, because the hardware
// pairs element e of lane group g of A with the same element of B.
//
// Inference (k_dn_infer) takes 16-pixel tiles: the 125 features that do not
// depend on the light enter layer 1 once per pixel, the 25 visibilities of a
// light as one more K-step per light, and layers 2..5 run per light.
//
// Training: k_dn_forward runs forward, loss and the backward pass to
// every layer's pre-activation gradient dz, and stores x, h and dz (BF16)
// sample-major, each lane's fragments as they stand in its registers;
// k_dn_wgrad forms dW = dz^T h per chunk of 1024 samples with MFMA (K =
// samples, transposed from those rows in registers) and bias sums; k_dn_reduce
// adds the chunk partials in a fixed order (deterministic gradients); k_dn_adam
// updates the FP32 master weights and re-packs their BF16 fragments.
#include <cmath>
#include <cstring>
#include <vector>

#include "internal.hpp"

namespace luz {

struct DnFrameDev {
    uint32_t width, height, num_lights, pad;
    const float* position;
    const float* normal;
    const uint8_t* shadow;
    const uint8_t* ao;
    float cam[3];
    float shadow_n, ao_n;
    float pad2;
    // per-pixel planes of the prepass: (camera distance or -1 on background,
    // normal.xyz) and the AO fraction
    const float4* pix;
    const float* ao_frac;
};

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kIn = LUZRT_DN_FEATURES, kHid = LUZRT_DN_HIDDEN, kOut = 2;
constexpr int kBlock = 256;
constexpr uint32_t kChunkRows = 1024;
constexpr int kX = 192;   // positions of a training row's inputs: 6 K-steps of 32, 42 of them zero
// inference: one 16-pixel tile per wave at a time, 8 waves per group sharing
// one copy of the weights in LDS
constexpr int kInferBlock = 512;
constexpr uint32_t kInferRounds = 4;   // bands of tiles per chunk an XCD sweeps in order

constexpr int oW1 = 0, oB1 = oW1 + kHid * kIn;
constexpr int oW2 = oB1 + kHid, oB2 = oW2 + kHid * kHid;
constexpr int oW3 = oB2 + kHid, oB3 = oW3 + kHid * kHid;
constexpr int oW4 = oB3 + kHid, oB4 = oW4 + kHid * kHid;
constexpr int oW5 = oB4 + kHid, oB5 = oW5 + kOut * kHid;
constexpr int kParams = oB5 + kOut;
static_assert(kParams == LUZRT_DN_PARAMS, "parameter count");
constexpr int kWOff[5] = {oW1, oW2, oW3, oW4, oW5};
constexpr int kBOff[5] = {oB1, oB2, oB3, oB4, oB5};

// Fragment table (one fragment = 64 lanes x 8 BF16 = 1 KB):
//   F2..F4(t,s) t<4 s<2 | G2..G4(t,s) | G5(t) t<4 | FG(t,s) t<4 s<5 | FV(t) t<4
//   | F5(s) s<2
// In training layer 5 (64 -> 2) runs in FP32 (dn_out_fp32); G5 holds W5^T for
// the backward pass.
// FG and FV hold layer 1 in an order that splits the features of a (pixel,
// light) sample into the 125 that do not depend on the light (one product per
// pixel in inference) and the 25 visibilities (one K-step per light).
// Lane group g only ever reads neighbours 8g .. 8g + 7 (those below 25):
//   FG, K-steps s < 4: element e is channel (AO, n.x, n.y, n.z)[e % 4] of
//       neighbour 8g + 2s + e / 4;
//   FG, K-step 4: element e is the relative depth of neighbour 8g + e;
//   FV: element e is the visibility of neighbour 8g + e.
// F5(s) s < 2 holds layer 5 for inference, where it runs on MFMA: output row 0
// and 1 are the BF16 rounding of W5's rows, rows 2 and 3 the BF16 rounding of
// what that leaves (W5 - hi), rows 4..15 zero, K in the hidden-layer order.
constexpr int kF2 = 0, kF3 = 8, kF4 = 16, kG2 = 24, kG3 = 32, kG4 = 40, kG5 = 48, kFG = 52, kFV = 72,
              kF5 = 76, kFragTrain = 76, kFragAll = 78;
// inference fragments in LDS: F2..F4 (24), then FG and FV (24), then F5 (2)
constexpr int kIF2 = 0, kIF3 = 8, kIF4 = 16, kIFG = 24, kIFV = 44, kIF5 = 48, kFragInfer = 50;

// Original feature index (6 n + channel) of element e of lane group g in
// inference K-step s (s == 5: the visibility step), or -1 for padding.
__host__ __device__ inline int infer_feature(int s, int g, int e) {
    if (s < 4) {
        const int n = 8 * g + 2 * s + (e >> 2), ch = e & 3;
        return n < 25 ? 6 * n + (ch == 0 ? 0 : ch + 2) : -1;
    }
    const int n = 8 * g + e;
    if (n >= 25) return -1;
    return s == 4 ? 6 * n + 2 : 6 * n + 1;
}

__host__ __device__ inline int khid(int s, int g, int e) { return 16 * (2 * s + (e >> 2)) + 4 * g + (e & 3); }

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// BF16 of two finite floats, round to nearest even (v_cvt_pk_bf16_f32): a in
// the low half, b in the high half.
__device__ inline uint32_t bf16_pack2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}
__device__ inline uint32_t bf16_bits(float f) { return bf16_pack2(f, 0.0f) & 0xFFFFu; }
// max(z, 0) for finite z on the bit pattern (negative floats are negative integers)
__device__ inline float relu_bits(float z) {
    const int b = __float_as_int(z);
    return __int_as_float(b > 0 ? b : 0);
}
__device__ inline float bf16_val(uint32_t h) { return __uint_as_float(h << 16); }
__device__ inline float clamp01f(float a) { return a < 0.0f ? 0.0f : (a > 1.0f ? 1.0f : a); }
__device__ inline bf16x8 as_bf16x8(uint4 q) { return __builtin_bit_cast(bf16x8, q); }
__device__ inline f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

struct DnArgs {
    DnFrameDev F;
    const uint4* frags;
    const float* params;
    uint32_t nsamples;
    uint32_t lights;           // max(L, 1)
    const uint32_t* samples;   // pixel | light << 24
    const float* target_ao;    // [npix]
    const float* target_vis;   // [L][npix]
    uint32_t row_base, cap;    // first training row of this call, rows of an array
    uint4* X;                  // [cap][kX] BF16, K-step order (infer_feature)
    uint4* H;                  // [4][cap][64] BF16, feature 16t + 4g + i at 16g + 4t + i
    uint4* Z;                  // [4][cap][64] BF16, likewise
    uint32_t* Y;               // [cap] two BF16
    float grad_scale;          // dLoss/dy = grad_scale * (y - target)
    float* loss_sum;
};

// The 6 channels of neighbour (qx, qy) of a pixel at distance dc from the camera.
struct Nb { float c0, c1, c2, c3, c4, c5; };

__device__ inline Nb dn_neighbour(const DnFrameDev& F, uint32_t qx, uint32_t qy, uint32_t light, float dc) {
    const size_t q = (size_t)qy * F.width + qx;
    const float4 px = F.pix[q];
    Nb r;
    if (px.x < 0.0f) {   // background
        r.c0 = 0.0f; r.c1 = 0.0f; r.c2 = 1.0f; r.c3 = 0.0f; r.c4 = 0.0f; r.c5 = 0.0f;
        return r;
    }
    const float d = px.x;
    r.c0 = F.ao_frac[q];
    r.c1 = F.num_lights ? 1.0f - (float)F.shadow[(size_t)light * F.width * F.height + q] / F.shadow_n
                        : 0.0f;
    float rel = dc > 0.0f ? (d - dc) / dc * 16.0f : 0.0f;
    r.c2 = rel < -1.0f ? -1.0f : (rel > 1.0f ? 1.0f : rel);
    r.c3 = px.y; r.c4 = px.z; r.c5 = px.w;
    return r;
}

// Prepass: camera distance (-1 on background pixels, whose normal is zero),
// normal and AO fraction of every pixel, each computed once per frame.
__global__ __launch_bounds__(256) void k_dn_prep(DnFrameDev F, float4* pix, float* ao_frac) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= F.width * F.height) return;
    const float* n = F.normal + (size_t)p * 3;
    const float nx = n[0], ny = n[1], nz = n[2];
    if (vlen(v3(nx, ny, nz)) == 0.0f) {
        pix[p] = make_float4(-1.0f, 0.0f, 0.0f, 0.0f);
        ao_frac[p] = 0.0f;
        return;
    }
    const float* P = F.position + (size_t)p * 3;
    const float d = vlen(v3(P[0] - F.cam[0], P[1] - F.cam[1], P[2] - F.cam[2]));
    pix[p] = make_float4(d, nx, ny, nz);
    ao_frac[p] = (float)F.ao[p] / F.ao_n;
}

__device__ inline float nb_channel(const Nb& b, int c) {
    return c == 0 ? b.c0 : c == 1 ? b.c1 : c == 2 ? b.c2 : c == 3 ? b.c3 : c == 4 ? b.c4 : b.c5;
}

// Features f0 .. f0+7 (BF16 bits, element e in half e of the uint4) of the sample
// at pixel (x, y), light `light`; zero beyond 150 and for invalid samples.
__device__ inline uint4 dn_features(const DnFrameDev& F, bool valid, uint32_t x, uint32_t y,
                                   uint32_t light, float dc, int f0) {
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    if (valid) {
        int cur = -1;
        Nb nb{};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            int f = f0 + e;
            if (f < kIn) {
                int n = f / 6, c = f - n * 6;
                if (n != cur) {
                    int dx = n % 5 - 2, dy = n / 5 - 2;
                    int qx = (int)x + dx, qy = (int)y + dy;
                    qx = qx < 0 ? 0 : (qx >= (int)F.width ? (int)F.width - 1 : qx);
                    qy = qy < 0 ? 0 : (qy >= (int)F.height ? (int)F.height - 1 : qy);
                    nb = dn_neighbour(F, (uint32_t)qx, (uint32_t)qy, light, dc);
                    cur = n;
                }
                w[e >> 1] |= bf16_bits(nb_channel(nb, c)) << (16 * (e & 1));
            }
        }
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// ReLU of a hidden layer's 4x4 tiles of one sample column (training; the bias
// is in the accumulators): the next layer's B fragments and the ReLU mask (bit
// t * 4 + i).
__device__ inline void dn_hidden_epilogue(const f32x4 (&acc)[4], uint4 (&hb)[2], uint32_t& mask) {
    uint32_t w[2][4];
    mask = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        float h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool on = acc[t][i] > 0.0f;
            h[i] = on ? acc[t][i] : 0.0f;
            mask |= (on ? 1u : 0u) << (t * 4 + i);
        }
        // elements e = (t & 1) * 4 + i of K-step s = t / 2
#pragma unroll
        for (int i = 0; i < 4; i += 2) w[t >> 1][((t & 1) * 4 + i) >> 1] = bf16_pack2(h[i], h[i + 1]);
    }
    hb[0] = make_uint4(w[0][0], w[0][1], w[0][2], w[0][3]);
    hb[1] = make_uint4(w[1][0], w[1][1], w[1][2], w[1][3]);
}

typedef short s16x2 __attribute__((ext_vector_type(2)));

// ReLU of a hidden layer's 4x4 tiles (bias already in the accumulators) into
// the next layer's B fragments (inference).  The ReLU is taken after rounding,
// on each BF16 half as a signed 16-bit integer (v_pk_max_i16 with 0): a value
// with its sign bit set, -0 and negative NaN included, becomes +0, as
// relu_bits before the rounding gives, and every other value is kept.
__device__ inline void dn_relu_pack(const f32x4 (&acc)[4], uint4 (&hb)[2]) {
    uint32_t w[2][4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
            const s16x2 h = __builtin_bit_cast(s16x2, bf16_pack2(acc[t][i], acc[t][i + 1]));
            w[t >> 1][((t & 1) * 4 + i) >> 1] =
                __builtin_bit_cast(uint32_t, __builtin_elementwise_max(h, (s16x2){0, 0}));
        }
    hb[0] = make_uint4(w[0][0], w[0][1], w[0][2], w[0][3]);
    hb[1] = make_uint4(w[1][0], w[1][1], w[1][2], w[1][3]);
}

// Layer 5 in FP32: the two outputs (without bias) of sample column j from the
// FP32 activations of layer 4 (lane (j, g) holds features 16t + 4g + i) and
// FP32 weights w5 ([2][64]); per lane in (t, i) order, then over the lane
// groups as ((g0 + g1) + (g2 + g3)).  FP32 keeps a correction that the weights
// cancel to about zero as precise as the box base it is added to.
__device__ inline void dn_out_fp32(const f32x4 (&h)[4], const float* w5, int g, float& y0, float& y1) {
    float p0 = 0.0f, p1 = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&w5[16 * t + 4 * g]);
        const f32x4 b = *reinterpret_cast<const f32x4*>(&w5[kHid + 16 * t + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            p0 = fmaf(a[i], h[t][i], p0);
            p1 = fmaf(b[i], h[t][i], p1);
        }
    }
    p0 += __shfl_xor(p0, 16);
    p1 += __shfl_xor(p1, 16);
    p0 += __shfl_xor(p0, 32);
    p1 += __shfl_xor(p1, 32);
    y0 = p0;
    y1 = p1;
}

// A 64 -> 64 layer (2 K-steps) on top of the accumulators: acc[t] += sum_s
// frag(t, s) * hb[s].
__device__ inline void dn_layer64(const uint4* sfrag, int fbase, int lane, const uint4 (&hb)[2],
                                  f32x4 (&acc)[4]) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t)
            acc[t] = mfma(as_bf16x8(sfrag[(fbase + t * 2 + s) * 64 + lane]), as_bf16x8(hb[s]), acc[t]);
}

// Backward through a hidden layer's ReLU: dz = dh * mask as the B fragments of
// the layer below (and as they are stored).
__device__ inline void dn_relu_back(const f32x4 (&dh)[4], uint32_t mask, uint4 (&zb)[2]) {
    uint32_t w[2][4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
            const float d0 = (mask >> (t * 4 + i)) & 1u ? dh[t][i] : 0.0f;
            const float d1 = (mask >> (t * 4 + i + 1)) & 1u ? dh[t][i + 1] : 0.0f;
            w[t >> 1][((t & 1) * 4 + i) >> 1] = bf16_pack2(d0, d1);
        }
    zb[0] = make_uint4(w[0][0], w[0][1], w[0][2], w[0][3]);
    zb[1] = make_uint4(w[1][0], w[1][1], w[1][2], w[1][3]);
}

// Index of neighbour n (< 25) of pixel (x, y), clamped to the image.
__device__ inline uint32_t dn_nb_index(const DnFrameDev& F, uint32_t x, uint32_t y, int n) {
    int qx = (int)x + n % 5 - 2, qy = (int)y + n / 5 - 2;
    qx = qx < 0 ? 0 : (qx >= (int)F.width ? (int)F.width - 1 : qx);
    qy = qy < 0 ? 0 : (qy >= (int)F.height ? (int)F.height - 1 : qy);
    return (uint32_t)qy * F.width + (uint32_t)qx;
}

// Sum of a value over the four lane groups (rows of 16 lanes) of a pixel
// column, as ((g0 + g1) + (g2 + g3)), in every lane: v_permlane16_swap pairs
// rows 0/1 and 2/3, v_permlane32_swap the two halves (VALU exchanges, no LDS
// round trip).
__device__ inline float col_sum(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const float s = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ inline uint32_t col_sum(uint32_t v) {
    const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    const uint32_t s = a[0] + a[1];
    const auto b = __builtin_amdgcn_permlane32_swap(s, s, false, false);
    return b[0] + b[1];
}

// Training forward, loss and backward of explicit samples, 16 per wave at a
// time (lane column j: sample j).
//
// What bounds it is latency: a call has a few thousand samples, so each wave
// runs one chain of gather, five layers and four layers back once or twice.
// The gather is one trip: lane group g reads neighbours 8g .. 8g + 7 of each
// sample straight from the G-buffer and count planes, all loads in flight
// together, and the centre's distance comes from the lane that read it.  (In
// feature order, with the neighbour changing at another element in each lane
// group, the loads came one after the other, in 64-sample waves, behind a
// prepass over the frame, and the rows were stored in 2-byte pieces: 8192
// samples of a 256x256 frame took 150 us, now 21 us.)  16-sample waves rather
// than 64: four times as many waves to spread over the CUs.
__global__ __launch_bounds__(kBlock) void k_dn_forward(DnArgs A) {
    __shared__ uint4 sfrag[kFragTrain * 64];
    __shared__ __align__(16) float sbias[4 * kHid + 4];
    __shared__ __align__(16) float sw5[kOut * kHid];
    {
        constexpr int kPer = kFragTrain * 64 / kBlock;   // all of a thread's loads in flight together
        static_assert(kPer * kBlock == kFragTrain * 64, "whole fragments per thread");
        uint4 fr[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i) fr[i] = A.frags[i * kBlock + threadIdx.x];
#pragma unroll
        for (int i = 0; i < kPer; ++i) sfrag[i * kBlock + threadIdx.x] = fr[i];
    }
    for (int i = threadIdx.x; i < kOut * kHid; i += kBlock) sw5[i] = A.params[oW5 + i];
    for (int i = threadIdx.x; i < 4 * kHid + kOut; i += kBlock)
        sbias[i] = A.params[i < 4 * kHid ? kBOff[i / kHid] + i % kHid : oB5 + (i - 4 * kHid)];
    __syncthreads();
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t nwaves = gridDim.x * (kBlock / 64);
    const DnFrameDev& F = A.F;
    const uint32_t npix = F.width * F.height;
    // the sample count is a multiple of 64: every tile is whole
    for (uint32_t base = (blockIdx.x * (kBlock / 64) + wave) * 16u; base < A.nsamples; base += nwaves * 16u) {
        const uint32_t sm = A.samples[base + (uint32_t)j];
        uint32_t p = sm & 0xFFFFFFu, l = sm >> 24;
        // caller-supplied samples outside the frame contribute nothing
        const bool in_frame = p < npix && l < A.lights;
        if (!in_frame) { p = 0; l = 0; }
        const size_t row = A.row_base + base + (uint32_t)j;
        const uint32_t px = p % F.width, py = p / F.width;
        float d[8], n3[8][3], ao[8], vis[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t q = dn_nb_index(F, px, py, 8 * g + e < 25 ? 8 * g + e : 0);
            const float* N = F.normal + (size_t)q * 3;
            const float* P = F.position + (size_t)q * 3;
            const float dist = vlen(v3(P[0] - F.cam[0], P[1] - F.cam[1], P[2] - F.cam[2]));
            n3[e][0] = N[0]; n3[e][1] = N[1]; n3[e][2] = N[2];
            ao[e] = (float)F.ao[q] / F.ao_n;
            vis[e] = F.num_lights ? 1.0f - (float)F.shadow[(size_t)l * npix + q] / F.shadow_n : 0.0f;
            d[e] = vlen(v3(N[0], N[1], N[2])) == 0.0f ? -1.0f : dist;   // -1: background
        }
        const float t_ao = g == 0 ? A.target_ao[p] : 0.0f;
        const float t_vis = g == 0 && F.num_lights ? A.target_vis[(size_t)l * npix + p] : 0.0f;
        // the centre is neighbour 12: element 4 of lane group 1
        const float dcv = __shfl(d[4], 16 + j);
        const bool valid = in_frame && dcv >= 0.0f;
        const float dc = valid ? dcv : 0.0f;
        // ---- features (all zero for an invalid sample) and the sums of the box base
        uint4 xb[6];
        float sa = 0.0f, sv = 0.0f;
        uint32_t cnt = 0;
        {
            float rel[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bool in = valid && 8 * g + e < 25, bg = d[e] < 0.0f;
                const float r = dc > 0.0f ? (d[e] - dc) / dc * 16.0f : 0.0f;
                rel[e] = !in ? 0.0f : (bg ? 1.0f : (r < -1.0f ? -1.0f : (r > 1.0f ? 1.0f : r)));
                const bool fg = in && !bg;
                ao[e] = fg ? ao[e] : 0.0f;
                vis[e] = fg ? vis[e] : 0.0f;
#pragma unroll
                for (int c = 0; c < 3; ++c) n3[e][c] = fg ? n3[e][c] : 0.0f;
                sa += ao[e];
                sv += vis[e];
                cnt += fg ? 1u : 0u;
            }
#pragma unroll
            for (int s = 0; s < 4; ++s)
                xb[s] = make_uint4(bf16_pack2(ao[2 * s], n3[2 * s][0]), bf16_pack2(n3[2 * s][1], n3[2 * s][2]),
                                   bf16_pack2(ao[2 * s + 1], n3[2 * s + 1][0]),
                                   bf16_pack2(n3[2 * s + 1][1], n3[2 * s + 1][2]));
            xb[4] = make_uint4(bf16_pack2(rel[0], rel[1]), bf16_pack2(rel[2], rel[3]), bf16_pack2(rel[4], rel[5]),
                               bf16_pack2(rel[6], rel[7]));
            xb[5] = make_uint4(bf16_pack2(vis[0], vis[1]), bf16_pack2(vis[2], vis[3]), bf16_pack2(vis[4], vis[5]),
                               bf16_pack2(vis[6], vis[7]));
        }
#pragma unroll
        for (int s = 0; s < 6; ++s) A.X[row * (kX / 8) + s * 4 + g] = xb[s];
        // the base the outputs are added to: the means of the AO fraction and of
        // the visibility over the window's foreground pixels, summed as k_dn_infer does
        const uint32_t c = col_sum(cnt);
        const float fc = (float)(c ? c : 1u);
        const float bao = col_sum(sa) / fc, bvis = col_sum(sv) / fc;
        // ---- layer 1: 150 (192) -> 64
        f32x4 acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = *reinterpret_cast<const f32x4*>(&sbias[16 * t + 4 * g]);
#pragma unroll
        for (int s = 0; s < 6; ++s)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[t] = mfma(as_bf16x8(sfrag[(s < 5 ? kFG + t * 5 + s : kFV + t) * 64 + lane]), as_bf16x8(xb[s]),
                              acc[t]);
        uint4 hb[2];
        uint32_t mask[4];
        // ---- layers 2..4: 64 -> 64
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (k > 0) {
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[t] = *reinterpret_cast<const f32x4*>(&sbias[k * kHid + 16 * t + 4 * g]);
                dn_layer64(sfrag, k == 1 ? kF2 : (k == 2 ? kF3 : kF4), lane, hb, acc);
            }
            dn_hidden_epilogue(acc, hb, mask[k]);
            uint4* h = A.H + ((size_t)k * A.cap + row) * 8 + 2 * g;
            h[0] = hb[0];
            h[1] = hb[1];
        }
        // ---- layer 5: 64 -> 2 in FP32 on layer 4's activations (as in dn_hidden_epilogue)
        float o0, o1;
        {
            f32x4 h[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) h[t][i] = acc[t][i] > 0.0f ? acc[t][i] : 0.0f;
            dn_out_fp32(h, sw5, g, o0, o1);
        }
        // ---- loss and backward
        float loss = 0.0f, d0 = 0.0f, d1 = 0.0f;
        if (g == 0 && valid) {
            const float e0 = (o0 + sbias[4 * kHid]) + bao - t_ao;
            const float e1 = (o1 + sbias[4 * kHid + 1]) + bvis - t_vis;
            loss = e0 * e0 + e1 * e1;
            d0 = A.grad_scale * e0;
            d1 = A.grad_scale * e1;
        }
        const uint32_t b01 = bf16_pack2(d0, d1);
        if (g == 0) A.Y[row] = b01;
        // dh4 = W5^T dy
        const uint4 db = make_uint4(g == 0 ? b01 : 0u, 0u, 0u, 0u);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            acc[t] = mfma(as_bf16x8(sfrag[(kG5 + t) * 64 + lane]), as_bf16x8(db), f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
        for (int k = 3; k >= 0; --k) {
            uint4 zb[2];
            dn_relu_back(acc, mask[k], zb);
            uint4* z = A.Z + ((size_t)k * A.cap + row) * 8 + 2 * g;
            z[0] = zb[0];
            z[1] = zb[1];
            if (k == 0) break;
            // dh_{k} = W_{k+1}^T dz_{k+1}  (fragments G2..G4 hold W2^T..W4^T)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            dn_layer64(sfrag, k == 3 ? kG4 : (k == 2 ? kG3 : kG2), lane, zb, acc);
        }
        // per-wave loss sum (lanes g == 0 hold the outputs)
        for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off);
        if (lane == 0) atomicAdd(A.loss_sum, loss);
    }
}

struct InferArgs {
    DnFrameDev F;
    const uint4* frags;
    const float* params;
    uint32_t lights;    // max(L, 1)
    uint32_t ntiles;    // 16-pixel tiles of the frame
    float* ao_out;      // [npix]
    float* vis_out;     // [L][npix]
};

// The per-pixel state a tile's light groups share: lane (j, g) holds pixel j
// of the tile and neighbours 8g + e (e < 8) of its 5x5 window.
struct InferTile {
    uint32_t vq[8];   // neighbour indices (0 off the window and for invalid pixels)
    uint32_t bo[8];   // visibility table offset: 0 for a foreground neighbour, else
                      // 2048 bytes (the table's zero half)
    float cnt, bao;   // foreground pixels of the window, box base of AO
    uint32_t pp;      // pixel index (0 beyond the frame)
    bool valid, inb;
};

// Buffer resource over `bytes` bytes at p for raw loads (32-bit offsets in a
// VGPR, no 64-bit address arithmetic per load).
__device__ inline __amdgpu_buffer_rsrc_t buf_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}

// The prepass record (camera distance or -1, normal) of pixel q.
__device__ inline float4 load_pix(__amdgpu_buffer_rsrc_t r, uint32_t q) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, q * 16u, 0, 0);
    return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}

// The shadow bytes of lights l0 .. l0+2 (clamped to the last light) at the
// tile's neighbour indices.
__device__ inline void dn_shadow_bytes(const DnFrameDev& F, uint32_t l0, const uint32_t (&vq)[8],
                                       uint32_t (&s8)[3][8]) {
    const uint32_t npix = F.width * F.height;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        const uint32_t l = l0 + p < F.num_lights ? l0 + p : F.num_lights - 1;
        const __amdgpu_buffer_rsrc_t r = buf_rsrc(F.shadow + (size_t)l * npix, npix);
#pragma unroll
        for (int e = 0; e < 8; ++e) s8[p][e] = __builtin_amdgcn_raw_buffer_load_b8(r, vq[e], 0, 0);
    }
}

// Lights l0 .. l0+P-1 of one 16-pixel tile: the visibility K-step FV on top of
// the light-independent accumulators `ag`, then layers 2..5 on MFMA.  Every
// weight fragment and bias read from LDS feeds the products of all P lights;
// the caller loaded the group's shadow bytes `s8`.  AO outputs are added to
// `aosum` in light order; the visibilities are written.
//
// Layer 5 takes layer 4's activations in BF16, as every other layer takes its
// inputs, and W5 as the sum of two BF16 parts (F5), so only the activation
// rounding (relative 2^-9 per term) separates it from the FP32 layer 5 of
// training.
template <int P>
__device__ inline void dn_light_group(const InferArgs& A, const uint4* sfrag, const float* sbias,
                                      const uint2* svt, uint32_t l0, int lane, int g,
                                      const f32x4 (&ag)[4], const InferTile& T, const uint32_t (&s8)[3][8],
                                      float b50, float b51, float& aosum) {
    const DnFrameDev& F = A.F;
    const uint32_t npix = F.width * F.height;
    const uint32_t L = F.num_lights;
    // the weight fragments are read from LDS at every use: an opaque lane
    // offset keeps the compiler from holding all 28 of them in registers
    // across the groups (which would leave one wave per SIMD)
    uint32_t ln = (uint32_t)lane;
    asm volatile("" : "+v"(ln));
    f32x4 acc[P][4];
    uint4 hb[P][2];
    float bvis[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        uint32_t w[4] = {0u, 0u, 0u, 0u};
        float sv = 0.0f;
        if (L) {
            // (BF16 bits, FP32 bits) of 1 - s / shadow_n, or zeros (+0.0f, which
            // the sum keeps) for a neighbour off the foreground
            uint2 tv[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
                tv[e] = *reinterpret_cast<const uint2*>(reinterpret_cast<const char*>(svt) +
                                                        ((s8[p][e] << 3) | T.bo[e]));
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                w[e >> 1] |= tv[e].x << (16 * (e & 1));
                sv += __uint_as_float(tv[e].y);
            }
        }
        bvis[p] = col_sum(sv) / T.cnt;
        hb[p][0] = make_uint4(w[0], w[1], w[2], w[3]);   // the visibility B operand
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const bf16x8 a = as_bf16x8(sfrag[(kIFV + t) * 64 + ln]);
#pragma unroll
        for (int p = 0; p < P; ++p) acc[p][t] = mfma(a, as_bf16x8(hb[p][0]), ag[t]);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) dn_relu_pack(acc[p], hb[p]);
#pragma unroll
    for (int k = 1; k < 4; ++k) {
        const int fb = k == 1 ? kIF2 : (k == 2 ? kIF3 : kIF4);
        uint4 fr[8];   // fragment (t, s) at t * 2 + s, all 8 in flight together
#pragma unroll
        for (int i = 0; i < 8; ++i) fr[i] = sfrag[(fb + i) * 64 + ln];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const f32x4 bk = *reinterpret_cast<const f32x4*>(&sbias[k * kHid + 16 * t + 4 * g]);
#pragma unroll
            for (int p = 0; p < P; ++p) acc[p][t] = bk;
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bf16x8 a = as_bf16x8(fr[t * 2 + s]);
#pragma unroll
                for (int p = 0; p < P; ++p) acc[p][t] = mfma(a, as_bf16x8(hb[p][s]), acc[p][t]);
            }
#pragma unroll
        for (int p = 0; p < P; ++p) dn_relu_pack(acc[p], hb[p]);
    }
    // layer 5: lane group 0 receives rows 0..3 of its pixel column, the high
    // and low parts of the two outputs
    f32x4 y[P];
    {
        const bf16x8 a0 = as_bf16x8(sfrag[(kIF5 + 0) * 64 + ln]), a1 = as_bf16x8(sfrag[(kIF5 + 1) * 64 + ln]);
#pragma unroll
        for (int p = 0; p < P; ++p) y[p] = mfma(a0, as_bf16x8(hb[p][0]), f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
        for (int p = 0; p < P; ++p) y[p] = mfma(a1, as_bf16x8(hb[p][1]), y[p]);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        if (g == 0 && T.inb) {
            const float o0 = y[p][0] + y[p][2], o1 = y[p][1] + y[p][3];
            aosum += T.valid ? (o0 + b50) + T.bao : 0.0f;
            if (L)
                A.vis_out[(size_t)(l0 + p) * npix + T.pp] = T.valid ? clamp01f((o1 + b51) + bvis[p]) : 0.0f;
        }
    }
}

// Inference, one 16-pixel tile per wave at a time (lane column j: pixel j of
// the tile): the light-independent part of layer 1 once per pixel (K-steps FG,
// bias folded into the accumulators), then the lights in groups of 3 (the
// last group 1 or 2), each light with the visibility K-step FV on top of it
// and layers 2..5.  A pixel's AO is the mean of its lights' AO outputs, summed
// in light order; background pixels give 0.
__global__ __launch_bounds__(kInferBlock, 2) void k_dn_infer(InferArgs A) {
    __shared__ uint4 sfrag[kFragInfer * 64];
    __shared__ __align__(16) float sbias[4 * kHid + 4];
    __shared__ uint2 svt[512];   // (BF16 bits, FP32 bits) of 1 - s / shadow_n; zeros
    for (int i = threadIdx.x; i < 24 * 64; i += kInferBlock) sfrag[kIF2 * 64 + i] = A.frags[kF2 * 64 + i];
    for (int i = threadIdx.x; i < 24 * 64; i += kInferBlock) sfrag[kIFG * 64 + i] = A.frags[kFG * 64 + i];
    for (int i = threadIdx.x; i < 2 * 64; i += kInferBlock) sfrag[kIF5 * 64 + i] = A.frags[kF5 * 64 + i];
    for (int i = threadIdx.x; i < 4 * kHid + kOut; i += kInferBlock)
        sbias[i] = A.params[i < 4 * kHid ? kBOff[i / kHid] + i % kHid : oB5 + (i - 4 * kHid)];
    const DnFrameDev& F = A.F;
    for (int i = threadIdx.x; i < 256; i += kInferBlock) {
        const float v = 1.0f - (float)i / F.shadow_n;
        svt[i] = make_uint2(bf16_bits(v), __float_as_uint(v));
        svt[256 + i] = make_uint2(0u, 0u);
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const uint32_t npix = F.width * F.height;
    const uint32_t L = F.num_lights;
    // The tiles go out in chunks of kInferRounds bands (a band: one tile per
    // wave of an XCD), chunk c to XCD c % 8 (blocks are dispatched round-robin
    // over the 8 XCDs): an XCD's waves sweep each of its chunks band after
    // band, so the window rows that neighbouring bands share are still in its
    // L2 when the next band reads them, and the chunks interleave the image
    // over the XCDs, which keeps their work even where whole regions are
    // background.  With a grid not a multiple of 8 every wave strides alone.
    const uint32_t nb = gridDim.x, wpb = kInferBlock / 64;
    const bool xcd = nb % 8 == 0;
    const uint32_t W = xcd ? (nb / 8) * wpb : nb * wpb;   // waves per band
    const uint32_t wx = (xcd ? blockIdx.x / 8 : blockIdx.x) * wpb + (threadIdx.x >> 6);
    const uint32_t c0 = xcd ? blockIdx.x % 8 : 0u, cstep = xcd ? 8u : 1u;
    const uint32_t C = kInferRounds * W;                   // tiles per chunk
    const float b50 = sbias[4 * kHid], b51 = sbias[4 * kHid + 1];
    const __amdgpu_buffer_rsrc_t rpix = buf_rsrc(F.pix, npix * 16u), rao = buf_rsrc(F.ao_frac, npix * 4u);
    for (uint32_t k = 0;; ++k) {
        const uint32_t base = (c0 + cstep * (k / kInferRounds)) * C;   // first tile of the chunk
        if (base >= A.ntiles) break;
        const uint32_t tile = base + (k % kInferRounds) * W + wx;
        if (tile >= A.ntiles) continue;   // the frame's last chunk ends early
        InferTile T;
        const uint32_t p = tile * 16u + (uint32_t)j;
        T.inb = p < npix;
        T.pp = T.inb ? p : 0u;
        const float d = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rpix, T.pp * 16u, 0, 0));
        T.valid = T.inb && d >= 0.0f;
        const float dc = T.valid ? d : 0.0f;
        const uint32_t px = T.pp % F.width, py = T.pp / F.width;
        if (__ballot(T.valid) == 0ull) {
            if (g == 0 && T.inb) {
                A.ao_out[T.pp] = 0.0f;
                for (uint32_t l = 0; l < L; ++l) A.vis_out[(size_t)l * npix + T.pp] = 0.0f;
            }
            continue;
        }
        // ---- layer 1, light-independent features: K-steps 0..3 (AO, normal)
        // of neighbours 8g + 2s + e / 4, then K-step 4: relative depth of
        // neighbours 8g + e, and the neighbour indices and foreground bits that
        // the visibility step reads per light.  Every neighbour index is
        // clamped to the image, so all loads are issued before the first is
        // used (invalid pixels and neighbours beyond the 25th select zeros).
        uint32_t nv[8];
        float4 vv[8];
        float av[8];
        bool in[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            nv[e] = dn_nb_index(F, px, py, 8 * g + e < 25 ? 8 * g + e : 0);
            in[e] = T.valid && 8 * g + e < 25;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            vv[e] = load_pix(rpix, nv[e]);
            av[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rao, nv[e] * 4u, 0, 0));
        }
        f32x4 ag[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) ag[t] = *reinterpret_cast<const f32x4*>(&sbias[16 * t + 4 * g]);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            uint32_t w[4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = 2 * s + h;
                const float4 v = in[e] ? vv[e] : make_float4(-1.0f, 0.0f, 0.0f, 0.0f);
                const float ao = v.x >= 0.0f ? av[e] : 0.0f;
                w[2 * h] = bf16_pack2(ao, v.y);     // background normals are zero
                w[2 * h + 1] = bf16_pack2(v.z, v.w);
            }
            const bf16x8 fb = as_bf16x8(make_uint4(w[0], w[1], w[2], w[3]));
#pragma unroll
            for (int t = 0; t < 4; ++t) ag[t] = mfma(as_bf16x8(sfrag[(kIFG + t * 5 + s) * 64 + lane]), fb, ag[t]);
        }
        {
            float f[8];
            float sa = 0.0f;
            uint32_t vfg = 0u;   // foreground bits of the neighbours 8g + e
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float dn = vv[e].x;
                const bool fg = in[e] && dn >= 0.0f;
                T.vq[e] = in[e] ? nv[e] : 0u;
                T.bo[e] = fg ? 0u : 2048u;
                vfg |= (fg ? 1u : 0u) << e;
                sa += fg ? av[e] : 0.0f;
                const float rel = dc > 0.0f ? (dn - dc) / dc * 16.0f : 0.0f;
                f[e] = !in[e] ? 0.0f : (!fg ? 1.0f : (rel < -1.0f ? -1.0f : (rel > 1.0f ? 1.0f : rel)));
            }
            const bf16x8 fb = as_bf16x8(make_uint4(bf16_pack2(f[0], f[1]), bf16_pack2(f[2], f[3]),
                                                   bf16_pack2(f[4], f[5]), bf16_pack2(f[6], f[7])));
            // sums over the four lane groups of a pixel column: ((g0 + g1) + (g2 + g3))
            sa = col_sum(sa);
            const uint32_t c = col_sum((uint32_t)__popc(vfg));
            T.cnt = (float)(c ? c : 1u);
            T.bao = sa / T.cnt;
#pragma unroll
            for (int t = 0; t < 4; ++t) ag[t] = mfma(as_bf16x8(sfrag[(kIFG + t * 5 + 4) * 64 + lane]), fb, ag[t]);
        }
        // ---- per light group: visibility K-step, layers 2..5
        float aosum = 0.0f;
        const uint32_t nl = A.lights;
        uint32_t sb[3][8];
        if (L) dn_shadow_bytes(F, 0, T.vq, sb);
        uint32_t l = 0;
        for (; l + 3 <= nl; l += 3) {
            if (L && l > 0) dn_shadow_bytes(F, l, T.vq, sb);
            dn_light_group<3>(A, sfrag, sbias, svt, l, lane, g, ag, T, sb, b50, b51, aosum);
        }
        if (L && l > 0 && l < nl) dn_shadow_bytes(F, l, T.vq, sb);
        if (nl - l == 2)
            dn_light_group<2>(A, sfrag, sbias, svt, l, lane, g, ag, T, sb, b50, b51, aosum);
        else if (nl - l == 1)
            dn_light_group<1>(A, sfrag, sbias, svt, l, lane, g, ag, T, sb, b50, b51, aosum);
        if (g == 0 && T.inb) A.ao_out[T.pp] = clamp01f(aosum / (float)nl);
    }
}

// dW[o][i] = sum_n dz[o][n] h[i][n] over one chunk of samples, in jobs of 64
// input positions (blockIdx.y: 0..2 layer 1, whose rows have 192, 3..5 layers
// 2..4, 6 layer 5); bias gradients = sum_n dz[o][n].  One partial per chunk.
//
// The rows are sample-major as k_dn_forward's lanes wrote them (whole lines;
// the feature-major form they had before was stored in 2-byte pieces and read
// with a stride of the batch capacity: 105 us for 65536 rows, now 19 us).  Lane
// (j, g) reads positions 4j .. 4j + 3 of samples 8g .. 8g + 7 of a K-step and
// transposes them in registers into four fragments, fragment t holding position
// 4j + t in row j.  A wave takes a quarter of the chunk for all 16 tiles of the
// job, and the four waves' sums are added in order.
struct WgArgs {
    const uint2* X;
    const uint2* H;
    const uint2* Z;
    const uint4* Y;
    uint32_t cap, rows;
    float* partial;   // [chunks][kParams]
};
constexpr int kWgJobs = 7;

// The four fragments of rows v[k] (sample k, positions 4j .. 4j + 3).
__device__ inline void wg_fragments(const uint2 (&v)[8], bf16x8 (&f)[4]) {
    uint32_t w[4][4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        w[0][m] = __builtin_amdgcn_perm(v[2 * m + 1].x, v[2 * m].x, 0x05040100u);
        w[1][m] = __builtin_amdgcn_perm(v[2 * m + 1].x, v[2 * m].x, 0x07060302u);
        w[2][m] = __builtin_amdgcn_perm(v[2 * m + 1].y, v[2 * m].y, 0x05040100u);
        w[3][m] = __builtin_amdgcn_perm(v[2 * m + 1].y, v[2 * m].y, 0x07060302u);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) f[t] = as_bf16x8(make_uint4(w[t][0], w[t][1], w[t][2], w[t][3]));
}

// Feature of position p of a 64-wide row.
__device__ inline int wg_feature(int p) { return 16 * ((p >> 2) & 3) + 4 * (p >> 4) + (p & 3); }

__global__ __launch_bounds__(kBlock) void k_dn_wgrad(WgArgs A) {
    __shared__ f32x4 sacc[kBlock / 64][16 * 64];
    __shared__ f32x4 sb[kBlock / 64][4 * 4];
    const int job = blockIdx.y, layer = job < 3 ? 0 : job - 2;
    const bool out = layer == 4;   // the output layer: its dz is the two values of Y
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const int wave = threadIdx.x >> 6;
    const uint2* Z = out ? nullptr : A.Z + (size_t)layer * A.cap * 16 + j;
    const uint32_t hstep = layer == 0 ? kX / 4 : 16;   // 8-byte words of a row
    const uint2* H = layer == 0 ? A.X + job * 16 + j : A.H + (size_t)(layer - 1) * A.cap * 16 + j;
    const uint32_t n_begin = blockIdx.x * kChunkRows;
    const uint32_t n_end = n_begin + kChunkRows < A.rows ? n_begin + kChunkRows : A.rows;
    const bf16x8 ones = as_bf16x8(make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u));
    f32x4 acc[4][4], bias[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        bias[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[t][u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // rows are a multiple of 64, so every K-step of 32 samples is whole; the
    // next K-step's rows are loaded while this one's are multiplied
    uint2 hv[8], zv[8];
    auto load = [&](uint32_t n0) {
        const size_t n = n0 + 8u * (uint32_t)g;
#pragma unroll
        for (int k = 0; k < 8; ++k) hv[k] = H[(n + k) * hstep];
        if (out) {
            const uint4 ya = A.Y[n / 4], yb = A.Y[n / 4 + 1];
            zv[0] = make_uint2(ya.x, ya.y);
            zv[1] = make_uint2(ya.z, ya.w);
            zv[2] = make_uint2(yb.x, yb.y);
            zv[3] = make_uint2(yb.z, yb.w);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) zv[k] = Z[(n + k) * 16];
        }
    };
    uint32_t n0 = n_begin + 32u * (uint32_t)wave;
    if (n0 < n_end) load(n0);
    while (n0 < n_end) {
        bf16x8 fz[4], fh[4];
        wg_fragments(hv, fh);
        if (out) {
            // row j < 2 is output j: its half of each sample's pair
            const uint32_t sel = j == 0 ? 0x05040100u : 0x07060302u;
            uint32_t w[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) w[m] = j < 2 ? __builtin_amdgcn_perm(zv[m].y, zv[m].x, sel) : 0u;
            fz[0] = as_bf16x8(make_uint4(w[0], w[1], w[2], w[3]));
        } else {
            wg_fragments(zv, fz);
        }
        n0 += 32u * (kBlock / 64);
        if (n0 < n_end) load(n0);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (out && t > 0) break;
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[t][u] = mfma(fz[t], fh[u], acc[t][u]);
            bias[t] = mfma(fz[t], ones, bias[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int u = 0; u < 4; ++u) sacc[wave][(t * 4 + u) * 64 + lane] = acc[t][u];
        if (j == 0) sb[wave][t * 4 + g] = bias[t];
    }
    __syncthreads();
    // wave t adds the tiles (t, 0..3) of the four waves: lane (j, g), element i
    // is dz row 4g + i (position 4 (4g + i) + t), input column j (position 4j + u)
    const int t = wave;
    if (out && t > 0) return;
    const int nin = layer == 0 ? kIn : kHid;
    float* part = A.partial + (size_t)blockIdx.x * kParams;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        f32x4 v = sacc[0][(t * 4 + u) * 64 + lane];
        for (int w = 1; w < kBlock / 64; ++w) v += sacc[w][(t * 4 + u) * 64 + lane];
        int in = 4 * j + u;
        if (layer == 0) {
            const int q = 64 * job + in;
            in = infer_feature(q / 32, (q & 31) >> 3, q & 7);
        } else {
            in = wg_feature(in);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 4 * g + i, o = out ? r : wg_feature(4 * r + t);
            if (in >= 0 && (!out || r < kOut)) part[kWOff[layer] + o * nin + in] = v[i];
        }
    }
    if (j == 0 && (job == 0 || job >= 3)) {
        f32x4 v = sb[0][t * 4 + g];
        for (int w = 1; w < kBlock / 64; ++w) v += sb[w][t * 4 + g];
        for (int i = 0; i < 4; ++i) {
            const int r = 4 * g + i;
            if (!out || r < kOut) part[kBOff[layer] + (out ? r : wg_feature(4 * r + t))] = v[i];
        }
    }
}

// The chunk partials added in order, four threads per parameter (each a
// quarter of the chunks, so that the loads of a long batch overlap).
__global__ __launch_bounds__(kBlock) void k_dn_reduce(const float* partial, uint32_t chunks, float* grad) {
    __shared__ float sh[kBlock];
    const uint32_t i = blockIdx.x * (kBlock / 4) + (threadIdx.x & 63u), q = threadIdx.x >> 6;
    const uint32_t per = (chunks + 3) / 4, c0 = q * per, c1 = c0 + per < chunks ? c0 + per : chunks;
    float s = 0.0f;
    if (i < (uint32_t)kParams) {
#pragma unroll 8
        for (uint32_t c = c0; c < c1; ++c) s += partial[(size_t)c * kParams + i];
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    if (q == 0 && i < (uint32_t)kParams) grad[i] = ((sh[threadIdx.x] + sh[64 + threadIdx.x]) + sh[128 + threadIdx.x]) + sh[192 + threadIdx.x];
}

// Writes parameter i (value w) to its places in the BF16 fragments.
__device__ inline void dn_pack_param(uint32_t i, float w, uint16_t* frags) {
    auto put = [&](int f, int row, int g, int e, float v) {
        frags[((size_t)f * 64 + row + 16 * g) * 8 + e] = (uint16_t)bf16_bits(v);
    };
    // K-step, lane group and element of hidden feature k (the inverse of khid)
    auto ks = [](int k) { return k >> 5; };
    auto kg = [](int k) { return (k >> 2) & 3; };
    auto ke = [](int k) { return ((k >> 4) & 1) * 4 + (k & 3); };
    const int p = (int)i;
    if (p < oB1) {
        const int o = p / kIn, k = p % kIn, n = k / 6, c = k % 6, g = n >> 3, m = n & 7, t = o >> 4;
        if (c == 1) put(kFV + t, o & 15, g, m, w);
        else if (c == 2) put(kFG + t * 5 + 4, o & 15, g, m, w);
        else put(kFG + t * 5 + (m >> 1), o & 15, g, (m & 1) * 4 + (c == 0 ? 0 : c - 2), w);
        return;
    }
    for (int layer = 1; layer < 4; ++layer) {
        const int q = p - kWOff[layer];
        if (q < 0 || q >= kHid * kHid) continue;
        const int o = q / kHid, k = q % kHid;
        put(kF2 + (layer - 1) * 8 + (o >> 4) * 2 + ks(k), o & 15, kg(k), ke(k), w);
        put(kG2 + (layer - 1) * 8 + (k >> 4) * 2 + ks(o), k & 15, kg(o), ke(o), w);
    }
    if (p >= oW5 && p < oB5) {
        const int o = (p - oW5) / kHid, k = (p - oW5) % kHid;
        put(kG5 + (k >> 4), k & 15, 0, o, w);
        const float hi = bf16_val(bf16_bits(w));
        put(kF5 + ks(k), o, kg(k), ke(k), hi);
        put(kF5 + ks(k), o + 2, kg(k), ke(k), w - hi);
    }
}

// One Adam step; each thread re-packs the parameter it updates.
__global__ void k_dn_adam(float* params, float* m, float* v, const float* grad, float lr_t, float b1,
                          float b2, float eps, uint16_t* frags) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (uint32_t)kParams) return;
    float gr = grad[i];
    float mi = b1 * m[i] + (1.0f - b1) * gr;
    float vi = b2 * v[i] + (1.0f - b2) * gr * gr;
    m[i] = mi;
    v[i] = vi;
    const float w = params[i] - lr_t * mi / (sqrtf(vi) + eps);
    params[i] = w;
    dn_pack_param(i, w, frags);
}

// BF16 fragments of every weight matrix from the FP32 master copy (positions
// that hold no parameter were zeroed when the fragments were allocated).
__global__ void k_dn_pack(const float* P, uint16_t* frags) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (uint32_t)kParams) dn_pack_param(i, P[i], frags);
}

// Input features of explicit samples, [count][150] BF16 bits (inspection).
__global__ __launch_bounds__(kBlock) void k_dn_features(DnFrameDev F, const uint32_t* samples,
                                                        uint32_t count, uint16_t* out) {
    const uint32_t id = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t i = id / 19, grp = id % 19;   // 19 groups of 8 cover 150 features
    if (i >= count) return;
    uint32_t sm = samples[i], p = sm & 0xFFFFFFu, l = sm >> 24;
    const uint32_t lights = F.num_lights ? F.num_lights : 1u;
    bool valid = p < F.width * F.height && l < lights;
    if (!valid) { p = 0; l = 0; }
    const float dcv = F.pix[p].x;
    valid = valid && dcv >= 0.0f;
    const float dc = valid ? dcv : 0.0f;
    uint4 fb = dn_features(F, valid, p % F.width, p / F.width, l, dc, 8 * (int)grp);
    const uint32_t ws[4] = {fb.x, fb.y, fb.z, fb.w};
    for (int e = 0; e < 8; ++e) {
        int f = 8 * (int)grp + e;
        if (f < kIn) out[(size_t)i * kIn + f] = (uint16_t)(ws[e >> 1] >> (16 * (e & 1)));
    }
}

inline uint32_t cdiv(uint64_t a, uint32_t b) { return (uint32_t)((a + b - 1) / b); }

}  // namespace
}  // namespace luz

using namespace luz;

struct luzrt_denoiser {
    uint32_t capacity = 0;     // training samples per gradient
    uint32_t rows = 0;         // samples accumulated since the last gradient
    uint32_t step = 0;         // Adam steps taken
    float* params = nullptr;   // FP32 master
    float* grad = nullptr;
    float* adam_m = nullptr;
    float* adam_v = nullptr;
    float* partial = nullptr;
    float* loss = nullptr;     // device loss sum
    uint16_t* frags = nullptr;
    uint4* X = nullptr;
    uint4* H = nullptr;
    uint4* Z = nullptr;
    uint32_t* Y = nullptr;
    DevBuf pix, ao_frac;    // prepass planes of the current frame
};

namespace {

void dn_free(luzrt_denoiser* d) {
    for (void* p : {(void*)d->params, (void*)d->grad, (void*)d->adam_m, (void*)d->adam_v,
                    (void*)d->partial, (void*)d->loss, (void*)d->frags, (void*)d->X, (void*)d->H,
                    (void*)d->Z, (void*)d->Y, d->pix.ptr, d->ao_frac.ptr})
        if (p) (void)hipFree(p);
    delete d;
}

luzrt_status frame_dev(luzrt_ctx* ctx, const luzrt_dn_frame* f, DnFrameDev& F) {
    if (!f || !f->position || !f->normal || !f->ao_counts || (f->num_lights && !f->shadow_counts))
        return fail(ctx, LUZRT_E_INVALID_ARG, "denoiser frame: null plane");
    if (f->width == 0 || f->height == 0 || (uint64_t)f->width * f->height > 0xFFFFFFull)
        return fail(ctx, LUZRT_E_LIMIT, "denoiser frame: %ux%u outside 1..2^24 pixels", f->width, f->height);
    if (f->num_lights > LUZRT_MAX_LIGHTS || f->ao_samples == 0 || (f->num_lights && f->shadow_samples == 0))
        return fail(ctx, LUZRT_E_INVALID_ARG, "denoiser frame: bad light or sample counts");
    std::memset(&F, 0, sizeof(F));
    F.width = f->width;
    F.height = f->height;
    F.num_lights = f->num_lights;
    F.position = f->position;
    F.normal = f->normal;
    F.shadow = f->shadow_counts;
    F.ao = f->ao_counts;
    for (int k = 0; k < 3; ++k) F.cam[k] = f->cam_pos[k];
    F.shadow_n = (float)(f->shadow_samples ? f->shadow_samples : 1u);
    F.ao_n = (float)f->ao_samples;
    return LUZRT_OK;
}

// Runs the per-pixel prepass of a frame into the given planes.
luzrt_status prep_frame(luzrt_ctx* ctx, DnFrameDev& F, DevBuf& pix, DevBuf& ao_frac) {
    const uint32_t npix = F.width * F.height;
    luzrt_status s;
    if ((s = ensure(ctx, pix, (size_t)npix * 16)) != LUZRT_OK) return s;
    if ((s = ensure(ctx, ao_frac, (size_t)npix * 4)) != LUZRT_OK) return s;
    k_dn_prep<<<cdiv(npix, 256), 256, 0, ctx->stream>>>(F, (float4*)pix.ptr, (float*)ao_frac.ptr);
    LUZ_HIP(ctx, hipGetLastError());
    F.pix = (const float4*)pix.ptr;
    F.ao_frac = (const float*)ao_frac.ptr;
    return LUZRT_OK;
}

luzrt_status repack(luzrt_ctx* ctx, luzrt_denoiser* d) {
    k_dn_pack<<<cdiv(kParams, 256), 256, 0, ctx->stream>>>(d->params, d->frags);
    LUZ_HIP(ctx, hipGetLastError());
    return LUZRT_OK;
}

}  // namespace

extern "C" {

luzrt_status luzrt_denoiser_create(luzrt_ctx* ctx, uint32_t batch_capacity, uint64_t seed,
                                   luzrt_denoiser** out) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!out) return fail(ctx, LUZRT_E_INVALID_ARG, "luzrt_denoiser_create: null argument");
    *out = nullptr;
    if (batch_capacity % 64 != 0 || batch_capacity > (1u << 22))
        return fail(ctx, LUZRT_E_LIMIT, "batch capacity %u: a multiple of 64 up to 2^22", batch_capacity);
    LUZ_HIP(ctx, hipSetDevice(ctx->device));
    auto* d = new luzrt_denoiser();
    d->capacity = batch_capacity;
    const uint32_t cap = batch_capacity ? batch_capacity : 64;
    const uint32_t chunks = cdiv(cap, kChunkRows);
    const size_t pb = (size_t)kParams * 4;
    struct A { void** p; size_t bytes; } allocs[] = {
        {(void**)&d->params, pb}, {(void**)&d->grad, pb}, {(void**)&d->adam_m, pb},
        {(void**)&d->adam_v, pb}, {(void**)&d->partial, pb * chunks}, {(void**)&d->loss, 256},
        {(void**)&d->frags, (size_t)kFragAll * 1024}, {(void**)&d->X, (size_t)kX * cap * 2},
        {(void**)&d->H, (size_t)4 * kHid * cap * 2}, {(void**)&d->Z, (size_t)4 * kHid * cap * 2},
        {(void**)&d->Y, (size_t)cap * 4}};
    for (auto& a : allocs) {
        hipError_t e = hipMalloc(a.p, a.bytes);
        if (e != hipSuccess) { dn_free(d); return hip_fail(ctx, e, "hipMalloc(denoiser)"); }
    }
    // fragment positions that hold no parameter stay zero
    LUZ_HIP(ctx, hipMemset(d->frags, 0, (size_t)kFragAll * 1024));
    LUZ_HIP(ctx, hipMemset(d->adam_m, 0, pb));
    LUZ_HIP(ctx, hipMemset(d->adam_v, 0, pb));
    LUZ_HIP(ctx, hipMemset(d->grad, 0, pb));
    LUZ_HIP(ctx, hipMemset(d->loss, 0, 256));
    // He-uniform initial weights (SplitMix64), zero biases
    std::vector<float> h(kParams, 0.0f);
    uint64_t st = seed;
    auto next = [&st]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return (double)((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0);
    };
    const int fan_in[5] = {kIn, kHid, kHid, kHid, kHid}, rows_out[5] = {kHid, kHid, kHid, kHid, kOut};
    for (int L = 0; L < 5; ++L) {
        double lim = std::sqrt(6.0 / fan_in[L]);
        for (int i = 0; i < rows_out[L] * fan_in[L]; ++i) h[kWOff[L] + i] = (float)((2.0 * next() - 1.0) * lim);
    }
    LUZ_HIP(ctx, hipMemcpy(d->params, h.data(), pb, hipMemcpyHostToDevice));
    luzrt_status s = repack(ctx, d);
    if (s != LUZRT_OK) { dn_free(d); return s; }
    *out = d;
    return LUZRT_OK;
}

luzrt_status luzrt_denoiser_destroy(luzrt_ctx* ctx, luzrt_denoiser* d) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!d) return LUZRT_OK;
    LUZ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    dn_free(d);
    return LUZRT_OK;
}

luzrt_status luzrt_denoiser_get_params(luzrt_ctx* ctx, luzrt_denoiser* d, float* host, uint32_t count) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!d || !host || count != (uint32_t)kParams)
        return fail(ctx, LUZRT_E_INVALID_ARG, "denoiser parameters: need %d floats", kParams);
    LUZ_HIP(ctx, hipMemcpyAsync(host, d->params, (size_t)kParams * 4, hipMemcpyDeviceToHost, ctx->stream));
    LUZ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return LUZRT_OK;
}

luzrt_status luzrt_denoiser_set_params(luzrt_ctx* ctx, luzrt_denoiser* d, const float* host, uint32_t count) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!d || !host || count != (uint32_t)kParams)
        return fail(ctx, LUZRT_E_INVALID_ARG, "denoiser parameters: need %d floats", kParams);
    for (uint32_t i = 0; i < count; ++i)
        if (!std::isfinite(host[i])) return fail(ctx, LUZRT_E_INVALID_ARG, "parameter %u is not finite", i);
    LUZ_HIP(ctx, hipMemcpyAsync(d->params, host, (size_t)kParams * 4, hipMemcpyHostToDevice, ctx->stream));
    LUZ_HIP(ctx, hipMemsetAsync(d->adam_m, 0, (size_t)kParams * 4, ctx->stream));
    LUZ_HIP(ctx, hipMemsetAsync(d->adam_v, 0, (size_t)kParams * 4, ctx->stream));
    d->step = 0;
    luzrt_status s = repack(ctx, d);
    if (s != LUZRT_OK) return s;
    LUZ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return LUZRT_OK;
}

luzrt_status luzrt_denoise(luzrt_ctx* ctx, luzrt_denoiser* d, const luzrt_dn_frame* f, float* ao_out,
                           float* vis_out) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!d || !ao_out || (f && f->num_lights && !vis_out))
        return fail(ctx, LUZRT_E_INVALID_ARG, "luzrt_denoise: null argument");
    InferArgs A{};
    luzrt_status s = frame_dev(ctx, f, A.F);
    if (s != LUZRT_OK) return s;
    const uint32_t npix = f->width * f->height;
    stage_begin(ctx, kStageDenoise);
    if ((s = prep_frame(ctx, A.F, d->pix, d->ao_frac)) != LUZRT_OK) return s;
    A.frags = reinterpret_cast<const uint4*>(d->frags);
    A.params = d->params;
    A.lights = f->num_lights ? f->num_lights : 1u;
    A.ntiles = cdiv(npix, 16);
    A.ao_out = ao_out;
    A.vis_out = vis_out;
    // as many groups as are resident at once (48 KB of LDS and the registers
    // of 8 waves each), so that no group waits for another to finish
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_dn_infer, kInferBlock, 0) !=
            hipSuccess || per_cu < 1)
        per_cu = 1;
    uint32_t groups = cdiv(A.ntiles, kInferBlock / 64);
    const uint32_t maxg = (uint32_t)(ctx->num_cus > 0 ? ctx->num_cus : 1) * (uint32_t)per_cu;
    if (groups > maxg) groups = maxg;
    k_dn_infer<<<groups, kInferBlock, 0, ctx->stream>>>(A);
    stage_end(ctx, kStageDenoise);
    LUZ_HIP(ctx, hipGetLastError());
    return LUZRT_OK;
}

luzrt_status luzrt_denoiser_features(luzrt_ctx* ctx, const luzrt_dn_frame* f, const uint32_t* samples,
                                     uint32_t count, uint16_t* out) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!samples || !out) return fail(ctx, LUZRT_E_INVALID_ARG, "luzrt_denoiser_features: null argument");
    DnFrameDev F;
    luzrt_status s = frame_dev(ctx, f, F);
    if (s != LUZRT_OK) return s;
    if (count == 0) return LUZRT_OK;
    DevBuf pix, ao_frac;
    s = prep_frame(ctx, F, pix, ao_frac);
    if (s == LUZRT_OK) {
        k_dn_features<<<cdiv((uint64_t)count * 19, kBlock), kBlock, 0, ctx->stream>>>(F, samples, count, out);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) s = hip_fail(ctx, e, "k_dn_features");
    }
    // the planes are released once the kernel has read them
    (void)hipStreamSynchronize(ctx->stream);
    if (pix.ptr) (void)hipFree(pix.ptr);
    if (ao_frac.ptr) (void)hipFree(ao_frac.ptr);
    return s;
}

luzrt_status luzrt_denoiser_accumulate(luzrt_ctx* ctx, luzrt_denoiser* d, const luzrt_dn_frame* f,
                                       const float* target_ao, const float* target_vis,
                                       const uint32_t* samples, uint32_t count, float grad_scale) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!d || !target_ao || !samples || (f && f->num_lights && !target_vis))
        return fail(ctx, LUZRT_E_INVALID_ARG, "luzrt_denoiser_accumulate: null argument");
    if (count % 64 != 0 || d->rows + count > d->capacity)
        return fail(ctx, LUZRT_E_LIMIT, "%u samples (a multiple of 64) over the batch capacity %u (%u used)",
                    count, d->capacity, d->rows);
    DnArgs A{};
    luzrt_status s = frame_dev(ctx, f, A.F);
    if (s != LUZRT_OK) return s;
    if (count == 0) return LUZRT_OK;
    A.frags = reinterpret_cast<const uint4*>(d->frags);
    A.params = d->params;
    A.nsamples = count;
    A.lights = f->num_lights ? f->num_lights : 1u;
    A.samples = samples;
    A.target_ao = target_ao;
    A.target_vis = target_vis;
    A.row_base = d->rows;
    A.cap = d->capacity;
    A.X = d->X;
    A.H = d->H;
    A.Z = d->Z;
    A.Y = d->Y;
    A.grad_scale = grad_scale;
    A.loss_sum = d->loss;
    // one 16-sample tile per wave, up to the two groups per CU that their
    // fragments in LDS leave room for
    uint32_t groups = cdiv(count, 16 * (kBlock / 64));
    const uint32_t maxg = (uint32_t)(ctx->num_cus > 0 ? ctx->num_cus : 1) * 2;
    if (groups > maxg) groups = maxg;
    k_dn_forward<<<groups, kBlock, 0, ctx->stream>>>(A);
    LUZ_HIP(ctx, hipGetLastError());
    d->rows += count;
    return LUZRT_OK;
}

luzrt_status luzrt_denoiser_gradient(luzrt_ctx* ctx, luzrt_denoiser* d, float* host_grad, float* loss_sum) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!d) return fail(ctx, LUZRT_E_INVALID_ARG, "luzrt_denoiser_gradient: null denoiser");
    hipStream_t st = ctx->stream;
    if (d->rows > 0) {
        WgArgs W{(const uint2*)d->X, (const uint2*)d->H, (const uint2*)d->Z, (const uint4*)d->Y, d->capacity, d->rows,
                 d->partial};
        const uint32_t chunks = cdiv(d->rows, kChunkRows);
        k_dn_wgrad<<<dim3(chunks, kWgJobs), kBlock, 0, st>>>(W);
        k_dn_reduce<<<cdiv(kParams, kBlock / 4), kBlock, 0, st>>>(d->partial, chunks, d->grad);
        LUZ_HIP(ctx, hipGetLastError());
    } else {
        LUZ_HIP(ctx, hipMemsetAsync(d->grad, 0, (size_t)kParams * 4, st));
    }
    d->rows = 0;
    if (host_grad) LUZ_HIP(ctx, hipMemcpyAsync(host_grad, d->grad, (size_t)kParams * 4, hipMemcpyDeviceToHost, st));
    if (loss_sum) LUZ_HIP(ctx, hipMemcpyAsync(loss_sum, d->loss, 4, hipMemcpyDeviceToHost, st));
    LUZ_HIP(ctx, hipMemsetAsync(d->loss, 0, 4, st));
    if (host_grad || loss_sum) LUZ_HIP(ctx, hipStreamSynchronize(st));
    return LUZRT_OK;
}

luzrt_status luzrt_denoiser_adam(luzrt_ctx* ctx, luzrt_denoiser* d, float lr, float beta1, float beta2,
                                 float eps) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!d || !(lr > 0.0f) || !(beta1 >= 0.0f && beta1 < 1.0f) || !(beta2 >= 0.0f && beta2 < 1.0f) || !(eps > 0.0f))
        return fail(ctx, LUZRT_E_INVALID_ARG, "luzrt_denoiser_adam: bad arguments");
    d->step++;
    // bias-corrected step size
    double c1 = 1.0 - std::pow((double)beta1, (double)d->step);
    double c2 = 1.0 - std::pow((double)beta2, (double)d->step);
    float lr_t = (float)(lr * std::sqrt(c2) / c1);
    k_dn_adam<<<cdiv(kParams, 256), 256, 0, ctx->stream>>>(d->params, d->adam_m, d->adam_v, d->grad, lr_t,
                                                          beta1, beta2, eps, d->frags);
    LUZ_HIP(ctx, hipGetLastError());
    return LUZRT_OK;
}

}  // extern "C"
