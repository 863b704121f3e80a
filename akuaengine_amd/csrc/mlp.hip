// mlp.hip -- forward, backward and Adam kernels of the warm-start network on the gfx950 MFMA
// units (v_mfma_f32_16x16x16_bf16: BF16 operands, FP32 accumulation).
//
// Every product is C(16x16) += A(16xK) B(Kx16).  For the 16x16x16 instruction lane l = 16 g + r
// supplies A[r][4g..4g+3] and B[4g..4g+3][r] and receives C[4g+i][r], i = 0..3.  A wave owns 16
// samples at a time, in the orientation C[unit][sample] = W^T H^T: the result is the next layer's B
// operand, so the passes forward and back keep their activations in registers.  The weight-gradient
// products contract over samples: their operands go through LDS as rows [unit][sample].
#include "mlp.h"

#include <algorithm>
#include <type_traits>

#include "pbf_kernels.h"

namespace akua {

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// float -> bf16 bits, round to nearest even (inputs here are finite).
__device__ __forceinline__ uint16_t to_bf16(float x) {
    uint32_t u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// BF16 weights in the orientations the products read, plus the FP32 vectors.
struct alignas(16) WeightsLds {
    uint16_t w1t[kMlpHid * kMlpIn];   // [o][f]
    uint16_t w2t[kMlpHid * kMlpHid];  // [o][i]
    uint16_t w3t[16 * kMlpHid];       // [o (padded to 16)][j]
    float b1[kMlpHid], b2[kMlpHid], b3[16];
    float mean[kMlpIn], inv[kMlpIn], ymul[kMlpOut];
};
__device__ void load_weights(const float* __restrict__ P, WeightsLds& W) {
    for (int t = threadIdx.x; t < kMlpIn * kMlpHid; t += blockDim.x) {
        const int f = t / kMlpHid, o = t % kMlpHid;
        W.w1t[o * kMlpIn + f] = to_bf16(P[kOffW1 + t]);
    }
    for (int t = threadIdx.x; t < kMlpHid * kMlpHid; t += blockDim.x) {
        const int i = t / kMlpHid, o = t % kMlpHid;
        W.w2t[o * kMlpHid + i] = to_bf16(P[kOffW2 + t]);
    }
    for (int t = threadIdx.x; t < 16 * kMlpHid; t += blockDim.x) {
        const int j = t / 16, o = t % 16;
        W.w3t[o * kMlpHid + j] = o < kMlpOut ? to_bf16(P[kOffW3 + j * kMlpOut + o]) : (uint16_t)0;
    }
    for (int t = threadIdx.x; t < kMlpHid; t += blockDim.x) {
        W.b1[t] = P[kOffB1 + t];
        W.b2[t] = P[kOffB2 + t];
    }
    for (int t = threadIdx.x; t < 16; t += blockDim.x) {
        W.b3[t] = t < kMlpOut ? P[kOffB3 + t] : 0.0f;
        W.mean[t] = P[kOffMean + t];
        W.inv[t] = P[kOffInv + t];
        if (t < kMlpOut) W.ymul[t] = P[kOffYmul + t];
    }
}

constexpr int kInferBlock = 256;
constexpr int kInferWaves = kInferBlock / 64;

__device__ __forceinline__ bf16x4 pack_bf16(float a, float b, float c, float d) {
    typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
    const bf16x2v lo = {(__bf16)a, (__bf16)b};  // v_cvt_pk_bf16_f32: round to nearest even
    const bf16x2v hi = {(__bf16)c, (__bf16)d};
    const uint32_t u0 = __builtin_bit_cast(uint32_t, lo), u1 = __builtin_bit_cast(uint32_t, hi);
    bf16x4 r;
    r[0] = (short)(u0 & 0xFFFFu);
    r[1] = (short)(u0 >> 16);
    r[2] = (short)(u1 & 0xFFFFu);
    r[3] = (short)(u1 >> 16);
    return r;
}

// Inference in the transposed orientation C[unit][sample] = W^T H^T: lane l = 16 g + r owns
// sample r; the accumulator of output tile m0 holds units 16 m0 + 4 g + i of that sample, which
// is exactly the B operand of the next layer's k-step m0, so activations stay in registers.  The
// weight fragments (A operands) are loaded from LDS into registers once per wave.
struct InferRegs {
    bf16x4 w1[4], w2[4][4], w3[4];
};

__device__ __forceinline__ void load_infer_regs(const WeightsLds& W, InferRegs& R) {
    const int l = __lane_id();
    const int r = l & 15, g = l >> 4;
#pragma unroll
    for (int m0 = 0; m0 < 4; ++m0) {
        R.w1[m0] = *reinterpret_cast<const bf16x4*>(W.w1t + (16 * m0 + r) * kMlpIn + 4 * g);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
            R.w2[m0][kk] = *reinterpret_cast<const bf16x4*>(W.w2t + (16 * m0 + r) * kMlpHid + 16 * kk + 4 * g);
        R.w3[m0] = *reinterpret_cast<const bf16x4*>(W.w3t + r * kMlpHid + 16 * m0 + 4 * g);
    }
}

// Normalised outputs y[i] = output 4g + i of sample row0 + r (meaningful for g == 0).
__device__ __forceinline__ f32x4 infer_tile(const WeightsLds& W, const InferRegs& R,
                                            const float* __restrict__ feat, uint32_t row0,
                                            uint32_t n) {
    const int l = __lane_id();
    const int r = l & 15, g = l >> 4;
    const uint32_t row = row0 + (uint32_t)r;
    bf16x4 xb;
    if (row < n) {
        const float4 v = *reinterpret_cast<const float4*>(feat + (size_t)row * kMlpIn + 4 * g);
        xb = pack_bf16((v.x - W.mean[4 * g + 0]) * W.inv[4 * g + 0],
                       (v.y - W.mean[4 * g + 1]) * W.inv[4 * g + 1],
                       (v.z - W.mean[4 * g + 2]) * W.inv[4 * g + 2],
                       (v.w - W.mean[4 * g + 3]) * W.inv[4 * g + 3]);
    } else {
        xb = bf16x4{0, 0, 0, 0};
    }
    bf16x4 h1[4], h2[4];
#pragma unroll
    for (int m0 = 0; m0 < 4; ++m0) {
        f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
        c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(R.w1[m0], xb, c, 0, 0, 0);
        const float* b = W.b1 + 16 * m0 + 4 * g;
        h1[m0] = pack_bf16(fmaxf(c[0] + b[0], 0.0f), fmaxf(c[1] + b[1], 0.0f),
                           fmaxf(c[2] + b[2], 0.0f), fmaxf(c[3] + b[3], 0.0f));
    }
#pragma unroll
    for (int m0 = 0; m0 < 4; ++m0) {
        f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
            c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(R.w2[m0][kk], h1[kk], c, 0, 0, 0);
        const float* b = W.b2 + 16 * m0 + 4 * g;
        h2[m0] = pack_bf16(fmaxf(c[0] + b[0], 0.0f), fmaxf(c[1] + b[1], 0.0f),
                           fmaxf(c[2] + b[2], 0.0f), fmaxf(c[3] + b[3], 0.0f));
    }
    f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
        c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(R.w3[kk], h2[kk], c, 0, 0, 0);
    const float* b = W.b3 + 4 * g;
    return f32x4{c[0] + b[0], c[1] + b[1], c[2] + b[2], c[3] + b[3]};
}

__global__ __launch_bounds__(kInferBlock) void k_mlp_eval(const float* __restrict__ P,
                                                          const float* __restrict__ feat,
                                                          uint32_t n, float* __restrict__ y) {
    __shared__ WeightsLds W;
    load_weights(P, W);
    __syncthreads();
    InferRegs R;
    load_infer_regs(W, R);
    const int l = __lane_id();
    const uint32_t tiles = (n + 15) / 16;
    const uint32_t wave = blockIdx.x * kInferWaves + threadIdx.x / 64;
    const uint32_t nwaves = gridDim.x * kInferWaves;
    for (uint32_t t = wave; t < tiles; t += nwaves) {
        const f32x4 o = infer_tile(W, R, feat, t * 16, n);
        const uint32_t row = t * 16 + (uint32_t)l;
        if (l < 16 && row < n)
            *reinterpret_cast<float4*>(y + (size_t)row * 4) =
                make_float4(o[0] * W.ymul[0], o[1] * W.ymul[1], o[2] * W.ymul[2], o[3] * W.ymul[3]);
    }
}

// The warm start of a learned step: x*_w = x*_pred + h * D for every particle slot of a scene,
// with D and the auxiliary lambda the network's outputs for the slot's features.
__global__ __launch_bounds__(kInferBlock) void k_mlp_apply(DeviceState d, const float* __restrict__ P,
                                                           float h, const float4* __restrict__ XsPred,
                                                           float4* __restrict__ XsWarm,
                                                           float* __restrict__ lamHat) {
    __shared__ WeightsLds W;
    load_weights(P, W);
    __syncthreads();
    InferRegs R;
    load_infer_regs(W, R);
    const int l = __lane_id();
    const uint32_t n = d.nslots;
    const uint32_t tiles = (n + 15) / 16;
    const uint32_t wave = blockIdx.x * kInferWaves + threadIdx.x / 64;
    const uint32_t nwaves = gridDim.x * kInferWaves;
    for (uint32_t t = wave; t < tiles; t += nwaves) {
        const f32x4 o = infer_tile(W, R, d.feat, t * 16, n);
        const uint32_t p = t * 16 + (uint32_t)l;
        if (l < 16 && p < n && p < d.scenes[d.chunkScene[p >> 8]].end) {
            const float4 x = XsPred[p];
            // the network was trained on targets within +-kMlpTargetClip normalised units: the
            // warm start does not extrapolate beyond them
            const float c = kMlpTargetClip;
            const float dx = fminf(fmaxf(o[0], -c), c) * W.ymul[0];
            const float dy = fminf(fmaxf(o[1], -c), c) * W.ymul[1];
            const float dz = fminf(fmaxf(o[2], -c), c) * W.ymul[2];
            XsWarm[p] = make_float4(x.x + h * dx, x.y + h * dy, x.z + h * dz, x.w);
            lamHat[p] = o[3] * W.ymul[3];
        }
    }
}

// Rows [unit][sample] of the gradient kernel and its weights' rows: 64 columns, padded so that a wave's
// 2-byte column stores and 8-byte row reads spread over the banks.
constexpr int kGradRow = kMlpGradSamples + 8;
constexpr int kGradW1Row = kMlpIn + 4;

struct alignas(16) GradLds {
    uint16_t w1t[kMlpHid * kGradW1Row];  // [o][f]
    uint16_t w2t[kMlpHid * kGradRow];    // [o][i]
    uint16_t w2[kMlpHid * kGradRow];     // [i][o]
    uint16_t w3t[kMlpOut * kGradRow];    // [o][j]
    uint16_t x[kMlpIn * kGradRow], h1[kMlpHid * kGradRow], h2[kMlpHid * kGradRow];
    uint16_t g3[kMlpOut * kGradRow], g2[kMlpHid * kGradRow], g1[kMlpHid * kGradRow];
};
static_assert(sizeof(GradLds) <= 65536, "one workgroup's LDS");

typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ bf16x4 lds4(const uint16_t* p) { return *reinterpret_cast<const bf16x4*>(p); }

__device__ __forceinline__ f32x4 mma(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Four values of one sample (column) into rows row0..row0+3.
__device__ __forceinline__ void put_column(uint16_t* rows, int row0, int column, bf16x4 v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) rows[(row0 + i) * kGradRow + column] = (uint16_t)v[i];
}

// Sum over the 16 lanes of equal l / 16, in every one of them.
__device__ __forceinline__ float sum16(float x) {
    const auto add = [&](auto ctrl) {
        x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xF, 0xF, false));
    };
    add(std::integral_constant<int, 0xB1>{});   // quad_perm [1, 0, 3, 2]
    add(std::integral_constant<int, 0x4E>{});   // quad_perm [2, 3, 0, 1]
    add(std::integral_constant<int, 0x141>{});  // row_half_mirror
    add(std::integral_constant<int, 0x140>{});  // row_mirror
    return x;
}

// Gradient partials, one row per workgroup.  64 samples at a time: each wave takes 16 forward and back
// in registers and leaves activations and gradients in LDS as rows [unit][sample]; then the waves share
// the 24 output tiles of the weight gradients, six each, contracted over all 64 samples.  So one row
// holds 64 samples' gradient without any sum across waves but the biases', and a workgroup per 64
// samples fills 128 CUs at 8,192 samples.  Bound by latency: the weights' and samples' loads, eleven
// dependent product chains and two barriers, once per workgroup.
// Measured at 8,192 samples: 29.3 us with a wave per 32 samples and its activations in LDS both ways
// (256 rows), 10.3 us here (128 rows).
__global__ __launch_bounds__(64 * kMlpGradWaves) void k_mlp_grad(const float* __restrict__ P,
                                                                 const float* __restrict__ feat,
                                                                 const float* __restrict__ targ,
                                                                 uint32_t n, MlpLossWeights lw,
                                                                 float* __restrict__ part) {
    __shared__ GradLds S;
    __shared__ float sums[kMlpGradWaves][2 * kMlpHid + kMlpOut + 1];  // bias gradients and loss by wave
    const int l = __lane_id();
    const int r = l & 15, g = l >> 4;
    const int wave = threadIdx.x >> 6;
    const int col = 16 * wave + r;  // this lane's sample among the 64
    constexpr int kThreads = 64 * kMlpGradWaves;
    // weights, four of a row (transposed: of a column) at a time
    for (int t = threadIdx.x; t < kMlpHid * kMlpIn / 4; t += kThreads) {
        const int o = t % kMlpHid, f = 4 * (t / kMlpHid);
        const float* w = P + kOffW1 + f * kMlpHid + o;
        *reinterpret_cast<bf16x4*>(&S.w1t[o * kGradW1Row + f]) = pack_bf16(w[0], w[kMlpHid], w[2 * kMlpHid], w[3 * kMlpHid]);
    }
    for (int t = threadIdx.x; t < kMlpHid * kMlpHid / 4; t += kThreads) {
        const int o = t % kMlpHid, i = 4 * (t / kMlpHid);
        const float* w = P + kOffW2 + i * kMlpHid + o;
        *reinterpret_cast<bf16x4*>(&S.w2t[o * kGradRow + i]) = pack_bf16(w[0], w[kMlpHid], w[2 * kMlpHid], w[3 * kMlpHid]);
        const float* v = P + kOffW2 + 4 * t;
        *reinterpret_cast<bf16x4*>(&S.w2[(t / 16) * kGradRow + 4 * (t % 16)]) = pack_bf16(v[0], v[1], v[2], v[3]);
    }
    for (int t = threadIdx.x; t < kMlpOut * kMlpHid / 4; t += kThreads) {
        const int o = t % kMlpOut, j = 4 * (t / kMlpOut);
        const float* w = P + kOffW3 + j * kMlpOut + o;
        *reinterpret_cast<bf16x4*>(&S.w3t[o * kGradRow + j]) = pack_bf16(w[0], w[kMlpOut], w[2 * kMlpOut], w[3 * kMlpOut]);
    }
    // per lane: its units' biases (16 m0 + 4 g + i), its features' normalisation, the outputs' scales,
    // and, where g is 0 (the outputs' lanes), rows of W3
    float b1[4][4], b2[4][4], b3[4], ymul[4], mean[4], inv[4];
    bf16x4 w3b[4];
    const bf16x4 zero4 = {0, 0, 0, 0};
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        mean[i] = P[kOffMean + 4 * g + i];
        inv[i] = P[kOffInv + 4 * g + i];
        b3[i] = P[kOffB3 + i];
        ymul[i] = P[kOffYmul + i];
#pragma unroll
        for (int m0 = 0; m0 < 4; ++m0) {
            b1[m0][i] = P[kOffB1 + 16 * m0 + 4 * g + i];
            b2[m0][i] = P[kOffB2 + 16 * m0 + 4 * g + i];
        }
    }
#pragma unroll
    for (int m0 = 0; m0 < 4; ++m0) {
        const float* w = P + kOffW3 + (16 * m0 + r) * kMlpOut;
        w3b[m0] = g == 0 ? pack_bf16(w[0], w[1], w[2], w[3]) : zero4;
    }
    const float invN = 1.0f / (float)n;
    f32x4 acc1 = zero, acc2[4] = {zero, zero, zero, zero}, acc3 = zero;
    float db1[4][4] = {}, db2[4][4] = {}, db3[4] = {}, loss = 0.0f;

    const uint32_t rounds = (n + kMlpGradSamples - 1u) / kMlpGradSamples;
    for (uint32_t q = blockIdx.x; q < rounds; q += gridDim.x) {
        const uint32_t row = q * kMlpGradSamples + (uint32_t)col;
        float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f), tg = f;
        if (row < n) {
            f = *reinterpret_cast<const float4*>(feat + (size_t)row * kMlpIn + 4 * g);
            if (g == 0) {  // the caller's array, of which only a float's alignment is asked
                const f32x4a4 v = *reinterpret_cast<const f32x4a4*>(targ + (size_t)row * kMlpOut);
                tg = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
        __syncthreads();  // the weights are in LDS; the round before has read its rows
        const bf16x4 x = row < n ? pack_bf16((f.x - mean[0]) * inv[0], (f.y - mean[1]) * inv[1],
                                             (f.z - mean[2]) * inv[2], (f.w - mean[3]) * inv[3])
                                 : zero4;
        put_column(S.x, 4 * g, col, x);
        // forward; bit 4 m0 + i of on1 and on2: the unit is active
        bf16x4 h1[4], h2[4];
        uint32_t on1 = 0u, on2 = 0u;
#pragma unroll
        for (int m0 = 0; m0 < 4; ++m0) {
            const f32x4 c = mma(lds4(&S.w1t[(16 * m0 + r) * kGradW1Row + 4 * g]), x, zero);
            float z[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                z[i] = c[i] + b1[m0][i];
                on1 |= (z[i] > 0.0f ? 1u : 0u) << (4 * m0 + i);
            }
            h1[m0] = pack_bf16(fmaxf(z[0], 0.0f), fmaxf(z[1], 0.0f), fmaxf(z[2], 0.0f), fmaxf(z[3], 0.0f));
            put_column(S.h1, 16 * m0 + 4 * g, col, h1[m0]);
        }
#pragma unroll
        for (int m0 = 0; m0 < 4; ++m0) {
            f32x4 c = zero;
#pragma unroll
            for (int k = 0; k < 4; ++k) c = mma(lds4(&S.w2t[(16 * m0 + r) * kGradRow + 16 * k + 4 * g]), h1[k], c);
            float z[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                z[i] = c[i] + b2[m0][i];
                on2 |= (z[i] > 0.0f ? 1u : 0u) << (4 * m0 + i);
            }
            h2[m0] = pack_bf16(fmaxf(z[0], 0.0f), fmaxf(z[1], 0.0f), fmaxf(z[2], 0.0f), fmaxf(z[3], 0.0f));
            put_column(S.h2, 16 * m0 + 4 * g, col, h2[m0]);
        }
        f32x4 y = zero;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            y = mma(r < kMlpOut ? lds4(&S.w3t[(r & 3) * kGradRow + 16 * k + 4 * g]) : zero4, h2[k], y);
        // output gradient of the mean weighted squared error, in normalised units
        float G[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (g == 0 && row < n) {
            const float t[4] = {tg.x, tg.y, tg.z, tg.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float tn = fminf(fmaxf(t[i] / ymul[i], -kMlpTargetClip), kMlpTargetClip);
                const float diff = (y[i] + b3[i]) - tn;
                loss += lw.w[i] * diff * diff;
                G[i] = 2.0f * lw.w[i] * diff * invN;
                db3[i] += G[i];
            }
        }
        const bf16x4 g3 = pack_bf16(G[0], G[1], G[2], G[3]);
        if (g == 0) put_column(S.g3, 0, col, g3);
        // dH2 = W3 G3, masked by layer 2's activity; dH1 = W2 G2, masked by layer 1's
        bf16x4 g2[4];
#pragma unroll
        for (int m0 = 0; m0 < 4; ++m0) {
            const f32x4 c = mma(w3b[m0], g3, zero);
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[i] = (on2 >> (4 * m0 + i)) & 1u ? c[i] : 0.0f;
                db2[m0][i] += e[i];
            }
            g2[m0] = pack_bf16(e[0], e[1], e[2], e[3]);
            put_column(S.g2, 16 * m0 + 4 * g, col, g2[m0]);
        }
#pragma unroll
        for (int m0 = 0; m0 < 4; ++m0) {
            f32x4 c = zero;
#pragma unroll
            for (int k = 0; k < 4; ++k) c = mma(lds4(&S.w2[(16 * m0 + r) * kGradRow + 16 * k + 4 * g]), g2[k], c);
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[i] = (on1 >> (4 * m0 + i)) & 1u ? c[i] : 0.0f;
                db1[m0][i] += e[i];
            }
            put_column(S.g1, 16 * m0 + 4 * g, col, pack_bf16(e[0], e[1], e[2], e[3]));
        }
        __syncthreads();
        // weight gradients over the 64 samples: wave w the tiles (w, 0..3) of W2, w of W1 and of W3
#pragma unroll
        for (int k = 0; k < kMlpGradSamples / 16; ++k) {
            const int at = 16 * k + 4 * g;
            const bf16x4 a2 = lds4(&S.h1[(16 * wave + r) * kGradRow + at]);
#pragma unroll
            for (int n0 = 0; n0 < 4; ++n0) acc2[n0] = mma(a2, lds4(&S.g2[(16 * n0 + r) * kGradRow + at]), acc2[n0]);
            acc1 = mma(lds4(&S.x[r * kGradRow + at]), lds4(&S.g1[(16 * wave + r) * kGradRow + at]), acc1);
            acc3 = mma(lds4(&S.h2[(16 * wave + r) * kGradRow + at]),
                       r < kMlpOut ? lds4(&S.g3[(r & 3) * kGradRow + at]) : zero4, acc3);
        }
    }

    float* out = part + (size_t)blockIdx.x * kMlpPartRow;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = 4 * g + i;
        out[kOffW1 + m * kMlpHid + 16 * wave + r] = acc1[i];
#pragma unroll
        for (int n0 = 0; n0 < 4; ++n0) out[kOffW2 + (16 * wave + m) * kMlpHid + 16 * n0 + r] = acc2[n0][i];
        if (r < kMlpOut) out[kOffW3 + (16 * wave + m) * kMlpOut + r] = acc3[i];
    }
    // biases and loss: over the wave's 16 samples, then over the waves
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int m0 = 0; m0 < 4; ++m0) {
            const float a = sum16(db1[m0][i]), b = sum16(db2[m0][i]);
            if (r == 0) {
                sums[wave][16 * m0 + 4 * g + i] = a;
                sums[wave][kMlpHid + 16 * m0 + 4 * g + i] = b;
            }
        }
        const float c = sum16(db3[i]);
        if (l == 0) sums[wave][2 * kMlpHid + i] = c;
    }
    loss = sum16(loss);
    if (l == 0) sums[wave][2 * kMlpHid + kMlpOut] = loss * invN;
    __syncthreads();
    const int t = threadIdx.x;
    if (t <= 2 * kMlpHid + kMlpOut) {
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < kMlpGradWaves; ++w) s += sums[w][t];
        out[t < kMlpHid                    ? kOffB1 + t
            : t < 2 * kMlpHid              ? kOffB2 + t - kMlpHid
            : t < 2 * kMlpHid + kMlpOut    ? kOffB3 + t - 2 * kMlpHid
                                           : kMlpTrainable] = s;
    }
}

// The sum of column p over the partial rows, in a fixed order: kSlices threads take every kSlices-th
// row, eight loads in flight, and the first adds theirs (valid in slice 0).  One thread per column
// walked 256 rows with one load after another: 9.4 us; 4.0 us with 128 rows in 8 slices.
constexpr int kSumColumns = 32, kSumSlices = 8;

__device__ __forceinline__ float column_sum(const float* __restrict__ part, int rows, int p, int slice, float* lds) {
    float s = 0.0f;
    if (p <= kMlpTrainable) {
        int w = slice;
        for (; w + 7 * kSumSlices < rows; w += 8 * kSumSlices) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = part[(size_t)(w + u * kSumSlices) * kMlpPartRow + p];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
        }
        for (; w < rows; w += kSumSlices) s += part[(size_t)w * kMlpPartRow + p];
    }
    lds[threadIdx.x] = s;
    __syncthreads();
    s = 0.0f;
    if (slice == 0)
#pragma unroll
        for (int u = 0; u < kSumSlices; ++u) s += lds[u * kSumColumns + threadIdx.x];
    return s;
}

__global__ __launch_bounds__(kSumColumns * kSumSlices) void k_mlp_reduce(const float* __restrict__ part, int rows,
                                                                         float* __restrict__ grad,
                                                                         float* __restrict__ loss) {
    __shared__ float lds[kSumColumns * kSumSlices];
    const int slice = threadIdx.x / kSumColumns, p = blockIdx.x * kSumColumns + threadIdx.x % kSumColumns;
    const float s = column_sum(part, rows, p, slice, lds);
    if (slice != 0 || p > kMlpTrainable) return;
    if (p < kMlpTrainable) grad[p] = s;
    else *loss = s;
}

__global__ __launch_bounds__(kSumColumns * kSumSlices) void k_mlp_adam(
    const float* __restrict__ part, int rows, float* __restrict__ P, float* __restrict__ M, float* __restrict__ V,
    float lr, float b1, float b2, float eps, float c1, float c2, float* __restrict__ loss) {
    __shared__ float lds[kSumColumns * kSumSlices];
    const int slice = threadIdx.x / kSumColumns, p = blockIdx.x * kSumColumns + threadIdx.x % kSumColumns;
    float p0 = 0.0f, m0 = 0.0f, v0 = 0.0f;
    if (slice == 0 && p < kMlpTrainable) {
        p0 = P[p];
        m0 = M[p];
        v0 = V[p];
    }
    const float s = column_sum(part, rows, p, slice, lds);
    if (slice != 0 || p > kMlpTrainable) return;
    if (p == kMlpTrainable) {
        *loss = s;
        return;
    }
    const float m = b1 * m0 + (1.0f - b1) * s;
    const float v = b2 * v0 + (1.0f - b2) * (s * s);
    M[p] = m;
    V[p] = v;
    P[p] = p0 - lr * (m * c1) / (sqrtf(v * c2) + eps);
}

}  // namespace

// Workgroups of an inference launch: the waves loop over the 16-sample tiles, and each workgroup
// first stages the weights in LDS, so the grid is one resident set and no more: the kernels'
// 128 VGPRs leave room for 4 waves per SIMD, i.e. 4 workgroups of 4 waves per CU (1,024 on 256
// CUs measured 59 us per 1M-sample launch against 69 us with 2,048).
static uint32_t infer_blocks(uint32_t tiles) {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
    const uint32_t resident = 4u * (uint32_t)cus;
    return std::max<uint32_t>(1u, std::min<uint32_t>((tiles + kInferWaves - 1) / kInferWaves, resident));
}

void launch_mlp_eval(hipStream_t st, const float* params, const float* feat, uint32_t n, float* y) {
    if (!n) return;
    const uint32_t tiles = (n + 15) / 16;
    const uint32_t blocks = infer_blocks(tiles);
    k_mlp_eval<<<blocks, kInferBlock, 0, st>>>(params, feat, n, y);
}

void launch_mlp_apply(hipStream_t st, const DeviceState& d, const float* params, float h,
                      const float4* XsPred, float4* XsWarm, float* lamHat) {
    if (!d.nslots) return;
    const uint32_t tiles = (d.nslots + 15) / 16;
    const uint32_t blocks = infer_blocks(tiles);
    k_mlp_apply<<<blocks, kInferBlock, 0, st>>>(d, params, h, XsPred, XsWarm, lamHat);
}

int launch_mlp_grad(hipStream_t st, const float* params, const float* feat, const float* targ,
                    uint32_t n, MlpLossWeights lw, float* part) {
    const int rows = (int)std::min<uint32_t>((n - 1u) / kMlpGradSamples + 1u, (uint32_t)kMlpPartRows);
    k_mlp_grad<<<rows, 64 * kMlpGradWaves, 0, st>>>(params, feat, targ, n, lw, part);
    return rows;
}

static constexpr int kSumBlocks = (kMlpPartRow + kSumColumns - 1) / kSumColumns;

void launch_mlp_reduce(hipStream_t st, const float* part, int rows, float* grad, float* loss) {
    k_mlp_reduce<<<kSumBlocks, kSumColumns * kSumSlices, 0, st>>>(part, rows, grad, loss);
}

void launch_mlp_adam(hipStream_t st, const float* part, int rows, float* params, float* m, float* v, float lr,
                     float beta1, float beta2, float eps, float c1, float c2, float* loss) {
    k_mlp_adam<<<kSumBlocks, kSumColumns * kSumSlices, 0, st>>>(part, rows, params, m, v, lr, beta1, beta2, eps, c1,
                                                                c2, loss);
}

}  // namespace akua
