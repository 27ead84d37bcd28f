// Learned subgrid-viscosity closure: a per-node MLP
//     features (12) -> 32 -> 32 -> 1,  SiLU hidden layers, softplus output
//     mu_sgs = scale * softplus(z3)
// evaluated with bf16 MFMA (FP32 accumulation) by whole wavefronts: lane L of
// a wave owns node L, the 64 nodes of the wave are the columns of the layer
// GEMMs (v_mfma_f32_16x16x16_bf16: four tiles of 16 nodes).  The layers are
// formed transposed, Z^T = W^T X^T: a product's accumulators then hold, lane by
// lane, what the next product takes as its right operand, and the activations
// pass from layer to layer in registers.
//
// Features of an element node (all from the diffusion kernel's pass 1):
//   G(i,j) = du_i/dx_j (9, row-major), rho, |u|, h = 2 det(J)^(1/3)
// standardised with a mean and inverse deviation stored with the weights.
//
// Parameter block (FP32, kMlpParams floats):
//   W1[12][32] b1[32] W2[32][32] b2[32] w3[32] b3 | mean[12] istd[12] scale
// the first kMlpTrain are trained; W[in][out] row-major.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace msod {

constexpr int kMlpIn = 12;
constexpr int kMlpH = 32;
enum MlpOffsets : int {
    kOW1 = 0,
    kOb1 = kOW1 + kMlpIn * kMlpH,
    kOW2 = kOb1 + kMlpH,
    kOb2 = kOW2 + kMlpH * kMlpH,
    kOw3 = kOb2 + kMlpH,
    kOb3 = kOw3 + kMlpH,
    kMlpTrain = kOb3 + 1,
    kOMean = kMlpTrain,
    kOIstd = kOMean + kMlpIn,
    kOScale = kOIstd + kMlpIn,
    kMlpParams = kOScale + 1
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Four floats to bf16 bits, round to nearest even
__device__ __forceinline__ s16x4 pack_bf16(f32x4 v)
{
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(s16x4, __builtin_convertvector(v, bf16x4));
}
// The hardware reciprocal (1 ulp) instead of a correctly rounded division:
// the network runs in bf16, whose rounding is 2^-9.
__device__ __forceinline__ float sigmoidf_(float z) { return __builtin_amdgcn_rcpf(1.f + __expf(-z)); }
__device__ __forceinline__ float siluf_(float z) { return z * sigmoidf_(z); }
__device__ __forceinline__ float softplusf_(float z) { return z > 20.f ? z : log1pf(__expf(z)); }

// 16x16x16 bf16 MFMA tile product on one wavefront: lane (r = lane%16,
// g = lane/16) supplies A[r][4g..4g+3] and B[4g..4g+3][r] and receives
// C[4g..4g+3][r].
__device__ __forceinline__ f32x4 mfma16(s16x4 a, s16x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Block-shared copy of the weights: the MFMA operands bf16, lane by lane as the
// forward pass takes them (left operands of W1^T and W2^T: lane (r, g) holds
// rows r, inputs 4g..4g+3 of a 16x16 tile).
struct MlpShared {
    s16x4 W1[2][64];   // [hidden tile]; inputs >= kMlpIn are zero
    s16x4 W2[4][64];   // [2*(input tile) + output tile]
    float b1[kMlpH], b2[kMlpH], w3[kMlpH];
    float mean[16], istd[16];  // standardisation; 0 past kMlpIn
    float b3, scale;
};

// All threads of the block; the caller synchronises afterwards.
__device__ inline void mlp_stage(MlpShared &s, const float *P)
{
    for (int i = threadIdx.x; i < 6 * 64; i += blockDim.x) {
        const int tile = i >> 6, r = i & 15, g = i >> 4 & 3;
        f32x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = 4 * g + q;
            if (tile < 2)
                v[q] = k < kMlpIn ? P[kOW1 + k * kMlpH + 16 * tile + r] : 0.f;
            else
                v[q] = P[kOW2 + (16 * ((tile - 2) >> 1) + k) * kMlpH + 16 * ((tile - 2) & 1) + r];
        }
        (tile < 2 ? s.W1[tile] : s.W2[tile - 2])[i & 63] = pack_bf16(v);
    }
    for (int i = threadIdx.x; i < kMlpH; i += blockDim.x) {
        s.b1[i] = P[kOb1 + i];
        s.b2[i] = P[kOb2 + i];
        s.w3[i] = P[kOw3 + i];
    }
    for (int i = threadIdx.x; i < 16; i += blockDim.x) {
        s.mean[i] = i < kMlpIn ? P[kOMean + i] : 0.f;
        s.istd[i] = i < kMlpIn ? P[kOIstd + i] : 0.f;
    }
    if (threadIdx.x == 0) {
        s.b3 = P[kOb3];
        s.scale = P[kOScale];
    }
}

// Features of one element node from its pass-1 quantities.
// Gij[i][j] = du_i/dx_j, hinv[i][d] = He(i,d).
template <typename T>
__device__ __forceinline__ void mlp_features(const T (&Gij)[3][3], T rho, const T (&u)[3],
                                             const T (&hinv)[3][3], float f[kMlpIn])
{
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) f[3 * i + j] = (float)Gij[i][j];
    f[9] = (float)rho;
    f[10] = sqrtf((float)(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]));
    const double det = (double)hinv[0][0] * ((double)hinv[1][1] * hinv[2][2] - (double)hinv[1][2] * hinv[2][1]) -
                       (double)hinv[0][1] * ((double)hinv[1][0] * hinv[2][2] - (double)hinv[1][2] * hinv[2][0]) +
                       (double)hinv[0][2] * ((double)hinv[1][0] * hinv[2][1] - (double)hinv[1][1] * hinv[2][0]);
    f[11] = 2.f * __builtin_amdgcn_rcpf(cbrtf(fabsf((float)det)));  // det J = 1/det He
}

// Orders this wave's LDS accesses (a wave's LDS operations complete in
// issue order; the fence keeps the compiler from moving them across).
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// z3 of the MLP for this lane's node (mu_sgs = scale*softplus(z3)); x(mt):
// the standardised bf16 inputs 4g..4g+3 of node 16 mt + r, for lane (r, g).  All
// 64 lanes of the wave call it.  No LDS besides the weights: the layers chain
// in registers and 3 lane exchanges sum the output layer (a forward pass that
// carried the hidden layer through LDS: 3.68 against 2.95 ms for the fused
// diffusion at 96^3 order 3).  The sums keep one order, over the units by fours
// and then by lane groups, in every caller.
template <class X>
__device__ __forceinline__ float mlp_z3(const MlpShared &s, X x)
{
    const int lane = threadIdx.x & 63, g = lane >> 4;
    f32x4 b1[2], b2[2], w3[2];
    s16x4 W1[2], W2[4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        b1[t] = *reinterpret_cast<const f32x4 *>(&s.b1[16 * t + 4 * g]);
        b2[t] = *reinterpret_cast<const f32x4 *>(&s.b2[16 * t + 4 * g]);
        w3[t] = *reinterpret_cast<const f32x4 *>(&s.w3[16 * t + 4 * g]);
        W1[t] = s.W1[t][lane];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) W2[t] = s.W2[t][lane];
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    float part[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        const s16x4 xb = x(mt);
        s16x4 h[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            f32x4 z = mfma16(W1[t], xb, zero);
#pragma unroll
            for (int q = 0; q < 4; ++q) z[q] = siluf_(z[q] + b1[t][q]);
            h[t] = pack_bf16(z);
        }
        float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const f32x4 z = mfma16(W2[2 + t], h[1], mfma16(W2[t], h[0], zero));
#pragma unroll
            for (int q = 0; q < 4; ++q) p[q] += siluf_(z[q] + b2[t][q]) * w3[t][q];
        }
        part[mt] = (p[0] + p[1]) + (p[2] + p[3]);
    }
    // sum over the four lane groups, group g keeping node tile g: each
    // exchange hands over the half of the tiles that the partner keeps
    const bool hi = lane & 32, odd = lane & 16;
    const float a0 = (odd ? part[1] : part[0]) + __shfl_xor(odd ? part[0] : part[1], 16);
    const float a1 = (odd ? part[3] : part[2]) + __shfl_xor(odd ? part[2] : part[3], 16);
    return (hi ? a1 : a0) + __shfl_xor(hi ? a0 : a1, 32) + s.b3;
}

// The same for features held by the lanes themselves.  scratch: this wave's LDS
// area, four tiles of 16 rows of 16 shorts, TS shorts apart, used by this wave
// only (no block barrier inside).  Inactive lanes pass any finite features.
template <int TS = 256>
__device__ __forceinline__ float mlp_forward_z3(const MlpShared &s, const float (&feat)[kMlpIn], short *scratch)
{
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    s16x4 *row = reinterpret_cast<s16x4 *>(&scratch[g * TS + r * 16]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        f32x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = (feat[4 * k + q] - s.mean[4 * k + q]) * s.istd[4 * k + q];
        row[k] = pack_bf16(v);
    }
    row[3] = s16x4{0, 0, 0, 0};
    wave_lds_sync();
    s16x4 xb[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) xb[mt] = *reinterpret_cast<const s16x4 *>(&scratch[mt * TS + r * 16 + 4 * g]);
    const float z3 = mlp_z3(s, [&](int mt) { return xb[mt]; });
    wave_lds_sync();
    return z3;
}

}  // namespace msod
