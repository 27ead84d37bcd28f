// Learned subgrid-viscosity closure: the GPU side of training and inference.
//
// The diffusive residual is affine in mu_sgs (elem_diffu.f90:70,146): at an
// element node a, mu_sgs enters the stress through mu_f' = mu_f + rho*mu_sgs
// and the heat conductivity through kappa += Cp*rho*mu_sgs/0.9.  Hence, for a
// nodal error field r (momentum x3, energy), the gradient of <r, R(mu_sgs)>
// with respect to mu_sgs(e,a) is
//   g(e,a) = rho gpvol sum_d sum_i He(i,d) [ sum_k D_d[r_mom_k](a) S_ki
//                                             + D_d[r_ener](a) (S u)_i ]
//            + r_ener(a) * Cp rho / 0.9 * W[grad T](a)
// with S = G + G^T - 2/3 div(u) I (G = grad u), D_d the 1-D derivative along
// direction d inside the element, and W[grad T] the element's transposed
// sweep of the heat flux (the same quantities the forward kernel forms).
// k_adjoint computes g for every element node; k_mlp_grad back-propagates it
// through the MLP with bf16 MFMA products and FP32 accumulation.
#include <cmath>

#include "msod_columns.h"
#include "msod_mlp.h"
#include "msod_closure.h"

namespace msod {

// ---------------------------------------------------------------------------
// element kernels: features (MODE 0) and mu_sgs gradients (MODE 1)
// ---------------------------------------------------------------------------
// One node per thread; several elements per workgroup while they fit 256 threads.
template <int P>
struct ElemShape {
    static constexpr int Q = P + 1;
    static constexpr int NN = Q * Q * Q;
    static constexpr int EPB = NN <= 128 ? 256 / NN : 1;
    static constexpr int NT = NN <= 128 ? 256 : ((NN + 63) / 64) * 64;
};

template <int P, int MODE>
__global__ void __launch_bounds__(ElemShape<P>::NT) k_closure_elem(ClosureElemArgs a)
{
    using S = ElemShape<P>;
    constexpr int Q = S::Q, NN = S::NN, EPB = S::EPB;
    __shared__ double sD[Q * Q];
    __shared__ double sA[EPB][5][NN];                  // rho, T, u0, u1, u2
    __shared__ double sE[EPB][MODE ? 4 : 1][NN];       // error field (MODE 1)
    __shared__ double sF[EPB][MODE ? 3 : 1][NN];       // heat flux, contravariant

    const int64_t groups = (a.nelem + EPB - 1) / EPB;
    // from the mesh's end, whose geometry the diffusion before left in the memory-
    // side cache (training step at 32^3 order 3 525 -> 520 us)
    const int64_t grp = groups - 1 - (int64_t)blockIdx.x;
    if (grp < 0) return;  // whole block
    const int t = threadIdx.x;
    for (int i = t; i < Q * Q; i += blockDim.x) sD[i] = a.tab.D[i];
    const int le = t / NN;
    const int l = t - le * NN;
    const int64_t e = grp * EPB + le;
    const bool active = (le < EPB) && (e < a.nelem);
    const int I = l % Q, J = (l / Q) % Q, K = l / (Q * Q);
    double r = 0, uu[3] = {0, 0, 0}, rerr_ener = 0;
    if (active) {
        const int64_t g = a.conn[a.lanes ? ElemEntry<P>{e, l}.entry() : e * NN + l];
        const int64_t np = a.npoin;
        r = a.rho[g];
        sA[le][0][l] = r;
        sA[le][1][l] = MODE ? a.Tem[g] : 0.0;
        for (int d = 0; d < 3; ++d) {
            uu[d] = a.u[g + d * np];
            sA[le][2 + d][l] = uu[d];
        }
        if (MODE) {
            for (int c = 0; c < 4; ++c) sE[le][c % (MODE ? 4 : 1)][l] = a.rerr[g + c * np];
            rerr_ener = a.rerr[g + 3 * np];
        }
    }
    __syncthreads();

    double h[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, G[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    double gT[3] = {0, 0, 0}, V[4][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, gv = 0;
    if (active) {
        const ElemEntry<P> en{e, l};
        const GeoPair<double> *gp = reinterpret_cast<const GeoPair<double> *>(a.geo) + (a.lanes ? en.pair() : e * 5 * NN + l);
        const int stride = a.lanes ? en.pair_stride() : NN;
        GeoNode<double> gn;
#pragma unroll
        for (int c = 0; c < 5; ++c) gn.v[c] = gp[c * stride];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int i = 0; i < 3; ++i) h[i][d] = gn.he(i + 3 * d);
        gv = gn.gvol();
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int Id = d == 0 ? I : (d == 1 ? J : K);
            const int stride = d == 0 ? 1 : (d == 1 ? Q : Q * Q);
            const int base = l - Id * stride;
            double aT = 0, aU0 = 0, aU1 = 0, aU2 = 0, aE[4] = {0, 0, 0, 0};
#pragma unroll 1
            for (int n = 0; n < Q; ++n) {
                const int s = base + n * stride;
                const double Dv = sD[Id * Q + n];
                aT += Dv * sA[le][1][s];
                aU0 += Dv * sA[le][2][s];
                aU1 += Dv * sA[le][3][s];
                aU2 += Dv * sA[le][4][s];
                if (MODE)
#pragma unroll
                    for (int c = 0; c < 4; ++c) aE[c] += Dv * sE[le][c % (MODE ? 4 : 1)][s];
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                gT[i] += h[i][d] * aT;
                G[0][i] += h[i][d] * aU0;
                G[1][i] += h[i][d] * aU1;
                G[2][i] += h[i][d] * aU2;
            }
            if (MODE)
#pragma unroll
                for (int c = 0; c < 4; ++c) V[c][d] = aE[c];
        }
    }
    if (MODE == 0) {
        if (active) {
            float f[kMlpIn];
            mlp_features<double>(G, r, uu, h, f);
#pragma unroll
            for (int k = 0; k < kMlpIn; ++k) a.feat[(e * NN + l) * kMlpIn + k] = f[k];
        }
        return;
    }
    // heat-flux transposed sweep W[grad T] at this node
    if (active)
#pragma unroll
        for (int d = 0; d < 3; ++d)
            sF[le][d % (MODE ? 3 : 1)][l] = gv * (h[0][d] * gT[0] + h[1][d] * gT[1] + h[2][d] * gT[2]);
    __syncthreads();
    if (!active) return;
    double WT = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int Id = d == 0 ? I : (d == 1 ? J : K);
        const int stride = d == 0 ? 1 : (d == 1 ? Q : Q * Q);
        const int base = l - Id * stride;
#pragma unroll 1
        for (int n = 0; n < Q; ++n) WT += sD[n * Q + Id] * sF[le][d % (MODE ? 3 : 1)][base + n * stride];
    }
    const double divU = G[0][0] + G[1][1] + G[2][2];
    double Sm[3][3], Su[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        double acc = 0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            Sm[i][j] = G[i][j] + G[j][i];
            acc += Sm[i][j] * uu[j];
        }
        Su[i] = acc - (2.0 / 3.0) * divU * uu[i];
        Sm[i][i] -= (2.0 / 3.0) * divU;
    }
    double acc = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int i = 0; i < 3; ++i)
            acc += h[i][d] * (V[0][d] * Sm[0][i] + V[1][d] * Sm[1][i] + V[2][d] * Sm[2][i] + V[3][d] * Su[i]);
    const double gnu = r * gv * acc + rerr_ener * a.Cp * r / 0.9 * WT;
    a.gnu[e * NN + l] = (float)gnu;
}

// ---------------------------------------------------------------------------
// MLP: inference into mu_sgs (reference layout), and parameter gradients
// ---------------------------------------------------------------------------
// Four features of a sample, from an address that need not be 16-byte aligned.
__device__ __forceinline__ f32x4 load_feat4(const float *p, bool aligned)
{
    if (aligned) return *reinterpret_cast<const f32x4 *>(p);
    return f32x4{p[0], p[1], p[2], p[3]};
}

// mu_sgs(nelem,nn) from the features [nelem*nn][12].  A workgroup takes kPE
// elements and at most kPL of their nodes: the samples are read in memory
// order, and the results change lanes in LDS, so that each store fills kPE
// consecutive elements of one node (the reference layout puts an element's
// nodes 8*nelem bytes apart; with the sample's lane storing it 82 us at 32^3
// order 3, now 68, most of it the activations).
constexpr int kPE = 16, kPL = 64;
__global__ void __launch_bounds__(256) k_mlp_predict(const float *P, const float *feat, int64_t nelem, int nn,
                                                     const int32_t *l2g, double *mu_sgs)
{
    __shared__ MlpShared s;
    __shared__ double out[kPE][kPL + 1];
    mlp_stage(s, P);
    __syncthreads();
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int64_t e0 = (int64_t)blockIdx.x * kPE;
    const int l0 = blockIdx.y * kPL, nl = nn - l0 < kPL ? nn - l0 : kPL;
    const int ne = (int)(nelem - e0 < kPE ? nelem - e0 : kPE), total = ne * nl;
    const bool aligned = ((uintptr_t)feat & 15) == 0;
    const short all = g < 3 ? -1 : 0;
    const s16x4 real = {all, all, all, all};
    const f32x4 mean = *reinterpret_cast<const f32x4 *>(&s.mean[4 * g]);
    const f32x4 istd = *reinterpret_cast<const f32x4 *>(&s.istd[4 * g]);
    for (int base = (threadIdx.x >> 6) * 64; base < total; base += 256) {
        const float z3 = mlp_z3(s, [&](int mt) {
            const int i = base + 16 * mt + r, ic = i < total ? i : total - 1;
            const int64_t smp = (e0 + ic / nl) * nn + l0 + ic % nl;
            // lanes of inputs 12..15 read 0..3 and hold zeros (an infinite
            // feature times zero would be a NaN)
            const f32x4 f = load_feat4(feat + smp * kMlpIn + (g < 3 ? 4 * g : 0), aligned);
            return pack_bf16((f - mean) * istd) & real;
        });
        const int i = base + lane;
        if (i < total) out[i / nl][i % nl] = (double)(s.scale * softplusf_(z3));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nl * kPE; i += 256) {
        const int e = i % kPE, l = i / kPE;
        if (e < ne) mu_sgs[e0 + e + nelem * (int64_t)l2g[l0 + l]] = out[e][l];
    }
}

// Parameter gradient.  A workgroup's four waves take four chunks of 64 samples
// at a time; its sum, chunk after chunk in a fixed order, goes to
// partial[blockIdx.x][kMlpTrain].
//
// The layers are formed transposed as in the forward pass (lane (r, g): sample
// r of a tile of 16, hidden units 4g..4g+3), so that forward and backward
// products chain in registers; one sigmoid per activation serves the value and
// the derivative.  Through the wave's own LDS go the operands of the weight
// gradients, which contract over the samples, and the sums over the output
// layer's 32 units (a lane per sample) and over the samples (a lane per unit),
// which keep one fixed sequential order.  What bounds it: the activations (64
// exponentials and reciprocals a sample) and the LDS.  2.1 M samples: 760 us
// with one wave per workgroup and every operand gathered from LDS in 16-bit
// pieces, 150 us now.
constexpr int kGW = 4;     // waves per workgroup
constexpr int kLH = 68;    // LDS row strides: 64 floats,
constexpr int kLT = 20;    // 16 floats or shorts, padded
struct MlpGradWave {
    float H2[kMlpH][kLH];  // silu(Z2), [unit][sample]
    float S[kMlpH][kLT];   // silu'(Z2), then dZ1, of one tile
    short H1[kMlpH][kLT];  // bf16 operands of one tile, [unit][sample]
    short D[kMlpH][kLT];   // dZ2, then dZ1
    short X[16][kLT];      // inputs
    float dz3[64];
};
union MlpGradShared {
    MlpGradWave w[kGW];
    float sum[kGW][kMlpTrain];  // the waves' chunk sums
};

__global__ void __launch_bounds__(64 * kGW, 2) k_mlp_grad(const float *P, const float *feat, const float *gnu,
                                                       int64_t nsamp, float *partial)
{
    __shared__ __attribute__((aligned(16))) MlpGradShared sh;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    MlpGradWave &L = sh.w[wave];
    // left operands: row r, columns 4g..4g+3
    s16x4 W1t[2], W2t[2][2], W2[2][2];  // W1^T[t]; W2^T[in][out]; W2[in][out]
    f32x4 b1[2], b2[2], w3[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        f32x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[q] = 4 * g + q < kMlpIn ? P[kOW1 + (4 * g + q) * kMlpH + 16 * t + r] : 0.f;
            b1[t][q] = P[kOb1 + 16 * t + 4 * g + q];
            b2[t][q] = P[kOb2 + 16 * t + 4 * g + q];
            w3[t][q] = P[kOw3 + 16 * t + 4 * g + q];
        }
        W1t[t] = pack_bf16(v);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = P[kOW2 + (16 * k + 4 * g + q) * kMlpH + 16 * t + r];
            W2t[k][t] = pack_bf16(v);
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = P[kOW2 + (16 * k + r) * kMlpH + 16 * t + 4 * g + q];
            W2[k][t] = pack_bf16(v);
        }
    }
    const auto Pu = (const __attribute__((address_space(4))) float *)P;
    const float scale = Pu[kOScale], w3c = P[kOw3 + (lane & 31)];
    f32x4 mean, istd;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        mean[q] = g < 3 ? P[kOMean + (g < 3 ? 4 * g + q : 0)] : 0.f;
        istd[q] = g < 3 ? P[kOIstd + (g < 3 ? 4 * g + q : 0)] : 0.f;
    }
    const bool aligned = ((uintptr_t)feat & 15) == 0;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    constexpr int kPT = (kMlpTrain + 64 * kGW - 1) / (64 * kGW);
    float run[kPT];  // the workgroup's sum of entries threadIdx.x + 256 j
#pragma unroll
    for (int j = 0; j < kPT; ++j) run[j] = 0.f;

    const int64_t nchunk = (nsamp + 63) / 64;
    for (int64_t c0 = blockIdx.x; c0 < nchunk; c0 += (int64_t)gridDim.x * kGW) {
        const int64_t chunk = c0 + (int64_t)gridDim.x * wave;
        f32x4 dW1[2] = {zero, zero}, dW2[2][2] = {{zero, zero}, {zero, zero}};
        float s23 = 0.f, s1 = 0.f, s3 = 0.f;  // lanes 0..31: dw3, db1; 32..63: db2; all: db3
        if (chunk < nchunk) {
            s16x4 xb[4], h1[4][2];
            f32x4 ds1[4][2], ds2[4][2];
            f32x4 f[4];
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                const int64_t i = chunk * 64 + 16 * mt + r;
                f[mt] = load_feat4(feat + (i < nsamp ? i : nsamp - 1) * kMlpIn + (g < 3 ? 4 * g : 0), aligned);
            }
            const int64_t me = chunk * 64 + lane;
            const float gv = gnu[me < nsamp ? me : nsamp - 1];
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                const bool valid = chunk * 64 + 16 * mt + r < nsamp;
                xb[mt] = pack_bf16((f[mt] - mean) * istd);
                if (!valid || g == 3) xb[mt] = s16x4{0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    f32x4 z = mfma16(W1t[t], xb[mt], zero);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float zz = z[q] + b1[t][q], sg = sigmoidf_(zz);
                        z[q] = zz * sg;
                        ds1[mt][t][q] = sg * (1.f + zz * (1.f - sg));
                    }
                    h1[mt][t] = pack_bf16(z);
                }
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const f32x4 z = mfma16(W2t[1][t], h1[mt][1], mfma16(W2t[0][t], h1[mt][0], zero));
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float zz = z[q] + b2[t][q], sg = sigmoidf_(zz);
                        L.H2[16 * t + 4 * g + q][16 * mt + r] = zz * sg;
                        ds2[mt][t][q] = sg * (1.f + zz * (1.f - sg));
                    }
                }
            }
            wave_lds_sync();
            float z3 = Pu[kOb3];
#pragma unroll
            for (int c = 0; c < kMlpH; ++c) z3 += L.H2[c][lane] * Pu[kOw3 + c];
            L.dz3[lane] = me < nsamp ? gv * scale * sigmoidf_(z3) : 0.f;
            wave_lds_sync();
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                const float d = L.dz3[16 * mt + r];
                s16x4 d2[2];
#pragma unroll
                for (int q = 0; q < 4; ++q) L.X[4 * g + q][r] = xb[mt][q];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    f32x4 v;
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = d * w3[t][q] * ds2[mt][t][q];
                    d2[t] = pack_bf16(v);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int n = 16 * t + 4 * g + q;
                        L.S[n][r] = ds2[mt][t][q];
                        L.H1[n][r] = h1[mt][t][q];
                        L.D[n][r] = d2[t][q];
                    }
                }
                wave_lds_sync();
                // dw3 = sum dz3 silu(Z2), db2 = sum dz3 w3 silu'(Z2), db3 = sum dz3
                {
                    const float *col = lane < 32 ? &L.H2[lane & 31][16 * mt] : L.S[lane & 31];
                    const float wl = lane < 32 ? 1.f : w3c;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const f32x4 z = *reinterpret_cast<const f32x4 *>(&L.dz3[16 * mt + 4 * i]);
                        const f32x4 v = *reinterpret_cast<const f32x4 *>(&col[4 * i]);
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            s23 += z[q] * wl * v[q];
                            s3 += z[q];
                        }
                    }
                }
                // dW2 = H1^T dZ2; dZ1^T = (W2 dZ2^T) silu'(Z1)
                s16x4 av[2], bv[2];
                f32x4 dz1[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    av[t] = *reinterpret_cast<const s16x4 *>(&L.H1[16 * t + r][4 * g]);
                    bv[t] = *reinterpret_cast<const s16x4 *>(&L.D[16 * t + r][4 * g]);
                }
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int k = 0; k < 2; ++k) dW2[k][t] = mfma16(av[k], bv[t], dW2[k][t]);
                    dz1[t] = mfma16(W2[t][1], d2[1], mfma16(W2[t][0], d2[0], zero)) * ds1[mt][t];
                }
                wave_lds_sync();
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const s16x4 d1 = pack_bf16(dz1[t]);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int n = 16 * t + 4 * g + q;
                        L.S[n][r] = dz1[t][q];
                        L.D[n][r] = d1[q];
                    }
                }
                wave_lds_sync();
                // db1 = sum dZ1; dW1 = X^T dZ1
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(&L.S[lane & 31][4 * i]);
#pragma unroll
                    for (int q = 0; q < 4; ++q) s1 += v[q];
                }
                const s16x4 xt = *reinterpret_cast<const s16x4 *>(&L.X[r][4 * g]);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    bv[t] = *reinterpret_cast<const s16x4 *>(&L.D[16 * t + r][4 * g]);
                    dW1[t] = mfma16(xt, bv[t], dW1[t]);
                }
                wave_lds_sync();
            }
        }
        // the chunks' sums, added in the order of the chunks
        __syncthreads();  // every wave is done with its part of the LDS
        float *sum = sh.sum[wave];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (4 * g + q < kMlpIn) sum[kOW1 + (4 * g + q) * kMlpH + 16 * t + r] = dW1[t][q];
#pragma unroll
                for (int k = 0; k < 2; ++k) sum[kOW2 + (16 * k + 4 * g + q) * kMlpH + 16 * t + r] = dW2[k][t][q];
            }
        sum[(lane < 32 ? kOw3 : kOb2) + (lane & 31)] = s23;
        if (lane < 32) sum[kOb1 + lane] = s1;
        if (lane == 0) sum[kOb3] = s3;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kPT; ++j) {
            const int i = threadIdx.x + 64 * kGW * j;
            if (i < kMlpTrain)
                for (int w = 0; w < kGW && c0 + (int64_t)gridDim.x * w < nchunk; ++w) run[j] += sh.sum[w][i];
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < kPT; ++j) {
        const int i = threadIdx.x + 64 * kGW * j;
        if (i < kMlpTrain) partial[(int64_t)blockIdx.x * kMlpTrain + i] = run[j];
    }
}

// Sum of the workgroups' rows in FP64: 64 columns per workgroup, 16 lanes of
// rows each, then a fixed tree (one thread per column over all rows: 248 us
// for 1024 rows, now 6).
__global__ void __launch_bounds__(1024) k_grad_reduce(const float *partial, int nblocks, float *grad)
{
    __shared__ double red[16][64];
    const int c = threadIdx.x & 63, k = threadIdx.x >> 6, j = blockIdx.x * 64 + c;
    double s = 0.0;
    if (j < kMlpTrain)
#pragma unroll 8
        for (int b = k; b < nblocks; b += 16) s += partial[(int64_t)b * kMlpTrain + j];
    red[k][c] = s;
    for (int h = 8; h > 0; h >>= 1) {
        __syncthreads();
        if (k < h) red[k][c] += red[k + h][c];
    }
    if (k == 0 && j < kMlpTrain) grad[j] = (float)red[0][c];
}

// Adam (Kingma & Ba 2015, Algorithm 1).  ob1 = 1 - b1, ob2 = 1 - b2 and the
// bias corrections c1, c2 come from the host in double.
__global__ void k_adam(float *P, const float *grad, float *m, float *v, float lr, float b1, float b2,
                       float ob1, float ob2, float eps, float c1, float c2)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= kMlpTrain) return;
    const float gj = grad[j];
    const float mj = b1 * m[j] + ob1 * gj;
    const float vj = b2 * v[j] + ob2 * gj * gj;
    m[j] = mj;
    v[j] = vj;
    P[j] -= lr * (mj / c1) / (sqrtf(vj / c2) + eps);
}

// r = 2 w_c (R_c - target_c) for the momentum and energy residuals; loss
// partial sums per block (w_c (R_c - target_c)^2).
__global__ void k_residual_error(const double *Rmom, const double *Rener, const double *target,
                                 const double *w, int64_t npoin, double *rerr, double *lpart)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < npoin;
         i += (int64_t)gridDim.x * blockDim.x) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const double R = c < 3 ? Rmom[i + c * npoin] : Rener[i];
            const double d = R - target[i + c * npoin];
            rerr[i + c * npoin] = 2.0 * w[c] * d;
            acc += w[c] * d * d;
        }
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) lpart[blockIdx.x] = red[0];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <int P, int MODE>
static hipError_t launch_elem_p(const ClosureElemArgs &a, hipStream_t s)
{
    using S = ElemShape<P>;
    const int64_t groups = (a.nelem + S::EPB - 1) / S::EPB;
    hipLaunchKernelGGL((k_closure_elem<P, MODE>), dim3((unsigned)groups), dim3(S::NT), 0, s, a);
    return hipGetLastError();
}

template <int MODE>
static hipError_t launch_elem(int porder, const ClosureElemArgs &a, hipStream_t s)
{
    switch (porder) {
    case 1: return launch_elem_p<1, MODE>(a, s);
    case 2: return launch_elem_p<2, MODE>(a, s);
    case 3: return launch_elem_p<3, MODE>(a, s);
    case 4: return launch_elem_p<4, MODE>(a, s);
    case 5: return launch_elem_p<5, MODE>(a, s);
    case 6: return launch_elem_p<6, MODE>(a, s);
    case 7: return launch_elem_p<7, MODE>(a, s);
    case 8: return launch_elem_p<8, MODE>(a, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_closure_features(int porder, const ClosureElemArgs &a, hipStream_t s)
{
    return launch_elem<0>(porder, a, s);
}

hipError_t launch_closure_adjoint(int porder, const ClosureElemArgs &a, hipStream_t s)
{
    return launch_elem<1>(porder, a, s);
}

hipError_t launch_mlp_predict(const float *P, const float *feat, int64_t nelem, int nn,
                              const int32_t *l2g, double *mu_sgs, hipStream_t s)
{
    hipLaunchKernelGGL(k_mlp_predict, dim3((unsigned)((nelem + kPE - 1) / kPE), (nn + kPL - 1) / kPL), dim3(256), 0, s,
                       P, feat, nelem, nn, l2g, mu_sgs);
    return hipGetLastError();
}

hipError_t launch_mlp_grad(const float *P, const float *feat, const float *gnu, int64_t nsamp,
                           float *partial, int nblocks, float *grad, hipStream_t s)
{
    hipLaunchKernelGGL(k_mlp_grad, dim3(nblocks), dim3(64 * kGW), 0, s, P, feat, gnu, nsamp, partial);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_grad_reduce, dim3((kMlpTrain + 63) / 64), dim3(1024), 0, s, partial, nblocks, grad);
    return hipGetLastError();
}

hipError_t launch_adam(float *P, const float *grad, float *m, float *v, int step, double lr, double b1,
                       double b2, double eps, hipStream_t s)
{
    const double c1 = 1.0 - std::pow(b1, step), c2 = 1.0 - std::pow(b2, step);
    hipLaunchKernelGGL(k_adam, dim3((kMlpTrain + 255) / 256), dim3(256), 0, s, P, grad, m, v, (float)lr,
                       (float)b1, (float)b2, (float)(1.0 - b1), (float)(1.0 - b2), (float)eps, (float)c1,
                       (float)c2);
    return hipGetLastError();
}

hipError_t launch_residual_error(const double *Rmom, const double *Rener, const double *target,
                                 const double *w, int64_t npoin, double *rerr, double *lpart, int nblocks,
                                 hipStream_t s)
{
    hipLaunchKernelGGL(k_residual_error, dim3(nblocks), dim3(256), 0, s, Rmom, Rener, target, w, npoin, rerr,
                       lpart);
    return hipGetLastError();
}

}  // namespace msod
