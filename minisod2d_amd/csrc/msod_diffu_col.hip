// Diffusive residual, column kernel (porder 1..kColMaxP); see msod_columns.h
// for the thread layout and msod_diffu.hip for the reference it stands for.
//
// Per slice K of the element's nodes:
//  1. rho, T, u of the slice in LDS; gradients along I and J from there, along
//     K from the thread's column; He gives grad rho, grad T, G = grad u, then
//     the stress tau and tau.u.
//  2. the contravariant fluxes F_d = gpvol sum_i He(i,d) Phi_i of the six flux
//     vectors Phi (grad rho, tau.u, grad T, the rows of tau): those of d = I, J
//     go to LDS, those of d = K are added at once into the column's six sums
//     W[K'] with D[K][K'].
//  3. the transposed sweeps along I and J from LDS into W[K].
// After the last slice Rmass = nu_e W0, Rmom = W3..W5, Rener = W1 + kappa_e W2,
// with nu_e and kappa_e of the target node.
//
// CLOSURE (FP64 storage): mu_sgs is not read but predicted by the learned
// closure (msod_mlp.h) from the velocity gradient before the stress is
// formed; its per-wave LDS scratch is the wave's own part of the flux buffer,
// free between the slice's first barrier and the fluxes.
#include <type_traits>

#include "msod_columns.h"
#include "msod_mlp.h"
#include "msod_closure.h"

namespace msod {

template <int P, bool COLORED, class A, bool CLOSURE, typename TA>
__global__ void __launch_bounds__(ColShape<P>::NT, 2) k_diffu_col(A a, const float *mlp)
{
    using S = ColShape<P>;
    using T = TA;
    using TG = typename A::G;
    constexpr int Q = S::Q, QQ = S::QQ, EPB = S::EPB, LANES = S::LANES, NT = S::NT;
    constexpr int LA = 2;  // line sources read ahead of their use (3 and 4: no faster; order 5 spills)
    struct alignas(2 * sizeof(T)) V2 { T x, y; };
    __shared__ T sD[Q * Q];
    __shared__ V2 sP[2][NT];  // one slice: (r,T) (u0,u1)
    __shared__ T sU2[NT];     // and u2
    __shared__ __attribute__((aligned(16))) V2 sF[6][NT];  // its fluxes along I (0..2) and J (3..5)
    __shared__ TG sMu[2][NT];                              // its mu_e, mu_sgs
    __shared__ typename std::conditional<CLOSURE, MlpShared, char>::type smlp;
    extern __shared__ __attribute__((aligned(16))) double sR[];  // node sums [5][US]

    const Plan &pl = a.plan;
    const int US = pl.ustride, t = threadIdx.x;
    const ColThread<P> th(t);
    const int tc = th.tc, le = th.le, I = th.I, J = th.J;
    const int64_t np = a.npoin;
    const auto D = uniform(a.tab.D);
    const uint32_t slot = xcd_slot(blockIdx.x, gridDim.x);
    const uint32_t b = pl.batches ? uniform(pl.batches)[slot] : slot;
    const uint32_t u0 = uniform(pl.uoff)[b], U = uniform(pl.uoff)[b + 1] - u0;
    const int64_t e0 = (int64_t)b * EPB;
    const bool active = t < LANES && e0 + le < a.nelem;

    uint32_t gn[Q];
#pragma unroll
    for (int k = 0; k < Q; ++k) gn[k] = __builtin_nontemporal_load(&pl.conn[((int64_t)b * Q + k) * LANES + tc]);
    // mu_e and mu_sgs in the reference layout (nelem,ngaus) put one element's
    // values 8*nelem bytes apart and neighbouring elements side by side: they are
    // loaded with the element as the fastest lane index and change lanes in LDS
    const int lem = tc % EPB, Im = tc / EPB % Q, Jm = tc / (EPB * Q);
    const int lm = line_ref<P>(Im) + Q * line_ref<P>(Jm), tm = t < LANES ? Im + Q * (lem + EPB * Jm) : t;
    const int64_t em = e0 + lem < a.nelem ? e0 + lem : a.nelem - 1;
    int32_t gl[Q];
#pragma unroll
    for (int k = 0; k < Q; ++k) gl[k] = a.tab.l2g[lm + QQ * line_ref<P>(k)];
    const bool has_sgs = !CLOSURE && a.mu_sgs;  // NULL: closure fallback
    const TG *mu_sgs = has_sgs ? a.mu_sgs : a.mu_e;
    TG mue, mus = (TG)0;
    auto load_mu = [&](int k) {
        const int64_t ge = em + a.nelem * (int64_t)gl[k];
        mue = a.mu_e[ge];
        if constexpr (!CLOSURE) mus = mu_sgs[ge];
    };
    typename A::F fr[Q], fT[Q], fmu[Q];
    typename A::U fu[Q][3];
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const int64_t g = gn[k];
        fr[k] = a.rho[g];
        fT[k] = a.Tem[g];
#pragma unroll
        for (int d = 0; d < 3; ++d) fu[k][d] = a.u[g + d * np];
        fmu[k] = a.mu_fluid[g];
    }
    load_mu(0);
    GeoNode<TG> gk = col_geo<P, false>(a.geo, b, 0, tc);
    col_table<P>(a.tab.D, sD);
    if constexpr (CLOSURE) mlp_stage(smlp, mlp);
    for (int i = t; i < 5 * US; i += NT) sR[i] = 0.0;
    const T Cp = (T)a.Cp, Pr = (T)a.Pr;

    T r[Q], Te[Q], muf[Q], u[Q][3], W[Q][6], nu[Q], kappa[Q];
    uint32_t li[Q], wn[S::UPT];
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        r[k] = (T)fr[k];
        Te[k] = (T)fT[k];
        muf[k] = (T)fmu[k];
#pragma unroll
        for (int d = 0; d < 3; ++d) u[k][d] = (T)fu[k][d];
#pragma unroll
        for (int f = 0; f < 6; ++f) W[k][f] = 0;
    }
    const int sI = tc - I, sJ = tc - J * EPB * Q;  // a line's source n: sI + n, sJ + n*EPB*Q

#pragma unroll
    for (int k = 0; k < Q; ++k) {
        // the previous slice's values were read before its second barrier
        sP[0][t] = V2{r[k], Te[k]};
        sP[1][t] = V2{u[k][0], u[k][1]};
        sU2[t] = u[k][2];
        sMu[0][tm] = mue;
        sMu[1][tm] = mus;
        if (k + 1 < Q) load_mu(k + 1);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        // line derivatives x[d] of rho, T, u; the slice's geometry is still in
        // flight.  The line sources, first along I, then J, are read LA ahead of
        // their use.
        T x[3][5];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int f = 0; f < 5; ++f) x[d][f] = 0;
        V2 s0[LA], s1[LA];
        T s2[LA], Dv[LA];
        auto read_source = [&](int s) {
            const int m = s < Q ? sI + s : sJ + (s - Q) * EPB * Q;
            s0[s % LA] = sP[0][m];
            s1[s % LA] = sP[1][m];
            s2[s % LA] = sU2[m];
            Dv[s % LA] = s < Q ? sD[I * Q + s] : sD[J * Q + s - Q];
        };
#pragma unroll
        for (int s = 0; s < LA; ++s) read_source(s);
#pragma unroll
        for (int n = 0; n < Q; ++n) {
            const T Dk = (T)col_D<P>(D, k, n);
            x[2][0] += Dk * r[n];
            x[2][1] += Dk * Te[n];
            x[2][2] += Dk * u[n][0];
            x[2][3] += Dk * u[n][1];
            x[2][4] += Dk * u[n][2];
        }
#pragma unroll
        for (int f = 0; f < 5; ++f) asm volatile("" : "+v"(x[2][f]));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2 * Q; ++s) {
            const int d = s < Q ? 0 : 1, n = s % LA;
            x[d][0] += Dv[n] * s0[n].x;
            x[d][1] += Dv[n] * s0[n].y;
            x[d][2] += Dv[n] * s1[n].x;
            x[d][3] += Dv[n] * s1[n].y;
            x[d][4] += Dv[n] * s2[n];
            asm volatile("" : "+v"(x[d][0]), "+v"(x[d][1]), "+v"(x[d][2]), "+v"(x[d][3]), "+v"(x[d][4]));
            if (s + LA < 2 * Q) read_source(s + LA);
            __builtin_amdgcn_sched_barrier(0);
        }
        // grad rho, grad T, G[i][j] = d u_i / d x_j = sum_d He(j,d) D_d[u_i]
        T gR[3], gT[3], G[3][3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const T h0 = (T)gk.he(i), h1 = (T)gk.he(3 + i), h2 = (T)gk.he(6 + i);
            gR[i] = h0 * x[0][0] + h1 * x[1][0] + h2 * x[2][0];
            gT[i] = h0 * x[0][1] + h1 * x[1][1] + h2 * x[2][1];
#pragma unroll
            for (int c = 0; c < 3; ++c) G[c][i] = h0 * x[0][2 + c] + h1 * x[1][2 + c] + h2 * x[2][2 + c];
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
            asm volatile("" : "+v"(gR[i]), "+v"(gT[i]), "+v"(G[0][i]), "+v"(G[1][i]), "+v"(G[2][i]));
        __builtin_amdgcn_sched_barrier(0);
        const T me = (T)sMu[0][tc], gv = (T)gk.gvol();
        T ms = has_sgs ? (T)sMu[1][tc] : (T)0;
        if constexpr (CLOSURE) {
            float f[kMlpIn];
            T hinv[3][3];
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int d = 0; d < 3; ++d) hinv[i][d] = (T)gk.he(i + 3 * d);
            mlp_features<T>(G, r[k], u[k], hinv, f);
            // idle lanes hold a real element node (finite features)
            const float z3 =
                mlp_forward_z3<NT * (int)sizeof(V2) / 2>(smlp, f, reinterpret_cast<short *>(&sF[0][t & ~63]));
            ms = (T)(smlp.scale * softplusf_(z3));
        }
        nu[k] = (T)a.c_rho * me / r[k];
        kappa[k] = muf[k] * Cp / Pr + (T)a.c_ener * me * Cp / Pr + Cp * r[k] * ms / (T)0.9;
        asm volatile("" : "+v"(nu[k]), "+v"(kappa[k]));
        __builtin_amdgcn_sched_barrier(0);
        const T mu_f = muf[k] + r[k] * ms, mu_t = mu_f + me;
        const T lam = mu_f * (T)(2.0 / 3.0) * (G[0][0] + G[1][1] + G[2][2]);
        T tau[3][3], tauU[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            T acc = 0;
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                tau[i][j] = mu_t * (G[i][j] + G[j][i]);
                acc += tau[i][j] * u[k][j];
            }
            tauU[i] = acc - lam * u[k][i];
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) tau[i][i] -= lam;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const T c0 = gv * (T)gk.he(3 * d), c1 = gv * (T)gk.he(3 * d + 1), c2 = gv * (T)gk.he(3 * d + 2);
            T F[6];
            F[0] = c0 * gR[0] + c1 * gR[1] + c2 * gR[2];
            F[1] = c0 * tauU[0] + c1 * tauU[1] + c2 * tauU[2];
            F[2] = c0 * gT[0] + c1 * gT[1] + c2 * gT[2];
#pragma unroll
            for (int i = 0; i < 3; ++i) F[3 + i] = c0 * tau[i][0] + c1 * tau[i][1] + c2 * tau[i][2];
            if (d < 2) {
#pragma unroll
                for (int c = 0; c < 3; ++c) sF[3 * (d < 2 ? d : 0) + c][t] = V2{F[2 * c], F[2 * c + 1]};
            } else {
#pragma unroll
                for (int n = 0; n < Q; ++n) {
                    const T Dk = (T)col_D<P>(D, k, n);  // transposed: l_n'(xi_k)
#pragma unroll
                    for (int f = 0; f < 6; ++f) {
                        W[n][f] += Dk * F[f];
                        // added now: sunk to its use, every F would stay live
                        asm volatile("" : "+v"(W[n][f]));
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (k + 1 < Q) {
            gk = col_geo<P, false>(a.geo, b, k + 1, tc);
        } else {
            col_list<P>(pl.unode + u0, U, wn);
#pragma unroll
            for (int n = 0; n < Q; ++n) li[n] = pl.lidx[((int64_t)b * Q + n) * LANES + tc];
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        V2 f0[LA], f1[LA], f2[LA];
        auto read_flux = [&](int s) {
            const int m = s < Q ? sI + s : sJ + (s - Q) * EPB * Q, c = s < Q ? 0 : 3;
            f0[s % LA] = sF[c][m];
            f1[s % LA] = sF[c + 1][m];
            f2[s % LA] = sF[c + 2][m];
            Dv[s % LA] = s < Q ? sD[s * Q + I] : sD[(s - Q) * Q + J];  // transposed: l_I'(xi_n)
        };
#pragma unroll
        for (int s = 0; s < LA; ++s) read_flux(s);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2 * Q; ++s) {
            const int n = s % LA;
            W[k][0] += Dv[n] * f0[n].x;
            W[k][1] += Dv[n] * f0[n].y;
            W[k][2] += Dv[n] * f1[n].x;
            W[k][3] += Dv[n] * f1[n].y;
            W[k][4] += Dv[n] * f2[n].x;
            W[k][5] += Dv[n] * f2[n].y;
#pragma unroll
            for (int f = 0; f < 6; ++f) asm volatile("" : "+v"(W[k][f]));
            if (s + LA < 2 * Q) read_flux(s + LA);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const double v[5] = {(double)(nu[k] * W[k][0]), (double)W[k][3], (double)W[k][4], (double)W[k][5],
                             (double)(W[k][1] + kappa[k] * W[k][2])};
        col_add<P, COLORED>(sR, US, active, le, li[k], v);
    }
    __syncthreads();  // every node sum of the batch done
    col_write<P, COLORED>(sR, US, wn, U, a.Rmass, a.Rmom, a.Rener, np);
}

template <int P, class A, bool CLOSURE, typename TA>
static hipError_t launch_p(const A &a, const float *mlp, hipStream_t s)
{
    if (a.plan.nb <= 0) return hipSuccess;
    auto *kernel = a.plan.mode == kAtomic ? k_diffu_col<P, false, A, CLOSURE, TA> : k_diffu_col<P, true, A, CLOSURE, TA>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)a.plan.nb), dim3(ColShape<P>::NT), sizeof(double) * 5 * a.plan.ustride, s,
                       a, mlp);
    return hipGetLastError();
}

template <class A, bool CLOSURE, typename TA>
hipError_t launch_diffu_col(int porder, const A &a, const float *mlp, hipStream_t s)
{
    switch (porder) {
    case 1: return launch_p<1, A, CLOSURE, TA>(a, mlp, s);
    case 2: return launch_p<2, A, CLOSURE, TA>(a, mlp, s);
    case 3: return launch_p<3, A, CLOSURE, TA>(a, mlp, s);
    case 4: return launch_p<4, A, CLOSURE, TA>(a, mlp, s);
    case 5: return launch_p<5, A, CLOSURE, TA>(a, mlp, s);
    default: return hipErrorInvalidValue;
    }
}

template hipError_t launch_diffu_col<DiffuArgs<double, double>, false, double>(int, const DiffuArgs<double, double> &, const float *, hipStream_t);
template hipError_t launch_diffu_col<DiffuArgs<double, double>, true, double>(int, const DiffuArgs<double, double> &, const float *, hipStream_t);
template hipError_t launch_diffu_col<DiffuArgs<float, float>, false, double>(int, const DiffuArgs<float, float> &, const float *, hipStream_t);
template hipError_t launch_diffu_col<DiffuArgs<float, float>, false, float>(int, const DiffuArgs<float, float> &, const float *, hipStream_t);
template hipError_t launch_diffu_col<DiffuArgs<float, double>, false, double>(int, const DiffuArgs<float, double> &, const float *, hipStream_t);
template hipError_t launch_diffu_col<DiffuArgs<float, float, float>, false, double>(int, const DiffuArgs<float, float, float> &, const float *, hipStream_t);
template hipError_t launch_diffu_col<DiffuSplitArgs, false, double>(int, const DiffuSplitArgs &, const float *, hipStream_t);

}  // namespace msod
