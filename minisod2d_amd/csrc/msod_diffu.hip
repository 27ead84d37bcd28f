// Diffusive residual (counterpart of full_diffusion_ijk,
// src/kernels/sources/elem_diffu.f90:10-197); see msod_columns.h for the thread
// layout.
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
// with nu_e and kappa_e of the target node (the reference multiplies kappa_e
// inside the sum; same value, other rounding).  It also re-reads He, gpvol and
// the six flux vectors at every source of the target's lines (:141-193), where
// step 2 publishes one component per direction.
//
// Storage types TG (geometry, mu_e, mu_sgs) and TF (nodal fields), FP64
// arithmetic (msod_kernels.h); the FP32-arithmetic form is msod_diffu_nodes.hip.
// CLOSURE (FP64 storage): mu_sgs is not read but predicted by the learned
// closure (msod_mlp.h) from the velocity gradient before the stress is
// formed; its per-wave LDS scratch is the wave's own part of the flux buffer,
// free between the slice's first barrier and the fluxes.
#include <algorithm>
#include <type_traits>

#include "msod_columns.h"
#include "msod_mlp.h"
#include "msod_closure.h"

namespace msod {

template <int P, bool COLORED, class A, bool CLOSURE>
__global__ void __launch_bounds__(ColShape<P>::NT, 2) k_diffu_col(A a, const float *mlp)
{
    using S = ColShape<P>;
    using T = double;
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
    const uint32_t slot = xcd_runs(blockIdx.x, gridDim.x);
    const uint32_t b = pl.batches ? uniform(pl.batches)[slot] : slot;
    const uint32_t u0 = uniform(pl.uoff)[b], U = uniform(pl.uoff)[b + 1] - u0;
    const int64_t e0 = (int64_t)b * EPB;
    const bool active = t < LANES && e0 + le < a.nelem;
    const int ec = col_color<COLORED>(pl, active, e0 + le);

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
        col_add<COLORED>(sR, US, active, ec, pl.rounds, li[k], v);
    }
    __syncthreads();  // every node sum of the batch done
    col_write<P, COLORED>(sR, US, wn, U, a.Rmass, a.Rmom, a.Rener, np);
}

// Orders above kNarrowP: the same walk, whose columns (r, T, u and the six sums)
// take up to 198 VGPRs.  nu and kappa wait in LDS for the end, mu_fluid is
// gathered a slice ahead, and the gradients replace the line derivatives one
// field at a time.  They add to the outputs from the registers
// (col_merge, col_scatter).  Against one node per thread: 40^3 order 6 1.86 ->
// 1.21 ms (1.32 with the line sources read one ahead: spills); 32^3 order 8,
// with one wave per SIMD, 2.40 -> 1.88 (two waves and 80 spilled VGPRs: 2.61);
// order 5, against the kernel above with LDS sums, 64^3 3.08 -> 2.64.
template <int P>
constexpr int kWideWaves = P == 8 ? 1 : 2;  // per SIMD

template <int P, class A, bool CLOSURE>
__global__ void __launch_bounds__(ColShape<P>::NT, (kWideWaves<P>)) k_diffu_wide(A a, const float *mlp)
{
    using S = ColShape<P>;
    using T = double;
    using TG = typename A::G;
    constexpr int Q = S::Q, QQ = S::QQ, EPB = S::EPB, LANES = S::LANES, NT = S::NT;
    constexpr bool AHEAD = kWideWaves<P> == 1;  // read line sources one ahead of their use
    constexpr bool SHARED = sizeof(typename A::O) == 4;  // col_add_shared
    struct alignas(2 * sizeof(T)) V2 { T x, y; };
    __shared__ T sD[Q * Q];
    __shared__ V2 sP[2][NT];  // one slice: (r,T) (u0,u1)
    __shared__ T sU2[NT];     // and u2
    __shared__ TG sMu[2][NT];                              // its mu_e, mu_sgs
    __shared__ V2 sN[Q][NT];                               // nu, kappa of the thread's nodes
    __shared__ typename std::conditional<CLOSURE, MlpShared, char>::type smlp;
    // its fluxes along I (0..2) and J (3..5); with FP32 outputs, at
    // the end, the node sums [5][US]
    extern __shared__ __attribute__((aligned(16))) double sR[];
    V2(*sF)[NT] = reinterpret_cast<V2(*)[NT]>(sR);

    const Plan &pl = a.plan;
    const int US = pl.ustride, t = threadIdx.x;
    const ColThread<P> th(t);
    const int tc = th.tc, le = th.le, I = th.I, J = th.J;
    const int64_t np = a.npoin;
    const auto D = uniform(a.tab.D);
    const uint32_t slot = xcd_runs(blockIdx.x, gridDim.x);
    const uint32_t b = pl.batches ? uniform(pl.batches)[slot] : slot;
    const int64_t e0 = (int64_t)b * EPB;
    const bool active = t < LANES && e0 + le < a.nelem;
    const uint32_t *conn = pl.conn + (int64_t)b * Q * LANES + tc;

    // mu_e and mu_sgs change lanes in LDS (k_diffu_col)
    const int lem = tc % EPB, Im = tc / EPB % Q, Jm = tc / (EPB * Q);
    const int lm = line_ref<P>(Im) + Q * line_ref<P>(Jm), tm = t < LANES ? Im + Q * (lem + EPB * Jm) : t;
    const int64_t em = e0 + lem < a.nelem ? e0 + lem : a.nelem - 1;
    const bool has_sgs = !CLOSURE && a.mu_sgs;  // NULL: closure fallback
    const TG *mu_sgs = has_sgs ? a.mu_sgs : a.mu_e;
    TG mue, mus = (TG)0;
    typename A::F fmu;
    auto load_mu = [&](int k) {
        const int64_t ge = em + a.nelem * (int64_t)a.tab.l2g[lm + QQ * line_ref<P>(k)];
        mue = a.mu_e[ge];
        if constexpr (!CLOSURE) mus = mu_sgs[ge];
        fmu = a.mu_fluid[conn[k * LANES]];
    };
    const T Cp = (T)a.Cp, Pr = (T)a.Pr;
    T r[Q], Te[Q], u[Q][3], W[Q][6];
    {
        uint32_t gn[Q];
#pragma unroll
        for (int k = 0; k < Q; ++k) gn[k] = conn[k * LANES];
        typename A::F fr[Q], fT[Q];
        typename A::U fu[Q][3];
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            const int64_t g = gn[k];
            fr[k] = a.rho[g];
            fT[k] = a.Tem[g];
#pragma unroll
            for (int d = 0; d < 3; ++d) fu[k][d] = a.u[g + d * np];
        }
        load_mu(0);
        col_table<P>(a.tab.D, sD);
        if constexpr (CLOSURE) mlp_stage(smlp, mlp);
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            r[k] = (T)fr[k];
            Te[k] = (T)fT[k];
#pragma unroll
            for (int d = 0; d < 3; ++d) u[k][d] = (T)fu[k][d];
        }
    }
    GeoNode<TG> gk = col_geo<P, false>(a.geo, b, 0, tc);
    const int sI = tc - I, sJ = tc - J * EPB * Q;  // a line's source n: sI + n, sJ + n*EPB*Q

    col_slices<Q>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = kc();
        // the previous slice's values were read before its second barrier
        sP[0][t] = V2{r[k], Te[k]};
        sP[1][t] = V2{u[k][0], u[k][1]};
        sU2[t] = u[k][2];
        sMu[0][tm] = mue;
        sMu[1][tm] = mus;
        const T muf = (T)fmu;
        if constexpr (k + 1 < Q) load_mu(k + 1);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        // line derivatives x[d] of rho, T, u; the slice's geometry is still in flight
        T x[3][5];
#pragma unroll
        for (int f = 0; f < 5; ++f) x[0][f] = x[1][f] = x[2][f] = 0;
        struct Src { V2 a, b; T c, D; };
        auto read_source = [&](int s) {
            const int m = s < Q ? sI + s : sJ + (s - Q) * EPB * Q;
            return Src{sP[0][m], sP[1][m], sU2[m], s < Q ? sD[I * Q + s] : sD[J * Q + s - Q]};
        };
        Src cur = read_source(0), nxt = cur;
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
            const int d = s < Q ? 0 : 1;
            if (AHEAD && s + 1 < 2 * Q) nxt = read_source(s + 1);
            if (!AHEAD && s > 0) cur = read_source(s);
            x[d][0] += cur.D * cur.a.x;
            x[d][1] += cur.D * cur.a.y;
            x[d][2] += cur.D * cur.b.x;
            x[d][3] += cur.D * cur.b.y;
            x[d][4] += cur.D * cur.c;
            asm volatile("" : "+v"(x[d][0]), "+v"(x[d][1]), "+v"(x[d][2]), "+v"(x[d][3]), "+v"(x[d][4]));
            __builtin_amdgcn_sched_barrier(0);
            if (AHEAD) cur = nxt;
        }
        // x[.][f] becomes the gradient: grad rho, grad T, G[c][i] = x[i][2 + c]
#pragma unroll
        for (int f = 0; f < 5; ++f) {
            T g[3];
#pragma unroll
            for (int i = 0; i < 3; ++i)
                g[i] = (T)gk.he(i) * x[0][f] + (T)gk.he(3 + i) * x[1][f] + (T)gk.he(6 + i) * x[2][f];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                x[i][f] = g[i];
                asm volatile("" : "+v"(x[i][f]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const T me = (T)sMu[0][tc];
        T ms = has_sgs ? (T)sMu[1][tc] : (T)0;
        if constexpr (CLOSURE) {
            float f[kMlpIn];
            T hinv[3][3], G[3][3];
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    hinv[i][d] = (T)gk.he(i + 3 * d);
                    G[i][d] = x[d][2 + i];
                }
            mlp_features<T>(G, r[k], u[k], hinv, f);
            // idle lanes hold a real element node (finite features)
            const float z3 =
                mlp_forward_z3<NT * (int)sizeof(V2) / 2>(smlp, f, reinterpret_cast<short *>(&sF[0][t & ~63]));
            ms = (T)(smlp.scale * softplusf_(z3));
        }
        sN[k][t] = V2{(T)a.c_rho * me / r[k], muf * Cp / Pr + (T)a.c_ener * me * Cp / Pr + Cp * r[k] * ms / (T)0.9};
        const T mu_f = muf + r[k] * ms, mu_t = mu_f + me;
        const T lam = mu_f * (T)(2.0 / 3.0) * (x[0][2] + x[1][3] + x[2][4]);
        // tau (symmetric): xx, yy, zz, xy, xz, yz; tau.u
        T tau[6] = {mu_t * (x[0][2] + x[0][2]), mu_t * (x[1][3] + x[1][3]), mu_t * (x[2][4] + x[2][4]),
                    mu_t * (x[1][2] + x[0][3]), mu_t * (x[2][2] + x[0][4]), mu_t * (x[2][3] + x[1][4])};
        constexpr int at[3][3] = {{0, 3, 4}, {3, 1, 5}, {4, 5, 2}};
        T tauU[3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
            tauU[i] = tau[at[i][0]] * u[k][0] + tau[at[i][1]] * u[k][1] + tau[at[i][2]] * u[k][2] - lam * u[k][i];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            tau[i] -= lam;
            asm volatile("" : "+v"(tau[i]), "+v"(tau[3 + i]), "+v"(tauU[i]));
        }
        __builtin_amdgcn_sched_barrier(0);
        const T gv = (T)gk.gvol();
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const T c0 = gv * (T)gk.he(3 * d), c1 = gv * (T)gk.he(3 * d + 1), c2 = gv * (T)gk.he(3 * d + 2);
            T F[6];
            F[0] = c0 * x[0][0] + c1 * x[1][0] + c2 * x[2][0];
            F[1] = c0 * tauU[0] + c1 * tauU[1] + c2 * tauU[2];
            F[2] = c0 * x[0][1] + c1 * x[1][1] + c2 * x[2][1];
#pragma unroll
            for (int i = 0; i < 3; ++i) F[3 + i] = c0 * tau[at[i][0]] + c1 * tau[at[i][1]] + c2 * tau[at[i][2]];
            if (d < 2) {
#pragma unroll
                for (int c = 0; c < 3; ++c) sF[3 * (d < 2 ? d : 0) + c][t] = V2{F[2 * c], F[2 * c + 1]};
            } else {
#pragma unroll
                for (int n = 0; n < Q; ++n) {
                    const T Dk = (T)col_D<P>(D, k, n);  // transposed: l_n'(xi_k)
#pragma unroll
                    for (int f = 0; f < 6; ++f) {
                        if constexpr (k == 0) W[n][f] = Dk * F[f];
                        else W[n][f] += Dk * F[f];
                        // added now: sunk to its use, every F would stay live
                        asm volatile("" : "+v"(W[n][f]));
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (k + 1 < Q) gk = col_geo<P, false>(a.geo, b, k + 1, tc);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        struct Flux { V2 a, b, c; T D; };
        auto read_flux = [&](int s) {
            const int m = s < Q ? sI + s : sJ + (s - Q) * EPB * Q, c = s < Q ? 0 : 3;
            // transposed: l_I'(xi_n)
            return Flux{sF[c][m], sF[c + 1][m], sF[c + 2][m], s < Q ? sD[s * Q + I] : sD[(s - Q) * Q + J]};
        };
        Flux fc = read_flux(0), fn = fc;
#pragma unroll
        for (int s = 0; s < 2 * Q; ++s) {
            if (AHEAD && s + 1 < 2 * Q) fn = read_flux(s + 1);
            if (!AHEAD && s > 0) fc = read_flux(s);
            W[k][0] += fc.D * fc.a.x;
            W[k][1] += fc.D * fc.a.y;
            W[k][2] += fc.D * fc.b.x;
            W[k][3] += fc.D * fc.b.y;
            W[k][4] += fc.D * fc.c.x;
            W[k][5] += fc.D * fc.c.y;
#pragma unroll
            for (int f = 0; f < 6; ++f) asm volatile("" : "+v"(W[k][f]));
            __builtin_amdgcn_sched_barrier(0);
            if (AHEAD) fc = fn;
        }
    });
    if constexpr (SHARED) {
        __syncthreads();  // the last slice's fluxes are read
        for (int i = t; i < 5 * US; i += NT) sR[i] = 0.0;
        __syncthreads();
    }
    uint32_t at[Q], li[Q];
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        at[k] = conn[k * LANES];
        li[k] = SHARED ? (uint32_t)pl.lidx[((int64_t)b * Q + k) * LANES + tc] : 0u;
    }
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const V2 c = sN[k][t];
        double v[5] = {(double)(c.x * W[k][0]), (double)W[k][3], (double)W[k][4], (double)W[k][5],
                       (double)(W[k][1] + c.y * W[k][2])};
        if constexpr (SHARED) {
            if (col_merge<P>(at[k], I, le, active && e0 + le + 1 < a.nelem, v) && active)
                col_add_shared(sR, US, li[k], at[k], v, a.Rmass, a.Rmom, a.Rener, np);
        } else if (col_merge<P>(at[k], I, le, active && e0 + le + 1 < a.nelem, v) && active)
            col_scatter(at[k], v, a.Rmass, a.Rmom, a.Rener, np);
    }
    if constexpr (SHARED) {
        __syncthreads();
        col_write_shared(pl, b, sR, NT, a.Rmass, a.Rmom, a.Rener, np);
    }
}

// Order 7: a column is shared by two threads (t and its mate HL threads on, in
// other waves), four nodes each: k_diffu_wide spills 48 to 83 registers there
// and takes 4.4-4.7 ms at 48^3 (3.7 with one wave per SIMD and no spills).
// Derivatives along K take the mate's half of the column through LDS once;
// each slice's K fluxes go to the own nodes and, through LDS, to the mate's.  E2
// elements of a batch per workgroup.  48^3: 3.09
// ms, one node per thread 3.49; with all four elements in a workgroup, alone on
// its CU, 3.56.
template <int P, int E2, class A, bool CLOSURE>
__global__ void __launch_bounds__(2 * E2 * ColShape<P>::QQ, 2) k_diffu_split(A a, const float *mlp)
{
    using S = ColShape<P>;
    using T = double;
    using TG = typename A::G;
    constexpr int Q = S::Q, QQ = S::QQ, EPB = S::EPB, LANES = S::LANES;
    constexpr int H = Q / 2, HL = E2 * QQ, NT = 2 * HL, PARTS = EPB / E2;
    static_assert(Q % 2 == 0 && HL % 64 == 0 && LANES == EPB * QQ, "whole waves per half");
    constexpr bool SHARED = sizeof(typename A::O) == 4;  // col_add_shared
    struct alignas(2 * sizeof(T)) V2 { T x, y; };
    __shared__ T sD[Q * Q];
    __shared__ V2 sP[2][NT];  // one slice: (r,T) (u0,u1)
    __shared__ T sU2[NT];     // and u2
    __shared__ TG sMu[2][NT];                              // its mu_e, mu_sgs
    __shared__ typename std::conditional<CLOSURE, MlpShared, char>::type smlp;
    // its fluxes along I (0..2), J (3..5) and K (6..8); at the start the columns'
    // values; with FP32 outputs, at the end, the node sums [5][US]
    extern __shared__ __attribute__((aligned(16))) double sR[];
    V2(*sF)[NT] = reinterpret_cast<V2(*)[NT]>(sR);

    const Plan &pl = a.plan;
    const int US = pl.ustride, t = threadIdx.x;
    const int half = __builtin_amdgcn_readfirstlane(t / HL), tl = t - half * HL, mate = half ? t - HL : t + HL;
    const int I = tl % Q, le = tl / Q % E2, J = tl / (Q * E2);
    const int64_t np = a.npoin;
    const auto D = uniform(a.tab.D);
    const uint32_t slot = xcd_runs(blockIdx.x, gridDim.x), bs = slot / PARTS, part = slot % PARTS;
    const uint32_t b = pl.batches ? uniform(pl.batches)[bs] : bs;
    const int64_t e0 = (int64_t)b * EPB + part * E2;
    const bool active = e0 + le < a.nelem;
    const int tc = I + Q * ((int)part * E2 + le + EPB * J), k0 = half * H;
    const uint32_t *conn = pl.conn + ((int64_t)b * Q + k0) * LANES + tc;
    // line_ref of slice j of half h (j a compile-time constant)
    auto ref = [](int h, int j) { return h ? (j == H - 1 ? 1 : H + j + 1) : (j == 0 ? 0 : j + 1); };

    // mu_e and mu_sgs change lanes in LDS (k_diffu_col)
    const int lem = tl % E2, Im = tl / E2 % Q, Jm = tl / (E2 * Q);
    const int lm = line_ref<P>(Im) + Q * line_ref<P>(Jm), tm = half * HL + Im + Q * (lem + E2 * Jm);
    const int64_t em = e0 + lem < a.nelem ? e0 + lem : a.nelem - 1;
    const bool has_sgs = !CLOSURE && a.mu_sgs;  // NULL: closure fallback
    const TG *mu_sgs = has_sgs ? a.mu_sgs : a.mu_e;
    TG mue, mus = (TG)0;
    typename A::F fmu;
    auto load_mu = [&](int k) {
        const int64_t ge = em + a.nelem * (int64_t)a.tab.l2g[lm + QQ * ref(half, k)];
        mue = a.mu_e[ge];
        if constexpr (!CLOSURE) mus = mu_sgs[ge];
        fmu = a.mu_fluid[conn[k * LANES]];
    };
    const T Cp = (T)a.Cp, Pr = (T)a.Pr;
    T r[H], Te[H], u[H][3], dz[H][5], W[H][6], nu[H], kappa[H];
    {
        uint32_t gn[H];
#pragma unroll
        for (int k = 0; k < H; ++k) gn[k] = conn[k * LANES];
        typename A::F fr[H], fT[H];
        typename A::U fu[H][3];
#pragma unroll
        for (int k = 0; k < H; ++k) {
            const int64_t g = gn[k];
            fr[k] = a.rho[g];
            fT[k] = a.Tem[g];
#pragma unroll
            for (int d = 0; d < 3; ++d) fu[k][d] = a.u[g + d * np];
        }
        load_mu(0);
        col_table<P>(a.tab.D, sD);
        if constexpr (CLOSURE) mlp_stage(smlp, mlp);
#pragma unroll
        for (int k = 0; k < H; ++k) {
            r[k] = (T)fr[k];
            Te[k] = (T)fT[k];
#pragma unroll
            for (int d = 0; d < 3; ++d) u[k][d] = (T)fu[k][d];
        }
    }
    GeoNode<TG> gk = col_geo<P, false>(a.geo, b, k0, tc);
    // derivatives along K: the mate's half of the column comes through LDS, two
    // fields at a time
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        auto field = [&](int k, int f) -> T { return f == 0 ? r[k] : (f == 1 ? Te[k] : u[k][f - 2]); };
        const int f0 = 2 * c, f1 = c < 2 ? 2 * c + 1 : f0;
        V2(*buf)[NT] = sF + (c == 1 ? H : 0);
        if (c == 2) __syncthreads();  // the first buffer is read
#pragma unroll
        for (int k = 0; k < H; ++k) buf[k][t] = V2{field(k, f0), field(k, f1)};
        __syncthreads();
#pragma unroll
        for (int j = 0; j < H; ++j) dz[j][f0] = dz[j][f1] = 0;
#pragma unroll
        for (int n = 0; n < H; ++n) {
            const V2 o = buf[n][mate];
#pragma unroll
            for (int j = 0; j < H; ++j) {
                const T Do = (T)D[ref(half, j) * Q + ref(half, n)], Dm = (T)D[ref(half, j) * Q + ref(1 - half, n)];
                dz[j][f0] += Do * field(n, f0) + Dm * o.x;
                if (c < 2) dz[j][f1] += Do * field(n, f1) + Dm * o.y;
            }
        }
#pragma unroll
        for (int j = 0; j < H; ++j) asm volatile("" : "+v"(dz[j][f0]), "+v"(dz[j][f1]));
        __builtin_amdgcn_sched_barrier(0);
    }
    // a line's source n: sI + n, sJ + n*E2*Q
    const int sI = t - I, sJ = t - J * E2 * Q;

    col_slices<H>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = kc();
        // the previous slice's values were read before its second barrier
        sP[0][t] = V2{r[k], Te[k]};
        sP[1][t] = V2{u[k][0], u[k][1]};
        sU2[t] = u[k][2];
        sMu[0][tm] = mue;
        sMu[1][tm] = mus;
        const T muf = (T)fmu;
        if constexpr (k + 1 < H) load_mu(k + 1);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        // line derivatives x[d] of rho, T, u; the slice's geometry is still in flight
        T x[3][5];
#pragma unroll
        for (int f = 0; f < 5; ++f) {
            x[0][f] = x[1][f] = 0;
            x[2][f] = dz[k][f];
        }
        struct Src { V2 a, b; T c, D; };
        auto read_source = [&](int s) {
            const int m = s < Q ? sI + s : sJ + (s - Q) * E2 * Q;
            return Src{sP[0][m], sP[1][m], sU2[m], s < Q ? sD[I * Q + s] : sD[J * Q + s - Q]};
        };
        Src cur = read_source(0), nxt = cur;
#pragma unroll
        for (int s = 0; s < 2 * Q; ++s) {
            const int d = s < Q ? 0 : 1;
            if (s + 1 < 2 * Q) nxt = read_source(s + 1);
            x[d][0] += cur.D * cur.a.x;
            x[d][1] += cur.D * cur.a.y;
            x[d][2] += cur.D * cur.b.x;
            x[d][3] += cur.D * cur.b.y;
            x[d][4] += cur.D * cur.c;
            asm volatile("" : "+v"(x[d][0]), "+v"(x[d][1]), "+v"(x[d][2]), "+v"(x[d][3]), "+v"(x[d][4]));
            __builtin_amdgcn_sched_barrier(0);
            cur = nxt;
        }
        // x[.][f] becomes the gradient: grad rho, grad T, G[c][i] = x[i][2 + c]
#pragma unroll
        for (int f = 0; f < 5; ++f) {
            T g[3];
#pragma unroll
            for (int i = 0; i < 3; ++i)
                g[i] = (T)gk.he(i) * x[0][f] + (T)gk.he(3 + i) * x[1][f] + (T)gk.he(6 + i) * x[2][f];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                x[i][f] = g[i];
                asm volatile("" : "+v"(x[i][f]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const T me = (T)sMu[0][t];
        T ms = has_sgs ? (T)sMu[1][t] : (T)0;
        if constexpr (CLOSURE) {
            float f[kMlpIn];
            T hinv[3][3], G[3][3];
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    hinv[i][d] = (T)gk.he(i + 3 * d);
                    G[i][d] = x[d][2 + i];
                }
            mlp_features<T>(G, r[k], u[k], hinv, f);
            // idle lanes hold a real element node (finite features)
            const float z3 =
                mlp_forward_z3<NT * (int)sizeof(V2) / 2>(smlp, f, reinterpret_cast<short *>(&sF[0][t & ~63]));
            ms = (T)(smlp.scale * softplusf_(z3));
        }
        nu[k] = (T)a.c_rho * me / r[k];
        kappa[k] = muf * Cp / Pr + (T)a.c_ener * me * Cp / Pr + Cp * r[k] * ms / (T)0.9;
        asm volatile("" : "+v"(nu[k]), "+v"(kappa[k]));
        const T mu_f = muf + r[k] * ms, mu_t = mu_f + me;
        const T lam = mu_f * (T)(2.0 / 3.0) * (x[0][2] + x[1][3] + x[2][4]);
        // tau (symmetric): xx, yy, zz, xy, xz, yz; tau.u
        T tau[6] = {mu_t * (x[0][2] + x[0][2]), mu_t * (x[1][3] + x[1][3]), mu_t * (x[2][4] + x[2][4]),
                    mu_t * (x[1][2] + x[0][3]), mu_t * (x[2][2] + x[0][4]), mu_t * (x[2][3] + x[1][4])};
        constexpr int at[3][3] = {{0, 3, 4}, {3, 1, 5}, {4, 5, 2}};
        T tauU[3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
            tauU[i] = tau[at[i][0]] * u[k][0] + tau[at[i][1]] * u[k][1] + tau[at[i][2]] * u[k][2] - lam * u[k][i];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            tau[i] -= lam;
            asm volatile("" : "+v"(tau[i]), "+v"(tau[3 + i]), "+v"(tauU[i]));
        }
        __builtin_amdgcn_sched_barrier(0);
        const T gv = (T)gk.gvol();
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const T c0 = gv * (T)gk.he(3 * d), c1 = gv * (T)gk.he(3 * d + 1), c2 = gv * (T)gk.he(3 * d + 2);
            T F[6];
            F[0] = c0 * x[0][0] + c1 * x[1][0] + c2 * x[2][0];
            F[1] = c0 * tauU[0] + c1 * tauU[1] + c2 * tauU[2];
            F[2] = c0 * x[0][1] + c1 * x[1][1] + c2 * x[2][1];
#pragma unroll
            for (int i = 0; i < 3; ++i) F[3 + i] = c0 * tau[at[i][0]] + c1 * tau[at[i][1]] + c2 * tau[at[i][2]];
#pragma unroll
            for (int c = 0; c < 3; ++c) sF[3 * d + c][t] = V2{F[2 * c], F[2 * c + 1]};
            if (d == 2) {
#pragma unroll
                for (int n = 0; n < H; ++n) {
                    const T Dk = (T)D[ref(half, k) * Q + ref(half, n)];  // transposed: l_n'(xi_k)
#pragma unroll
                    for (int f = 0; f < 6; ++f) {
                        if constexpr (k == 0) W[n][f] = Dk * F[f];
                        else W[n][f] += Dk * F[f];
                        // added now: sunk to its use, every F would stay live
                        asm volatile("" : "+v"(W[n][f]));
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (k + 1 < H) gk = col_geo<P, false>(a.geo, b, k0 + k + 1, tc);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        struct Flux { V2 a, b, c; T D; };
        auto read_flux = [&](int s) {
            const int m = s < Q ? sI + s : sJ + (s - Q) * E2 * Q, c = s < Q ? 0 : 3;
            // transposed: l_I'(xi_n)
            return Flux{sF[c][m], sF[c + 1][m], sF[c + 2][m], s < Q ? sD[s * Q + I] : sD[(s - Q) * Q + J]};
        };
        Flux fc = read_flux(0), fn = fc;
#pragma unroll
        for (int s = 0; s < 2 * Q; ++s) {
            if (s + 1 < 2 * Q) fn = read_flux(s + 1);
            W[k][0] += fc.D * fc.a.x;
            W[k][1] += fc.D * fc.a.y;
            W[k][2] += fc.D * fc.b.x;
            W[k][3] += fc.D * fc.b.y;
            W[k][4] += fc.D * fc.c.x;
            W[k][5] += fc.D * fc.c.y;
#pragma unroll
            for (int f = 0; f < 6; ++f) asm volatile("" : "+v"(W[k][f]));
            __builtin_amdgcn_sched_barrier(0);
            fc = fn;
        }
        // the mate's slice
        const V2 m0 = sF[6][mate], m1 = sF[7][mate], m2 = sF[8][mate];
#pragma unroll
        for (int n = 0; n < H; ++n) {
            const T Dk = (T)D[ref(1 - half, k) * Q + ref(half, n)];
            W[n][0] += Dk * m0.x;
            W[n][1] += Dk * m0.y;
            W[n][2] += Dk * m1.x;
            W[n][3] += Dk * m1.y;
            W[n][4] += Dk * m2.x;
            W[n][5] += Dk * m2.y;
#pragma unroll
            for (int f = 0; f < 6; ++f) asm volatile("" : "+v"(W[n][f]));
        }
        __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (SHARED) {
        __syncthreads();  // the last slice's fluxes are read
        for (int i = t; i < 5 * US; i += NT) sR[i] = 0.0;
        __syncthreads();
    }
    uint32_t at[H], li[H];
#pragma unroll
    for (int k = 0; k < H; ++k) {
        at[k] = conn[k * LANES];
        li[k] = SHARED ? (uint32_t)pl.lidx[((int64_t)b * Q + k0 + k) * LANES + tc] : 0u;
    }
#pragma unroll
    for (int k = 0; k < H; ++k) {
        double v[5] = {(double)(nu[k] * W[k][0]), (double)W[k][3], (double)W[k][4], (double)W[k][5],
                       (double)(W[k][1] + kappa[k] * W[k][2])};
        if constexpr (SHARED) {
            if (col_merge<P, E2>(at[k], I, le, active && e0 + le + 1 < a.nelem, v) && active)
                col_add_shared(sR, US, li[k], at[k], v, a.Rmass, a.Rmom, a.Rener, np);
        } else if (col_merge<P, E2>(at[k], I, le, active && e0 + le + 1 < a.nelem, v) && active)
            col_scatter(at[k], v, a.Rmass, a.Rmom, a.Rener, np);
    }
    if constexpr (SHARED) {
        __syncthreads();
        col_write_shared(pl, b, sR, NT, a.Rmass, a.Rmom, a.Rener, np);
    }
}

template <int P, class A, bool CLOSURE>
static hipError_t launch_p(const A &a, const float *mlp, hipStream_t s)
{
    if (a.plan.nb <= 0) return hipSuccess;
    const bool atomic = a.plan.mode == kAtomic;
    const bool registers = P > kNarrowP && atomic && sizeof(typename A::O) == 8;
    const size_t sums = registers ? 0 : sizeof(double) * 5 * a.plan.ustride, fluxes = sizeof(double) * 12 * ColShape<P>::NT;
    const dim3 grid((unsigned)a.plan.nb), block(ColShape<P>::NT);
    if constexpr (P > kNarrowP)
        if (!atomic) return hipErrorInvalidValue;  // one node per thread there (nodes_for_colors)
    if constexpr (CLOSURE && (P == 4 || P == 5 || P == 8)) {
        return hipErrorInvalidValue;  // and there (nodes_for_atomics)
    } else if constexpr (P == 7) {
        constexpr int E2 = 2, EPB = ColShape<P>::EPB, QQ = ColShape<P>::QQ;
        const size_t part = sizeof(double) * 2 * 9 * 2 * QQ;  // fluxes per element
        hipLaunchKernelGGL((k_diffu_split<P, E2, A, CLOSURE>), dim3((unsigned)(a.plan.nb * (EPB / E2))), dim3(2 * E2 * QQ),
                           std::max(E2 * part, sums), s, a, mlp);
    } else if constexpr (P > kNarrowP) {
        hipLaunchKernelGGL((k_diffu_wide<P, A, CLOSURE>), grid, block, std::max(fluxes, sums), s, a, mlp);
    } else if constexpr (P == 4 && sizeof(typename A::O) == 4) {
        if (!atomic) return hipErrorInvalidValue;  // one node per thread there (nodes_for_colors)
        hipLaunchKernelGGL((k_diffu_col<P, false, A, CLOSURE>), grid, block, sums, s, a, mlp);
    } else {
        hipLaunchKernelGGL((atomic ? k_diffu_col<P, false, A, CLOSURE> : k_diffu_col<P, true, A, CLOSURE>), grid,
                           block, sums, s, a, mlp);
    }
    return hipGetLastError();
}

template <class A, bool CLOSURE>
static hipError_t launch_order(int porder, const A &a, const float *mlp, hipStream_t s)
{
    switch (porder) {
    case 1: return launch_p<1, A, CLOSURE>(a, mlp, s);
    case 2: return launch_p<2, A, CLOSURE>(a, mlp, s);
    case 3: return launch_p<3, A, CLOSURE>(a, mlp, s);
    case 4: return launch_p<4, A, CLOSURE>(a, mlp, s);
    case 5: return launch_p<5, A, CLOSURE>(a, mlp, s);
    case 6: return launch_p<6, A, CLOSURE>(a, mlp, s);
    case 7: return launch_p<7, A, CLOSURE>(a, mlp, s);
    case 8: return launch_p<8, A, CLOSURE>(a, mlp, s);
    default: return hipErrorInvalidValue;
    }
}

template <class A>
hipError_t launch_diffu(int porder, const A &a, hipStream_t s)
{
    return launch_order<A, false>(porder, a, nullptr, s);
}

hipError_t launch_diffu_closure(int porder, const DiffuArgs<double, double> &a, const float *mlp, hipStream_t s)
{
    return launch_order<DiffuArgs<double, double>, true>(porder, a, mlp, s);
}

template hipError_t launch_diffu(int, const DiffuArgs<double, double> &, hipStream_t);
template hipError_t launch_diffu(int, const DiffuArgs<float, float> &, hipStream_t);
template hipError_t launch_diffu(int, const DiffuArgs<float, double> &, hipStream_t);
template hipError_t launch_diffu(int, const DiffuArgs<float, float, float> &, hipStream_t);
template hipError_t launch_diffu(int, const DiffuSplitArgs &, hipStream_t);

}  // namespace msod
