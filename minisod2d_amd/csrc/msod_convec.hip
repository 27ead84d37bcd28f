// Convective residual (counterpart of full_convec_ijk,
// src/kernels/sources/elem_convec.f90:198-431, with the energy fluxes of
// full_convec_ijk_split, :674-832); see msod_columns.h for the thread layout.
//
// With He(:,d) of the TARGET node a folded into the source values,
//   U_n = sum_i He(i,d) u_i(n),  Q_n = sum_i He(i,d) q_i(n),
// every term of the split form is, over the three directions d and the
// sources n of a line (D = D[I_d(a)][n]),
//   S3 = sum D (Q_n + U_a r_n)          (div q + u.grad r)
//   S4 = sum D U_n                      (div u)
//   M_i = sum D [(U_n + U_a) q_i(n) + (r_a U_n + Q_a) u_i(n) + 4 He(i,d) p(n)]
//   X = sum D [(U_n + U_a) rH(n) + (r_a U_n + Q_a) H(n)]
//   Rmass = (S3 + r_a S4)/2,  Rmom_i = (M_i + u_i S3 + q_i S4)/4,
//   Rener = (X + H_a S3 + rH_a S4)/4
// with H = E + |u|^2/2 and rH = r H: the terms of elem_convec.f90:228-428 and
// :694-697, collected by the factors they share.  The result equals the
// reference's algebra exactly in real arithmetic; rounding differs at the
// 1e-16 level.
//
// Storage types TG (geometry) and TF (nodal fields), FP64 arithmetic
// (msod_kernels.h); the FP32-arithmetic form is msod_convec_nodes.hip.  Without a
// pressure array the pressure is recovered as p = (gamma-1)(E - rho|u|^2/2)
// from the stored state.
#include "msod_columns.h"

namespace msod {

// One direction's factors of the target node.
template <typename T>
struct ConvecDir { T h0, h1, h2, Ua, Qa, dp; };

// The sums of one target node; ra, u, q: its own values.
template <typename T>
struct ConvecSums {
    T S3 = 0, S4 = 0, X = 0, M[3] = {0, 0, 0};
    template <class G>
    __device__ __forceinline__ ConvecDir<T> direction(const G &g, int d, const T (&u)[3], const T (&q)[3]) const
    {
        const T h0 = (T)g.he(3 * d), h1 = (T)g.he(3 * d + 1), h2 = (T)g.he(3 * d + 2);
        return ConvecDir<T>{h0, h1, h2, h0 * u[0] + h1 * u[1] + h2 * u[2], h0 * q[0] + h1 * q[1] + h2 * q[2], (T)0};
    }
    __device__ __forceinline__ void source(ConvecDir<T> &x, T ra, T Dv, T rs, T ps, T Hs, T us0, T us1, T us2, T qs0, T qs1, T qs2)
    {
        const T Un = x.h0 * us0 + x.h1 * us1 + x.h2 * us2;
        const T Qn = x.h0 * qs0 + x.h1 * qs1 + x.h2 * qs2;
        S3 += Dv * (Qn + x.Ua * rs);
        S4 += Dv * Un;
        x.dp += Dv * ps;
        const T S1 = Dv * (Un + x.Ua), S2 = Dv * (ra * Un + x.Qa);
        M[0] += S1 * qs0 + S2 * us0;
        M[1] += S1 * qs1 + S2 * us1;
        M[2] += S1 * qs2 + S2 * us2;
        X += (S1 * rs + S2) * Hs;  // S1 rH + S2 H
        // summed here: left to the compiler the sums sink to the
        // end of the slice and every source's values stay live
        asm volatile("" : "+v"(S3), "+v"(S4), "+v"(x.dp), "+v"(M[0]), "+v"(M[1]), "+v"(M[2]), "+v"(X));
    }
    __device__ __forceinline__ void finish(const ConvecDir<T> &x)
    {
        const T dp4 = (T)4 * x.dp;
        M[0] += x.h0 * dp4;
        M[1] += x.h1 * dp4;
        M[2] += x.h2 * dp4;
        asm volatile("" : "+v"(M[0]), "+v"(M[1]), "+v"(M[2]));
    }
    __device__ __forceinline__ void values(T gv, T ra, T Ha, const T (&u)[3], const T (&q)[3], double (&v)[5]) const
    {
        v[0] = (double)(gv * ((T)0.5 * (S3 + ra * S4)));
#pragma unroll
        for (int i = 0; i < 3; ++i) v[1 + i] = (double)(gv * ((T)0.25 * (M[i] + u[i] * S3 + q[i] * S4)));
        v[4] = (double)(gv * ((T)0.25 * (X + Ha * S3 + ra * Ha * S4)));
    }
};

template <int P, bool COLORED, class A>
__global__ void __launch_bounds__(ColShape<P>::NT, 2) k_convec_col(A a)
{
    using S = ColShape<P>;
    using T = double;
    using TG = typename A::G;
    constexpr int Q = S::Q, EPB = S::EPB, LANES = S::LANES, NT = S::NT;
    struct alignas(2 * sizeof(T)) V2 { T x, y; };
    __shared__ T sD[Q * Q];
    __shared__ V2 sP[4][NT];  // one slice: (r,p) (u0,u1) (u2,q0) (q1,q2)
    __shared__ T sH[NT];      // and H
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
    const bool active = t < LANES && (int64_t)b * EPB + le < a.nelem;
    const int ec = col_color<COLORED>(pl, active, (int64_t)b * EPB + le);
    // FP32 state with FP64 outputs comes without a pressure array
    constexpr bool kRecover = sizeof(typename A::F) == 4 && sizeof(typename A::Pt) == 4 && sizeof(typename A::O) == 8;

    uint32_t gn[Q];
#pragma unroll
    for (int k = 0; k < Q; ++k) gn[k] = __builtin_nontemporal_load(&pl.conn[((int64_t)b * Q + k) * LANES + tc]);
    GeoNode<TG> geo[2];
    geo[0] = col_geo<P, true>(a.geo, b, 0, tc);
    typename A::F fr[Q], fE[Q], fq[Q][3];
    typename A::U fu[Q][3];
    typename A::Pt fp[Q];
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const int64_t g = gn[k];
        fr[k] = a.rho[g];
        fE[k] = a.E[g];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            fu[k][d] = a.u[g + d * np];
            fq[k][d] = a.q[g + d * np];
        }
        if constexpr (!kRecover) fp[k] = a.pr[g];
    }
    col_table<P>(a.tab.D, sD);
    for (int i = t; i < 5 * US; i += NT) sR[i] = 0.0;

    T r[Q], p[Q], H[Q], u[Q][3], q[Q][3];
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        r[k] = (T)fr[k];
        const T E = (T)fE[k];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            u[k][d] = (T)fu[k][d];
            q[k][d] = (T)fq[k][d];
        }
        const T ke = u[k][0] * u[k][0] * (T)0.5 + u[k][1] * u[k][1] * (T)0.5 + u[k][2] * u[k][2] * (T)0.5;
        if constexpr (kRecover)
            // p = (gamma-1)(E - rho|u|^2/2), in FP64 whatever T: the difference cancels
            p[k] = (T)(a.gamma_m1 * ((double)E - (double)r[k] * 0.5 *
                                                     ((double)u[k][0] * u[k][0] + (double)u[k][1] * u[k][1] +
                                                      (double)u[k][2] * u[k][2])));
        else
            p[k] = (T)fp[k];
        H[k] = E + ke;
    }
    uint32_t wn[S::UPT];
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const T ra = r[k], Ha = H[k];
        if (k > 0) __syncthreads();  // the previous slice is read
        sP[0][t] = V2{ra, p[k]};
        sP[1][t] = V2{u[k][0], u[k][1]};
        sP[2][t] = V2{u[k][2], q[k][0]};
        sP[3][t] = V2{q[k][1], q[k][2]};
        sH[t] = Ha;
        const uint32_t li = __builtin_nontemporal_load(&pl.lidx[((int64_t)b * Q + k) * LANES + tc]);
        if (k + 1 < Q)
            geo[(k + 1) & 1] = col_geo<P, true>(a.geo, b, k + 1, tc);
        else
            col_list<P>(pl.unode + u0, U, wn);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        const GeoNode<TG> &gk = geo[k & 1];
        ConvecSums<T> sum;
        // Steps 0..2Q-1: the sources along I, then J, from LDS; a source's
        // record is read while the one before it is used, and every other
        // step a source along K, which needs no LDS, is used as well, so that
        // the LDS reads spread over all of the slice's arithmetic.  The
        // scheduling barriers keep the order (and the registers).
        ConvecDir<T> dz = sum.direction(gk, 2, u[k], q[k]), dl = sum.direction(gk, 0, u[k], q[k]);
        const int sI = tc - I, sJ = tc - J * EPB * Q;
        auto slot = [&](int s) { return s < Q ? sI + s : sJ + (s - Q) * EPB * Q; };
        V2 c0 = sP[0][sI], c1 = sP[1][sI], c2 = sP[2][sI], c3 = sP[3][sI];
        T cH = sH[sI], cD = sD[I * Q];
#pragma unroll
        for (int s = 0; s < 2 * Q; ++s) {
            const int m = slot(s + 1 < 2 * Q ? s + 1 : s);
            const V2 n0 = sP[0][m], n1 = sP[1][m], n2 = sP[2][m], n3 = sP[3][m];
            const T nH = sH[m], nD = s + 1 < Q ? sD[I * Q + s + 1] : sD[J * Q + (s + 1 < 2 * Q ? s + 1 - Q : 0)];
            __builtin_amdgcn_sched_barrier(0);
            if (s % 2 == 0) {
                const int n = s / 2;
                sum.source(dz, ra, (T)col_D<P>(D, k, n), r[n], p[n], H[n], u[n][0], u[n][1], u[n][2], q[n][0], q[n][1], q[n][2]);
            }
            sum.source(dl, ra, cD, c0.x, c0.y, cH, c1.x, c1.y, c2.x, c2.y, c3.x, c3.y);
            if (s == Q - 1) {
                sum.finish(dl);
                dl = sum.direction(gk, 1, u[k], q[k]);
            }
            __builtin_amdgcn_sched_barrier(0);
            c0 = n0;
            c1 = n1;
            c2 = n2;
            c3 = n3;
            cH = nH;
            cD = nD;
        }
        sum.finish(dl);
        sum.finish(dz);
        double v[5];
        sum.values((T)gk.gvol(), ra, Ha, u[k], q[k], v);
        col_add<COLORED>(sR, US, active, ec, pl.rounds, li, v);
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // every node sum of the batch done
    col_write<P, COLORED>(sR, US, wn, U, a.Rmass, a.Rmom, a.Rener, np);
}

// Orders above kNarrowP: the same walk within 256 VGPRs, of which the column
// takes up to 162.  The directions follow one another (one set of factors live)
// and the geometry has one buffer, whose pairs are loaded anew for the next
// slice as soon as a direction is done with them.  The atomic mode adds to the
// outputs from the registers (col_merge, col_scatter).  Against one node per
// thread with everything read from LDS: 48^3 order 7 4.05 -> 2.56 ms, FP32
// split 3.21 -> 2.18; 40^3 order 6 1.96 -> 1.03; 32^3 order 8 1.96 -> 1.49; order 5,
// against the kernel above with LDS sums, 64^3 2.60 -> 2.38.  Of order 7's 2.56
// ms, outputs take about a third (2.0 ms of 3.07 without any, 2.4 with plain
// stores, before neighbours' nodes were merged); the rest is the FP64 work and
// LDS reads of two waves per SIMD.
template <int P, bool COLORED, class A>
__global__ void __launch_bounds__(ColShape<P>::NT, 2) k_convec_wide(A a)
{
    using S = ColShape<P>;
    using T = double;
    using TG = typename A::G;
    constexpr int Q = S::Q, EPB = S::EPB, LANES = S::LANES, NT = S::NT;
    constexpr bool SHARED = !COLORED && sizeof(typename A::O) == 4;  // col_add_shared
    struct alignas(2 * sizeof(T)) V2 { T x, y; };
    __shared__ T sD[Q * Q];
    __shared__ V2 sP[4][NT];  // one slice: (r,p) (u0,u1) (u2,q0) (q1,q2)
    __shared__ T sH[NT];      // and H
    extern __shared__ __attribute__((aligned(16))) double sR[];  // coloured mode, FP32 outputs: node sums [5][US]

    const Plan &pl = a.plan;
    const int US = pl.ustride, t = threadIdx.x;
    const ColThread<P> th(t);
    const int tc = th.tc, le = th.le, I = th.I, J = th.J;
    const int64_t np = a.npoin;
    const auto D = uniform(a.tab.D);
    const uint32_t slot = xcd_runs(blockIdx.x, gridDim.x);
    const uint32_t b = pl.batches ? uniform(pl.batches)[slot] : slot;
    const bool active = t < LANES && (int64_t)b * EPB + le < a.nelem;
    const int ec = col_color<COLORED>(pl, active, (int64_t)b * EPB + le);
    constexpr bool kRecover = sizeof(typename A::F) == 4 && sizeof(typename A::Pt) == 4 && sizeof(typename A::O) == 8;

    T r[Q], p[Q], H[Q], u[Q][3], q[Q][3];
    GeoNode<TG> geo;
    {
        uint32_t gn[Q];
#pragma unroll
        for (int k = 0; k < Q; ++k) gn[k] = pl.conn[((int64_t)b * Q + k) * LANES + tc];
        typename A::F fr[Q], fE[Q], fq[Q][3];
        typename A::U fu[Q][3];
        typename A::Pt fp[Q];
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            const int64_t g = gn[k];
            fr[k] = a.rho[g];
            fE[k] = a.E[g];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                fu[k][d] = a.u[g + d * np];
                fq[k][d] = a.q[g + d * np];
            }
            if constexpr (!kRecover) fp[k] = a.pr[g];
        }
        geo = col_geo<P, true>(a.geo, b, 0, tc);
        col_table<P>(a.tab.D, sD);
        if constexpr (COLORED || SHARED)
            for (int i = t; i < 5 * US; i += NT) sR[i] = 0.0;
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            r[k] = (T)fr[k];
            const T E = (T)fE[k];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                u[k][d] = (T)fu[k][d];
                q[k][d] = (T)fq[k][d];
            }
            const T ke = u[k][0] * u[k][0] * (T)0.5 + u[k][1] * u[k][1] * (T)0.5 + u[k][2] * u[k][2] * (T)0.5;
            if constexpr (kRecover)
                p[k] = (T)(a.gamma_m1 * ((double)E - (double)r[k] * 0.5 *
                                                         ((double)u[k][0] * u[k][0] + (double)u[k][1] * u[k][1] +
                                                          (double)u[k][2] * u[k][2])));
            else
                p[k] = (T)fp[k];
            H[k] = E + ke;
        }
    }
    // the next slice's place in the outputs: its node, or (coloured) its
    // position in the batch's list
    uint32_t at = COLORED ? pl.lidx[(int64_t)b * Q * LANES + tc] : pl.conn[(int64_t)b * Q * LANES + tc], li = 0;
    if constexpr (SHARED) li = pl.lidx[(int64_t)b * Q * LANES + tc];
    const int sI = tc - I, sJ = tc - J * EPB * Q;
    col_slices<Q>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = kc();
        const T ra = r[k], Ha = H[k];
        if (k > 0) __syncthreads();  // the previous slice is read
        sP[0][t] = V2{ra, p[k]};
        sP[1][t] = V2{u[k][0], u[k][1]};
        sP[2][t] = V2{u[k][2], q[k][0]};
        sP[3][t] = V2{q[k][1], q[k][2]};
        sH[t] = Ha;
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        ConvecSums<T> sum;
        auto next_geo = [&](int c) {
            if (k + 1 < Q) geo.v[c] = col_geo_pair<P, true>(a.geo, b, k + 1, tc, c);
        };
        // the sources along I, then J; each read one ahead of its use
        struct Rec { V2 a, b, c, d; T H, D; };
        auto read = [&](int m, const T *Dv) { return Rec{sP[0][m], sP[1][m], sP[2][m], sP[3][m], sH[m], *Dv}; };
        Rec ra0 = read(sI, sD + I * Q), rb0;
        ConvecDir<T> x = sum.direction(geo, 2, u[k], q[k]);
#pragma unroll
        for (int n = 0; n < Q; ++n) {
            sum.source(x, ra, (T)col_D<P>(D, k, n), r[n], p[n], H[n], u[n][0], u[n][1], u[n][2], q[n][0], q[n][1], q[n][2]);
            __builtin_amdgcn_sched_barrier(0);
        }
        sum.finish(x);
        T gv = (T)geo.gvol();
        asm volatile("" : "+v"(gv));
        next_geo(3);
        next_geo(4);
        auto use = [&](const Rec &c) {
            __builtin_amdgcn_sched_barrier(0);
            sum.source(x, ra, c.D, c.a.x, c.a.y, c.H, c.b.x, c.b.y, c.c.x, c.c.y, c.d.x, c.d.y);
            __builtin_amdgcn_sched_barrier(0);
        };
        // a line's q sources, the first of them in ra0; ends with the record at
        // `then` in ra0
        auto line = [&](int m, int step, const T *Dv, int then, const T *Dthen) {
            if constexpr (Q % 2) {
#pragma unroll
                for (int n = 0; n < Q - 1; n += 2) {
                    m += step;
                    rb0 = read(m, ++Dv);
                    use(ra0);
                    m += step;
                    ra0 = read(m, ++Dv);
                    use(rb0);
                }
                rb0 = read(then, Dthen);
                use(ra0);
                ra0 = rb0;
            } else {
#pragma unroll
                for (int n = 0; n < Q - 2; n += 2) {
                    m += step;
                    rb0 = read(m, ++Dv);
                    use(ra0);
                    m += step;
                    ra0 = read(m, ++Dv);
                    use(rb0);
                }
                rb0 = read(m + step, Dv + 1);
                use(ra0);
                ra0 = read(then, Dthen);
                use(rb0);
            }
        };
        x = sum.direction(geo, 0, u[k], q[k]);
        line(sI, 1, sD + I * Q, sJ, sD + J * Q);
        sum.finish(x);
        next_geo(0);
        x = sum.direction(geo, 1, u[k], q[k]);
        line(sJ, EPB * Q, sD + J * Q, sJ, sD + J * Q);
        sum.finish(x);
        next_geo(1);
        next_geo(2);
        double v[5];
        sum.values(gv, ra, Ha, u[k], q[k], v);
        const uint32_t here = at, li_here = li;
        if (k + 1 < Q) {
            const int64_t i = ((int64_t)b * Q + k + 1) * LANES + tc;
            at = COLORED ? pl.lidx[i] : pl.conn[i];
            if constexpr (SHARED) li = pl.lidx[i];
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (COLORED) {
            col_add<true>(sR, US, active, ec, pl.rounds, here, v);
        } else if constexpr (SHARED) {
            if (col_merge<P>(here, I, le, active && (int64_t)b * EPB + le + 1 < a.nelem, v) && active)
                col_add_shared(sR, US, li_here, here, v, a.Rmass, a.Rmom, a.Rener, np);
        } else if (col_merge<P>(here, I, le, active && (int64_t)b * EPB + le + 1 < a.nelem, v) && active)
            col_scatter(here, v, a.Rmass, a.Rmom, a.Rener, np);
        __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (COLORED) {
        const uint32_t u0 = uniform(pl.uoff)[b], U = uniform(pl.uoff)[b + 1] - u0;
        uint32_t wn[S::UPT];
        col_list<P>(pl.unode + u0, U, wn);
        __syncthreads();
        col_write<P, true>(sR, US, wn, U, a.Rmass, a.Rmom, a.Rener, np);
    }
    if constexpr (SHARED) {
        __syncthreads();
        col_write_shared(pl, b, sR, NT, a.Rmass, a.Rmom, a.Rener, np);
    }
}

template <int P, class A>
static hipError_t launch_p(const A &a, hipStream_t s)
{
    if (a.plan.nb <= 0) return hipSuccess;
    const bool atomic = a.plan.mode == kAtomic;
    const bool registers = P > kNarrowP && atomic && sizeof(typename A::O) == 8;
    const size_t sums = registers ? 0 : sizeof(double) * 5 * a.plan.ustride;
    if constexpr (P > kNarrowP) {
        if constexpr (P != 6)
            if (!atomic) return hipErrorInvalidValue;  // one node per thread there (nodes_for_colors)
        hipLaunchKernelGGL((atomic || P != 6 ? k_convec_wide<P, false, A> : k_convec_wide<P, P == 6, A>),
                           dim3((unsigned)a.plan.nb), dim3(ColShape<P>::NT), sums, s, a);
    } else
        hipLaunchKernelGGL((atomic ? k_convec_col<P, false, A> : k_convec_col<P, true, A>),
                           dim3((unsigned)a.plan.nb), dim3(ColShape<P>::NT), sums, s, a);
    return hipGetLastError();
}

template <class A>
hipError_t launch_convec(int porder, const A &a, hipStream_t s)
{
    switch (porder) {
    case 1: return launch_p<1, A>(a, s);
    case 2: return launch_p<2, A>(a, s);
    case 3: return launch_p<3, A>(a, s);
    case 4: return launch_p<4, A>(a, s);
    case 5: return launch_p<5, A>(a, s);
    case 6: return launch_p<6, A>(a, s);
    case 7: return launch_p<7, A>(a, s);
    case 8: return launch_p<8, A>(a, s);
    default: return hipErrorInvalidValue;
    }
}

template hipError_t launch_convec(int, const ConvecArgs<double, double> &, hipStream_t);
template hipError_t launch_convec(int, const ConvecArgs<float, float> &, hipStream_t);
template hipError_t launch_convec(int, const ConvecArgs<float, double> &, hipStream_t);
template hipError_t launch_convec(int, const ConvecArgs<float, float, float> &, hipStream_t);
template hipError_t launch_convec(int, const ConvecSplitArgs &, hipStream_t);

}  // namespace msod
