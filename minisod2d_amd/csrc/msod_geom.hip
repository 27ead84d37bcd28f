// Geometry kernel: He and gpvol of every element node from the node
// coordinates (counterpart of elem_jacobian, src/fem/sources/jacobian_oper.f90:7-136,
// which the reference driver runs on the device once per mesh,
// src/app/sources/main.f90:292-295).
//
//   Je(i,j) = sum_a dNgp(i,a,g) * coord(connec(e,a), j)
//   det     = Je11 Je22 Je33 + Je12 Je23 Je31 + Je13 Je21 Je32
//           - Je31 Je22 Je13 - Je32 Je23 Je11 - Je33 Je21 Je12
//   He      = cofactor(Je)^T / det,   gpvol = wgp(g) * det
//
// The sum over a runs over the nonzero entries of dNgp(i,:,g) only, in
// increasing a (the zero terms of the reference's dense dot_product add
// nothing); for a tensor-product hexahedron these are the q nodes on the
// grid line of g in direction i.
//
// What it has to move is 80 bytes written per element node (2.6 of 3.2 GB at
// 64^3, p=4); the chip fills memory at 6.7 TB/s and copies at 4.3.  One
// workgroup takes EC consecutive elements:
//   1. their connec into LDS, neighbouring lanes reading neighbouring
//      elements of one node: the layout (nelem,nnode) puts one element's
//      nodes 4*nelem bytes apart, so EC elements fill a 64-byte sector;
//   then, EB elements at a time, one thread per element node throughout:
//   2. the nodes' coordinates, loaded a step ahead, into LDS;
//   3. Je, det and He, gpvol stored from the thread, He into LDS;
//   4. He written back in 16-byte pieces as the contiguous block that it
//      forms in He(3,3,ngaus,nelem).
// A thread meets the same g in every step, so its 3*q weights and LDS
// offsets stay in registers; padding points at a node of zeros behind the
// element's.  Tables with more than q entries in a row (no tensor product)
// are read from memory in every step.  The stores are
// non-temporal: 836 us at 64^3, p=4 (3.8 TB/s) against 926.  Weights read in
// every step, 8-byte stores and gathers after the barrier took 1614 us; half
// as many elements a step 1069, twice as many 823, three times 984.
#include "msod_kernels.h"
#include "msod_geom.h"

namespace msod {

template <int P>
struct GeomShape {
    static constexpr int Q = P + 1;
    static constexpr int NN = Q * Q * Q;
    static constexpr int EB = NN <= 128 ? 256 / NN / 2 * 2 : 1;  // elements per step
    static constexpr int NT = (EB * NN + 63) / 64 * 64;
    // elements per workgroup: a whole number of steps, connec within 12 KB
    static constexpr int EC_RAW = 3072 / NN < 16 ? 3072 / NN : 16;
    static constexpr int EC = EC_RAW < EB ? EB : EC_RAW / EB * EB;
};

// REG: every row of the tables has at most q entries
template <int P, bool REG>
__global__ void __launch_bounds__(GeomShape<P>::NT) k_elem_jacobian(GeomArgs a)
{
    using S = GeomShape<P>;
    constexpr int Q = S::Q, NN = S::NN, EB = S::EB, EC = S::EC, NT = S::NT;
    typedef double pair_t __attribute__((ext_vector_type(2), aligned(8)));
    __shared__ int32_t sC[EC * NN];
    __shared__ double sX[EB * (NN + 1) * 3];
    __shared__ double sH[EB * NN * 9];
    const int t = threadIdx.x;
    const int64_t ec0 = (int64_t)xcd_range(blockIdx.x, gridDim.x) * EC;
    const int nec = (int)(a.nelem - ec0 < EC ? a.nelem - ec0 : EC);

    for (int i = t; i < EC * NN; i += NT) {
        const int eb = i % EC, n = i / EC;
        sC[eb * NN + n] = eb < nec ? a.connec[(ec0 + eb) + a.nelem * (int64_t)n] : 1;
    }
    for (int i = t; i < EB * 3; i += NT) sX[((i / 3 + 1) * (NN + 1) - 1) * 3 + i % 3] = 0.0;
    // the thread's node g of element eb of each step
    const int eb = t / NN, g = t - eb * NN;
    const bool mine = t < EB * NN;
    double w[3][REG ? Q : 1];
    int at[3][REG ? Q : 1];
    double wg = 0.0;
    if (mine) wg = a.wgp[g];
    if constexpr (REG) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int k = 0; k < Q; ++k) {
                const int row = (k * 3 + d) * NN + g;
                const bool in = mine && k < a.mz;
                w[d][k] = in ? a.nzw[row] : 0.0;
                at[d][k] = (eb * (NN + 1) + (in ? (int)a.nza[row] : NN)) * 3;
            }
    }
    unsigned bad_conn = 0, bad_det = 0;
    double x[3];
    auto load = [&](int c0) {
        const bool live = mine && c0 + eb < nec;
        int64_t ip = live ? (int64_t)sC[(c0 + eb) * NN + g] - 1 : 0;
        if (ip < 0 || ip >= a.npoin) {  // reported, read as node 1
            ++bad_conn;
            ip = 0;
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) x[j] = a.coord[ip + a.npoin * j];
    };
    __syncthreads();
    load(0);
    for (int c0 = 0; c0 < nec; c0 += EB) {
        const int64_t e0 = ec0 + c0;
        const int ne = nec - c0 < EB ? nec - c0 : EB;
        if (mine) {
#pragma unroll
            for (int j = 0; j < 3; ++j) sX[(eb * (NN + 1) + g) * 3 + j] = x[j];
        }
        __syncthreads();  // sX staged; the previous step's write-back is done with sH
        if (c0 + EB < nec) load(c0 + EB);
        if (mine) {
            double Je[3][3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                double s0 = 0.0, s1 = 0.0, s2 = 0.0;
                if constexpr (REG) {
#pragma unroll
                    for (int k = 0; k < Q; ++k) {
                        s0 += w[d][k] * sX[at[d][k]];
                        s1 += w[d][k] * sX[at[d][k] + 1];
                        s2 += w[d][k] * sX[at[d][k] + 2];
                    }
                } else {
                    for (int k = 0; k < a.mz; ++k) {
                        const int row = (k * 3 + d) * NN + g;
                        const double wk = a.nzw[row];
                        const double *xs = sX + (eb * (NN + 1) + (int)a.nza[row]) * 3;
                        s0 += wk * xs[0];
                        s1 += wk * xs[1];
                        s2 += wk * xs[2];
                    }
                }
                Je[d][0] = s0;
                Je[d][1] = s1;
                Je[d][2] = s2;
            }
            const double det = Je[0][0] * Je[1][1] * Je[2][2] + Je[0][1] * Je[1][2] * Je[2][0] +
                               Je[0][2] * Je[1][0] * Je[2][1] - Je[2][0] * Je[1][1] * Je[0][2] -
                               Je[2][1] * Je[1][2] * Je[0][0] - Je[2][2] * Je[1][0] * Je[0][1];
            // cofactors c(i,j) = (-1)^(i+j) minor(i,j); He(i,j) = c(j,i) / det
            double c[3][3];
            c[0][0] = Je[1][1] * Je[2][2] - Je[2][1] * Je[1][2];
            c[0][1] = -(Je[1][0] * Je[2][2] - Je[2][0] * Je[1][2]);
            c[0][2] = Je[1][0] * Je[2][1] - Je[2][0] * Je[1][1];
            c[1][0] = -(Je[0][1] * Je[2][2] - Je[2][1] * Je[0][2]);
            c[1][1] = Je[0][0] * Je[2][2] - Je[2][0] * Je[0][2];
            c[1][2] = -(Je[0][0] * Je[2][1] - Je[2][0] * Je[0][1]);
            c[2][0] = Je[0][1] * Je[1][2] - Je[1][1] * Je[0][2];
            c[2][1] = -(Je[0][0] * Je[1][2] - Je[1][0] * Je[0][2]);
            c[2][2] = Je[0][0] * Je[1][1] - Je[1][0] * Je[0][1];
            const double rdet = 1.0 / det;
            double *H = sH + t * 9;  // He(:,:,g,e) column-major
#pragma unroll
            for (int ii = 0; ii < 3; ++ii)
#pragma unroll
                for (int jj = 0; jj < 3; ++jj) H[ii + 3 * jj] = rdet * c[jj][ii];
            if (eb < ne) {
                __builtin_nontemporal_store(wg * det, a.gpvol + (e0 + eb) * NN + g);
                bad_det += !(det > 0.0);
            }
        }
        __syncthreads();
        double *He = a.He + e0 * NN * 9;
        const int n9 = ne * NN * 9;
        for (int i = t * 2; i + 1 < n9; i += NT * 2)
            __builtin_nontemporal_store(*(const pair_t *)(sH + i), (pair_t *)(He + i));
        if ((n9 & 1) && t == 0) He[n9 - 1] = sH[n9 - 1];
    }
    if (bad_conn) atomicAdd(&a.counts[0], (unsigned long long)bad_conn);
    if (bad_det) atomicAdd(&a.counts[1], (unsigned long long)bad_det);
}

template <int P>
static hipError_t launch_p(const GeomArgs &a, hipStream_t s)
{
    using S = GeomShape<P>;
    const dim3 grid((unsigned)((a.nelem + S::EC - 1) / S::EC)), block(S::NT);
    if (a.mz <= S::Q)
        hipLaunchKernelGGL((k_elem_jacobian<P, true>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((k_elem_jacobian<P, false>), grid, block, 0, s, a);
    return hipGetLastError();
}

hipError_t launch_elem_jacobian(int porder, const GeomArgs &a, hipStream_t s)
{
    if (a.nelem <= 0) return hipSuccess;
    switch (porder) {
    case 1: return launch_p<1>(a, s);
    case 2: return launch_p<2>(a, s);
    case 3: return launch_p<3>(a, s);
    case 4: return launch_p<4>(a, s);
    case 5: return launch_p<5>(a, s);
    case 6: return launch_p<6>(a, s);
    case 7: return launch_p<7>(a, s);
    case 8: return launch_p<8>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace msod
