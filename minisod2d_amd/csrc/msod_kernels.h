// Internal interface between the runtime (msod_runtime.hip) and the kernel
// translation units.  All pointers are device pointers.
//
// Element data are in the lane layout of msod_columns.h, which orders the nodes
// of an element by (I,J,K); l = I + q*(J + q*K) is the lexicographic index in the
// reference's 1-D SOD order, (I,J,K) = (AtoI,AtoJ,AtoK) - 1.
//   geo    He(i,k) (component c = i + 3k) and gpvol of each element node as five
//          pairs (c = 0,1 | 2,3 | 4,5 | 6,7 | 8 and gpvol): a node's ten values
//          in five 16-byte (FP64) or 8-byte (FP32) loads, each wave's load
//          contiguous (GeoNode)
// tab.D[q*q] is the 1-D derivative D[i*q+n] = l_n'(xi_i); tab.l2g[nn] maps l
// to the 0-based reference (Gmsh) node number, used for arrays kept in the
// reference layout (mu_e, mu_sgs).
//
// Assembly plan (built once per mesh by the runtime).  Elements are grouped
// into batches of ColShape<P>::EPB consecutive elements, one workgroup each,
// which sums its elements' contributions to every node of the batch in LDS and
// writes each of the batch's distinct nodes once.  Above kNarrowP, in the atomic
// mode, it adds from registers and needs conn alone; with FP32 outputs the nodes
// that several element nodes of the batch share are summed in LDS all the same,
// in FP64, and rounded once (unode lists them alone):
//   conn          0-based global node of each element node
//   lidx          position of that node in its batch's node list (kAlone: not listed)
//   uoff [nbatch+1]  node list of batch b: unode[uoff[b] .. uoff[b+1])
//   unode [..]    sorted distinct global nodes of each batch; bit 31 set when
//                 this batch is the first writer of the node (host plan)
//   batches[nb]   the batches processed by one launch.  Null: 0 .. nb-1 in mesh
//                 order
// Two ways to combine the batches' partial sums at nodes shared between batches
// (mode):
//   kColored: batches are coloured so that batches of one colour share no
//     node; one launch per colour, each node written with a plain store by its
//     first batch and read-add-stored by later ones.  No atomics, no zero-fill,
//     and the summation order is fixed (bitwise reproducible).
//   kAtomic: one launch over all batches, FP64 atomics into zeroed outputs.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace msod {

constexpr int kMaxP = 8;
// Orders whose batches sum in LDS.  Above, an element's share of the nodes that
// meet in a batch is small and the sums cost occupancy: order 5, 64^3, 5.68 ms
// for the pair with them and 5.01 without; order 4 gains 1 to 3% without
// (convection 128^3 10.44 -> 10.07 ms), but only where a batch's elements follow
// each other along I: otherwise it loses 15% (64^3 1.95 -> 2.24 ms, order 2, 100^3
// 1.84 -> 2.65), order 5 7%.
constexpr int kNarrowP = 4;
enum AssemblyMode { kColored = 0, kAtomic = 1 };
constexpr uint16_t kAlone = 0xffff;

// Elements per batch: ColShape<P>::EPB for run-time porder.
int batch_size(int porder);
// Those of the kernels with one node per thread: Shape<P>::BATCH and CShape<P>::BATCH.
int nodes_batch_size(int porder);
int nodes_convec_batch_size(int porder);

struct Tables {
    const double *D;      // [q*q]
    const int32_t *l2g;   // [nn]
};

struct Plan {
    const uint32_t *conn;
    const uint16_t *lidx;
    const uint32_t *uoff;
    const uint32_t *unode;
    const uint32_t *batches;
    int64_t nb;
    int mode;
    int ustride;  // stride of the node sums: the most nodes of any batch
    const uint8_t *ecol;  // coloured mode: colour of each element within its batch
    int rounds;           // and the most colours of any batch
    int kpb;              // one node per thread (msod_nodes.h): batches per workgroup
};

// Kernel arguments.  Storage types: TG for the element-sized arrays (geo;
// in the diffusion also mu_e, mu_sgs), TF for the nodal fields.  The
// kernels compute in FP64 whatever the storage: on gfx950 an FP64 FMA issues
// at the rate of an unpacked FP32 one, so FP32 storage buys bytes, not time
// in the ALUs, and FP64 arithmetic keeps rounding out of the derivative
// sweeps (whose cancellation would amplify FP32 rounding by about 1/h).
//   <double, double>  FP64 form (the reference's operands)
//   <float,  float>   FP32 storage of every input
//   <float,  double>  FP32 element arrays, FP64 nodal fields
// TO: type of the outputs, FP64, or FP32 for callers built at the
// reference's default real kind (rp = 4); the sums before the output stay
// FP64.  TU, TP: storage of the velocity and of the pressure where it differs
// from the other nodal fields (the FP32 split keeps both in FP64: the
// velocity is differentiated twice in the diffusive momentum residual, the
// pressure gradient dominates the convective one).  The kernels take the
// argument type as a template parameter and read the storage types from it.
template <typename TG, typename TF, typename TO = double, typename TU = TF, typename TP = TF>
struct ConvecArgs {
    using G = TG;
    using F = TF;
    using O = TO;
    using U = TU;
    using Pt = TP;
    int64_t nelem, npoin;
    Plan plan;
    const TG *geo;
    const TU *u;
    const TF *q, *rho, *E;
    const TP *pr;                    // nullptr: recover pressure from E
    double gamma_m1;                 // gamma-1, used when pr == nullptr
    TO *Rmass, *Rmom, *Rener;
    Tables tab;
};

template <typename TG, typename TF, typename TO = double, typename TU = TF>
struct DiffuArgs {
    using G = TG;
    using F = TF;
    using O = TO;
    using U = TU;
    int64_t nelem, npoin;
    Plan plan;
    const TG *geo;
    const TF *rho, *Tem, *mu_fluid;
    const TU *u;
    const TG *mu_e, *mu_sgs;
    double Cp, Pr, c_rho, c_ener;
    TO *Rmass, *Rmom, *Rener;
    Tables tab;
};

// The FP32 split: FP32 geometry and nodal fields, FP64 velocity (and
// pressure), FP64 arithmetic and outputs.
using ConvecSplitArgs = ConvecArgs<float, float, double, double, double>;
using DiffuSplitArgs = DiffuArgs<float, float, double, double>;

// Launchers (return hipError_t of the launch); A is a ConvecArgs or
// DiffuArgs instantiation.
template <class A>
hipError_t launch_convec(int porder, const A &a, hipStream_t s);
template <class A>
hipError_t launch_diffu(int porder, const A &a, hipStream_t s);
// FP32 storage and FP32 gathers, fluxes and derivative sweeps; FP64 node sums,
// assembly and (convection) pressure recovery.
hipError_t launch_convec_fp32(int porder, const ConvecArgs<float, float> &a, hipStream_t s);
hipError_t launch_diffu_fp32(int porder, const DiffuArgs<float, float> &a, hipStream_t s);
// The kernels with one node per thread (msod_nodes.h), FP64 arithmetic.
template <class A>
hipError_t launch_convec_nodes(int porder, const A &a, hipStream_t s);
template <class A>
hipError_t launch_diffu_nodes(int porder, const A &a, hipStream_t s);

// Zero Rmass (n), Rmom (3n), Rener (n).
hipError_t launch_zero_outputs(double *Rmass, double *Rmom, double *Rener, int64_t n,
                               hipStream_t s);
hipError_t launch_zero_outputs(float *Rmass, float *Rmom, float *Rener, int64_t n, hipStream_t s);
// Zero the listed nodes of the three outputs.
template <typename TO>
hipError_t launch_zero_nodes(TO *Rmass, TO *Rmom, TO *Rener, int64_t npoin, const uint32_t *nodes,
                             int64_t count, hipStream_t s);

// Lane-layout geometry from the reference layouts, of geo_elems(porder, nelem)
// elements.
template <typename T>
hipError_t launch_build_geo(int porder, const T *He, const T *gpvol, int64_t nelem, const int32_t *l2g, T *geo,
                            hipStream_t s);
// Elements that geo, conn and lidx hold: nelem, padded to whole batches.
int64_t geo_elems(int porder, int64_t nelem);

// He and gpvol of one element node from geo: He(i,k) = he(i + 3k), with the
// component index a compile-time constant (a register of the loaded pair, no
// copy: the values stay in flight until used).
template <typename T>
using GeoPair = T __attribute__((ext_vector_type(2)));

template <typename T>
struct GeoNode {
    GeoPair<T> v[5];
    __device__ __forceinline__ T he(int c) const { return (c & 1) ? v[c >> 1].y : v[c >> 1].x; }
    __device__ __forceinline__ T gvol() const { return v[4].y; }
};

// Blocks of a launch are dealt to the chip's 8 XCDs round robin (block i to
// XCD i % 8), each XCD with its own L2.  xcd_range gives every XCD a
// contiguous range of [0, n), so that neighbours (which share nodes and cache
// lines) meet in the same L2.  Bijective for any n.
__device__ __forceinline__ uint32_t xcd_range(uint32_t i, uint32_t n)
{
    constexpr uint32_t kXcd = 8;
    const uint32_t x = i % kXcd, k = i / kXcd, q = n / kXcd, r = n % kXcd;
    return x * q + (x < r ? x : r) + k;
}

}  // namespace msod
