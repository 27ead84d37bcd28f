// One node per thread: batches, records and assembly of the kernels in
// msod_convec_nodes.hip and msod_diffu_nodes.hip.  They serve
//   * the FP32-arithmetic form: its results are FP32 rounding, so another order
//     of the FP32 operations is another result (columns: 9e-7 off in relative L2,
//     48^3 p=7 3.14 -> 2.5 ms for the diffusion);
//   * short launches in the default mode, the closure's network where the columns
//     run out of registers (nodes_for_atomics), and the diffusion of orders 4 and 5
//     where a batch's elements form no rows (nodes_for_order);
//   * the coloured mode where they are faster (nodes_for_colors), and where the
//     batches of the column kernels, up to five times as large, need
//     more than 32 colours (elements in little spatial order).
// Their layouts are element-major with the element-local node index l,
//   geo   [nelem][5][nn][2]  GeoNode's five pairs
//   conn, lidx  [nelem][nn]
// and their plan's batches hold Shape<P>::BATCH elements (convection
// CShape<P>::BATCH).  A workgroup takes kpb consecutive batches of the launch's
// list.
#pragma once

#include "msod_kernels.h"

namespace msod {

constexpr int kMaxKpb = 16;           // batches per workgroup, at most (LDS list of the block's batches)
constexpr int kBatchesPerBlock = 8;   // batches per workgroup (convection: measured best of 1..16 at p=4)
static_assert(kBatchesPerBlock <= kMaxKpb, "the block's batch list holds kpb entries");

template <int P>
struct Shape {
    static constexpr int Q = P + 1;
    static constexpr int NN = Q * Q * Q;
    // one node per thread; several elements per pass while they fit 256 threads
    static constexpr int EPB = NN <= 128 ? 256 / NN : 1;
    static constexpr int NT = NN <= 128 ? 256 : ((NN + 63) / 64) * 64;
    // elements per batch: about 512 element nodes, a whole number of passes
    static constexpr int BATCH_RAW = 512 / NN < 1 ? 1 : (512 / NN > 64 ? 64 : 512 / NN);
    static constexpr int BATCH = BATCH_RAW < EPB ? EPB : (BATCH_RAW / EPB) * EPB;
    static constexpr int NPASS = BATCH / EPB;
    static constexpr int UMAX = BATCH * NN;
};

// The convection's batches: Shape<P>'s, except from porder 6 on, where one
// element fills a workgroup; there two elements per batch (two passes) share
// a face in the node sums and halve the write phases per element (48^3 p=7:
// 4.75 -> 4.01 ms).  The diffusion measured slower with two (3.58 -> 3.81 ms):
// each kernel has its own plan where the sizes differ.
template <int P>
struct CShape {
    static constexpr int Q = Shape<P>::Q;
    static constexpr int NN = Shape<P>::NN;
    static constexpr int EPB = Shape<P>::EPB;
    static constexpr int NT = Shape<P>::NT;
    static constexpr int BATCH = NN >= 343 ? 2 * EPB : Shape<P>::BATCH;
    static constexpr int NPASS = BATCH / EPB;
    static constexpr int UMAX = BATCH * NN;
};

// Workgroups of a launch: each takes kpb consecutive batches of the list.
inline unsigned plan_blocks(const Plan &p) { return (unsigned)((p.nb + p.kpb - 1) / p.kpb); }

// NT: non-temporal loads (the geometry is read once per call).
template <int NN, bool NT, typename T>
__device__ __forceinline__ GeoNode<T> load_geo(const T *geo, int64_t e, int l)
{
    const GeoPair<T> *p = reinterpret_cast<const GeoPair<T> *>(geo) + e * 5 * NN + l;
    GeoNode<T> g;
#pragma unroll
    for (int k = 0; k < 5; ++k) g.v[k] = NT ? __builtin_nontemporal_load(&p[k * NN]) : p[k * NN];
    return g;
}

// Entry i of a launch's batch list (Plan::batches); a null list is mesh order.
__device__ __forceinline__ uint32_t plan_batch(const uint32_t *batches, uint32_t i)
{
    return batches ? batches[i] : i;
}

// Write phase shared by the kernels: the batch's node sums sR[c][i]
// (c = Rmass, Rmom x3, Rener) go to the outputs.  Thread t holds entries t,
// t + NT, ... of the batch's node list in registers (wn), loaded when the
// batch started.  Atomic mode: every entry is added atomically onto the
// zero-filled outputs (agent-scope FP64 atomics, performed past the L2; a
// plain store of the nodes no other batch holds was tried and is much
// slower, since those lines also take atomics).  Coloured mode: the first
// writer stores, the others add.
template <int UMAX, int NT, typename TO>
__device__ __forceinline__ void write_batch_nodes(int mode, const uint32_t (&wn)[(UMAX + NT - 1) / NT],
                                                  uint32_t U, const double (*sR)[UMAX], TO *Rmass,
                                                  TO *Rmom, TO *Rener, int64_t npoin)
{
#pragma unroll
    for (int j = 0; j < (UMAX + NT - 1) / NT; ++j) {
        const uint32_t i = threadIdx.x + j * NT;
        if (i >= U) break;
        const uint32_t w = wn[j];
        const int64_t g = w & 0x7fffffffu;
        TO *dst[5] = {Rmass + g, Rmom + g, Rmom + npoin + g, Rmom + 2 * npoin + g, Rener + g};
        if (mode == kAtomic) {
#pragma unroll
            for (int c = 0; c < 5; ++c) unsafeAtomicAdd(dst[c], (TO)sR[c][i]);
        } else if (w >> 31) {
#pragma unroll
            for (int c = 0; c < 5; ++c) *dst[c] = (TO)sR[c][i];
        } else {
#pragma unroll
            for (int c = 0; c < 5; ++c) *dst[c] += (TO)sR[c][i];
        }
    }
}

// Adds the five residual values of every element node of a pass into the
// batch's node sums, one element of the pass after the other: the nodes of
// one element are distinct, so no two threads of a round touch the same sum,
// and the summation order (pass, then element, within the batch) is fixed.
// Every thread of the block calls it (uniform control flow, barriers).
// In the atomic mode, whose global sums have no fixed order anyway, the
// batch sums use LDS atomics instead (no rounds); the caller synchronises
// before the batch is written.
template <int UMAX, int EPB>
__device__ __forceinline__ void add_pass(double (*sR)[UMAX], int mode, int le, bool active, uint32_t li,
                                         const double (&v)[5])
{
    if (mode == kAtomic) {
        if (active) {
#pragma unroll
            for (int c = 0; c < 5; ++c)
                __hip_atomic_fetch_add(&sR[c][li], v[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        return;
    }
#pragma unroll 1
    for (int k = 0; k < EPB; ++k) {
        if (active && le == k) {
#pragma unroll
            for (int c = 0; c < 5; ++c) sR[c][li] += v[c];
        }
        __syncthreads();
    }
}

}  // namespace msod
