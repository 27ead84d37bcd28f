// Column kernels: shapes, data layout and device helpers (porder 1..kMaxP).
//
// A workgroup takes the EPB elements of one batch.  Thread t < LANES owns the
// column of the Q nodes (I, J, 0..Q-1) of one element:
//   t = I + Q*(le + EPB*J),  le the element within the batch
// and walks it slice by slice (K = 0..Q-1).  The derivative along K stays in
// the thread's registers; those along I and J read the slice's values from
// LDS (2Q sources instead of 3Q).  Everything is unrolled over K, so a
// source costs its FP64 work and its LDS reads with immediate offsets, and no
// address arithmetic.  Up to kNarrowP the batch's node sums are in LDS too; the
// kernels above it add to the outputs from registers (msod_convec.hip,
// msod_diffu.hip).  msod_nodes.h says which calls take one node per thread instead.
//
// Against one node per thread (all three directions from LDS, rolled loops)
// the FP64 kernels issue a quarter to a third fewer VALU instructions and
// two thirds (convection) or half (diffusion) of the LDS reads per element
// node: 128^3 order 4 12.6 -> 10.3 ms (convection) and 12.9 -> 10.7 ms
// (diffusion); 64^3 1.61 -> 1.33 and 1.77 -> 1.47; order 3, 96^3 2.32 -> 2.01 and
// 2.42 -> 2.18; order 2, 100^3 1.17 -> 0.83 and 0.99 -> 0.97.  What bounds them now:
// their traffic at the rate of a large copy (45 GB, 10.4 ms at 128^3), and two
// waves per SIMD (208-230 VGPRs), whose FP64 work and LDS reads alone take 7.1 ms
// (convection, 128^3).
//
// The launch takes the batches in mesh order (xcd_runs), one workgroup each:
// neighbouring batches run side by side and share lines in L2 (order 4, 128^3
// convection: 15.9 ms in colour order).  A workgroup that walked several batches with the
// next one's gathers in flight was slower (128^3 14.6-15.5 ms): its waits for
// the gathers wait for the atomics issued after them as well.
//
// Lane layout of the element-sized arrays (entry (b, K, t) of batch b):
//   conn, lidx  [b][K][LANES]
//   geo         [b][K][5][LANES] pairs (GeoNode's five pairs)
// so that a wave's loads are contiguous.  I, J, K count the nodes of a line
// from one end to the other (ascending xi), unlike the reference's 1-D order
// (both ends first): with it, and with the elements side by side between I
// and J, consecutive lanes gather consecutive nodes of a mesh numbered along its
// rows, and the L1 serves four of them with one access.  The last batch is
// padded with copies of the last element, so that every load is unconditional.
#pragma once

#include <type_traits>

#include "msod_kernels.h"

namespace msod {

template <int P>
struct ColShape {
    static constexpr int Q = P + 1;
    static constexpr int QQ = Q * Q;
    static constexpr int NN = Q * QQ;
    // 256 threads: 10 elements at order 4, whose rows of 41 nodes share more
    // lines and nodes than two batches of 5 (64^3: convection 1.41 -> 1.31 ms,
    // diffusion 1.70 -> 1.61; 128^3: 10.65 -> 10.30 and 12.05 -> 11.20).  Above
    // kNarrowP the rows matter most, as they merge the neighbours' nodes
    // (convection 40^3 order 6: one element 1.29 ms, two 1.16, five 1.03; 48^3
    // order 7: one 3.07, two 2.67, four 2.56).
    static constexpr int NT = 256;
    static constexpr int EPB = NT / QQ;         // elements of a batch
    static constexpr int LANES = EPB * QQ;
    static constexpr int UMAX = EPB * NN;       // element nodes, and most distinct nodes, of a batch
    static constexpr int UPT = (UMAX + NT - 1) / NT;
};

// Position m of a line (0..P, ascending xi) in the reference's 1-D order
// (0: xi = -1, 1: xi = +1, 2..P: the interior), and back.
template <int P>
__host__ __device__ constexpr int line_ref(int m) { return m == 0 ? 0 : (m == P ? 1 : m + 1); }
template <int P>
__host__ __device__ constexpr int line_pos(int s) { return s == 0 ? 0 : (s == 1 ? P : s - 1); }

// Entry of element node (e, l) in the element-sized arrays: conn at entry(),
// geo's pair c at pair() + c*pair_stride().
template <int P>
struct ElemEntry {
    using S = ColShape<P>;
    int64_t e;
    int l;
    __device__ __forceinline__ int64_t slice() const { return (e / S::EPB) * S::Q + line_pos<P>(l / S::QQ); }
    __device__ __forceinline__ int lane() const
    {
        return line_pos<P>(l % S::Q) + S::Q * ((int)(e % S::EPB) + S::EPB * line_pos<P>(l / S::Q % S::Q));
    }
    __device__ __forceinline__ int64_t entry() const { return slice() * S::LANES + lane(); }
    __device__ __forceinline__ int64_t pair() const { return slice() * 5 * S::LANES + lane(); }
    static constexpr int pair_stride() { return S::LANES; }
};

// Uniform read-only data (the derivative table, the batch list): read through
// the constant address space, so that the loads are scalar (SGPRs, lgkmcnt).
// Through a plain pointer the compiler must assume that the kernel's atomics
// change them, loads them into VGPRs and waits for every load in flight.
template <typename T>
using Uniform = const __attribute__((address_space(4))) T *;
template <typename T>
__device__ __forceinline__ Uniform<T> uniform(const T *p)
{
    return (Uniform<T>)p;
}

// Workgroup i's batch (xcd_range's purpose): every XCD takes runs of kXcdRun
// neighbouring batches in turn, so that all XCDs stay in one region of the mesh,
// whose lines they find in the memory-side cache.  With one eighth of the mesh
// per XCD they do not where consecutive elements leave the rows of nodes and each
// line is read again a plane of elements later: elements ordered along z, order 4,
// 40^3 convection 805 us, in runs of 32 622 (256: 624, 2048: 804, 1: 604), diffusion
// 753 and 611; 62^3 3122 and 2081; 39^3 order 7 2886 and 2010.  Elements along the
// rows: 62^3 order 4 1277 and 1194, 128^3 11.05 and 10.60 ms, 25^3 112 and 111 us; order
// 7 diffusion 39^3 1767 and 1753 (runs of 1: 1876).
__device__ __forceinline__ uint32_t xcd_runs(uint32_t i, uint32_t n)
{
    constexpr uint32_t kXcd = 8, kXcdRun = 32;
    const uint32_t x = i % kXcd, k = i / kXcd, whole = n / (kXcd * kXcdRun) * (kXcd * kXcdRun);
    if (i < whole) return k / kXcdRun * (kXcd * kXcdRun) + x * kXcdRun + k % kXcdRun;
    return whole + xcd_range(i - whole, n - whole);
}

// One thread's place in its batch.
template <int P>
struct ColThread {
    int tc, le, I, J;
    __device__ __forceinline__ ColThread(int t)
    {
        using S = ColShape<P>;
        tc = t < S::LANES ? t : S::LANES - 1;  // idle threads load a real entry
        I = tc % S::Q;
        le = tc / S::Q % S::EPB;
        J = tc / (S::Q * S::EPB);
    }
};

// The derivative table in ascending line order: sD[i*Q + n] = l_n'(xi_i).
template <int P, typename T>
__device__ __forceinline__ void col_table(const double *D, T *sD)
{
    constexpr int Q = P + 1;
    const int t = threadIdx.x;
    if (t < Q * Q) sD[t] = (T)D[line_ref<P>(t / Q) * Q + line_ref<P>(t % Q)];
}
// Its entry (i, n), i and n compile-time constants (a scalar load).
template <int P>
__device__ __forceinline__ double col_D(Uniform<double> D, int i, int n)
{
    return D[line_ref<P>(i) * (P + 1) + line_ref<P>(n)];
}

// Pair c of entry (b, K, tc).
template <int P, bool NTL, typename T>
__device__ __forceinline__ GeoPair<T> col_geo_pair(const T *geo, uint32_t b, int K, int tc, int c)
{
    using S = ColShape<P>;
    const GeoPair<T> *p = reinterpret_cast<const GeoPair<T> *>(geo) + ((int64_t)b * S::Q + K) * 5 * S::LANES + tc;
    return NTL ? __builtin_nontemporal_load(&p[c * S::LANES]) : p[c * S::LANES];
}
// GeoNode of entry (b, K, tc).
template <int P, bool NTL, typename T>
__device__ __forceinline__ GeoNode<T> col_geo(const T *geo, uint32_t b, int K, int tc)
{
    using S = ColShape<P>;
    const GeoPair<T> *p = reinterpret_cast<const GeoPair<T> *>(geo) + ((int64_t)b * S::Q + K) * 5 * S::LANES + tc;
    GeoNode<T> g;
#pragma unroll
    for (int c = 0; c < 5; ++c) g.v[c] = NTL ? __builtin_nontemporal_load(&p[c * S::LANES]) : p[c * S::LANES];
    return g;
}

// Colour of the element e of a batch, within it (coloured mode).
template <bool COLORED>
__device__ __forceinline__ int col_color(const Plan &pl, bool active, int64_t e)
{
    return COLORED && active ? pl.ecol[e] : 0;
}

// Adds one slice's five residual values to the batch's node sums sR[c*US + li].
// Atomic mode: LDS atomics.  Coloured mode: one colour of the batch's elements
// (ec, Plan::ecol) after the other, so that the order of the sums is fixed
// (barriers: uniform control flow).  A row of elements has two colours; one
// element after the other, ten rounds a slice at order 4, made the coloured pair
// 15% slower than one node per thread.
template <bool COLORED>
__device__ __forceinline__ void col_add(double *sR, int US, bool active, int ec, int rounds, uint32_t li, const double (&v)[5])
{
    if constexpr (!COLORED) {
        if (active) {
#pragma unroll
            for (int c = 0; c < 5; ++c)
                __hip_atomic_fetch_add(&sR[c * US + li], v[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    } else {
#pragma unroll 1
        for (int k = 0; k < rounds; ++k) {
            if (active && ec == k) {
#pragma unroll
                for (int c = 0; c < 5; ++c) sR[c * US + li] += v[c];
            }
            __syncthreads();
        }
    }
}

// f(0), f(1), .. f(Q - 1) with compile-time arguments: a loop that is unrolled
// whatever its size (order 8's slices pass the compiler's limit).
template <int Q, class F, int K = 0>
__device__ __forceinline__ void col_slices(const F &f)
{
    if constexpr (K < Q) {
        f(std::integral_constant<int, K>{});
        col_slices<Q, F, K + 1>(f);
    }
}

// The last node of an element's I line and the first of its right neighbour's
// sit in neighbouring lanes: where they are one node of the mesh, its values
// are summed in the right lane (both active), and the left one has nothing to
// write (false).
template <int P, int EPB = ColShape<P>::EPB>
__device__ __forceinline__ bool col_merge(uint32_t node, int I, int le, bool both, double (&v)[5])
{
    const uint32_t next = __shfl_down(node, 1);  // by every lane
    const bool give = both && I == P && le + 1 < EPB && (threadIdx.x & 63) != 63 &&
                      next == node;
#pragma unroll
    for (int c = 0; c < 5; ++c) v[c] += __shfl_up(give ? v[c] : 0.0, 1);
    return !give;
}

// One element node's values to the outputs (atomic mode).
template <typename TO>
__device__ __forceinline__ void col_scatter(uint32_t node, const double (&v)[5], TO *Rmass, TO *Rmom, TO *Rener, int64_t npoin)
{
    const int64_t g = node;
    unsafeAtomicAdd(Rmass + g, (TO)v[0]);
    unsafeAtomicAdd(Rmom + g, (TO)v[1]);
    unsafeAtomicAdd(Rmom + npoin + g, (TO)v[2]);
    unsafeAtomicAdd(Rmom + 2 * npoin + g, (TO)v[3]);
    unsafeAtomicAdd(Rener + g, (TO)v[4]);
}

// Orders above kNarrowP with FP32 outputs (atomic mode): a value rounded to float
// at every element node, as col_scatter would, loses bits where elements of a
// batch meet.  So nodes that several lanes hold after col_merge are summed in
// LDS, sR[c*US + li], and each goes out rounded once; the others go out at once,
// a row of elements whole (33^3 order 5 convection 271 us, 29^3 order 6 305; with
// the merged nodes in LDS as well 349 and 388, rounded at every node 259 and 302).
template <typename TO>
__device__ __forceinline__ void col_add_shared(double *sR, int US, uint32_t li, uint32_t node, const double (&v)[5], TO *Rmass,
                                               TO *Rmom, TO *Rener, int64_t npoin)
{
    if (li == kAlone) {
        col_scatter(node, v, Rmass, Rmom, Rener, npoin);
    } else {
#pragma unroll
        for (int c = 0; c < 5; ++c)
            __hip_atomic_fetch_add(&sR[c * US + li], v[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}
// The shared nodes' sums to the outputs.  Sums of zero change nothing (where a
// batch is split between workgroups, its list holds the other part's nodes too).
template <typename TO>
__device__ __forceinline__ void col_write_shared(const Plan &pl, uint32_t b, const double *sR, int NT, TO *Rmass, TO *Rmom,
                                                 TO *Rener, int64_t npoin)
{
    const uint32_t u0 = uniform(pl.uoff)[b], U = uniform(pl.uoff)[b + 1] - u0;
    for (uint32_t i = threadIdx.x; i < U; i += NT) {
        const int64_t g = pl.unode[u0 + i];
        TO *dst[5] = {Rmass + g, Rmom + g, Rmom + npoin + g, Rmom + 2 * npoin + g, Rener + g};
#pragma unroll
        for (int c = 0; c < 5; ++c) {
            const double v = sR[c * pl.ustride + i];
            if (v != 0.0) unsafeAtomicAdd(dst[c], (TO)v);
        }
    }
}

// A thread's entries t, t + NT, ... of a batch's node list.
template <int P>
__device__ __forceinline__ void col_list(const uint32_t *unode, uint32_t U, uint32_t (&wn)[ColShape<P>::UPT])
{
#pragma unroll
    for (int j = 0; j < ColShape<P>::UPT; ++j) {
        const uint32_t i = threadIdx.x + j * ColShape<P>::NT;
        wn[j] = unode[i < U ? i : U - 1];
    }
}

// The batch's node sums to the outputs, each distinct node once (atomically
// onto zeroed outputs; coloured: stored by the node's first writer, added by
// the others).
template <int P, bool COLORED, typename TO>
__device__ __forceinline__ void col_write(double *sR, int US, const uint32_t (&wn)[ColShape<P>::UPT],
                                          uint32_t U, TO *Rmass, TO *Rmom, TO *Rener, int64_t npoin)
{
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));  // no index or address of the sums held across the batch
#pragma unroll
    for (int j = 0; j < ColShape<P>::UPT; ++j) {
        const uint32_t i = t + j * ColShape<P>::NT;
        if (i >= U) break;
        const uint32_t w = wn[j];
        const int64_t g = w & 0x7fffffffu;
        TO *dst[5] = {Rmass + g, Rmom + g, Rmom + npoin + g, Rmom + 2 * npoin + g, Rener + g};
        TO v[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) v[c] = (TO)sR[c * US + i];
        if constexpr (!COLORED) {
#pragma unroll
            for (int c = 0; c < 5; ++c) unsafeAtomicAdd(dst[c], v[c]);
        } else if (w >> 31) {
#pragma unroll
            for (int c = 0; c < 5; ++c) *dst[c] = v[c];
        } else {
#pragma unroll
            for (int c = 0; c < 5; ++c) *dst[c] += v[c];
        }
    }
}

}  // namespace msod
