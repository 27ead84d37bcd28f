// Device geometry: arguments of the elem_jacobian kernel (msod_geom.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace msod {

struct GeomArgs {
    const int32_t *connec;   // (nelem,nnode) reference layout, 1-based
    const double *coord;     // (npoin,3)
    const double *wgp;       // [ngaus]
    // nonzero entries k = 0.. of dNgp(d,:,g) at row (k*3 + d)*ngaus + g, in
    // increasing a; shorter rows are padded with weight 0 and a = nnode, a node
    // whose coordinates the kernel holds as zeros
    const uint16_t *nza;     // local node a (0-based)
    const double *nzw;       // dNgp(d,a,g)
    int64_t nelem, npoin;
    int mz;                  // longest row
    double *He;              // He(3,3,ngaus,nelem)
    double *gpvol;           // gpvol(1,ngaus,nelem)
    unsigned long long *counts;  // [0] connec entries outside 1..npoin, [1] det(Je) <= 0
};

hipError_t launch_elem_jacobian(int porder, const GeomArgs &a, hipStream_t s);

}  // namespace msod
