// Building blocks of the kernels that keep element tensors in a wave's lanes
// and contract them with v_mfma_f64_4x4x4.
//
// A lane is lo + 4 el + 16 hi: the instruction's four independent 4 x 4 x 4
// products are four elements.  It takes A[i][k] at (hi = k, lo = i) and
// B[k][j] at (hi = k, lo = j) and returns D[i][j] at (hi = i, lo = j), so both
// operands are contracted over hi, and
//   data as A, operator as B:  D(hi = the data's lo, lo = new index)
//   operator as A, data as B:  D(hi = new index, lo = the data's lo).
// Alternating the two forms contracts one axis after the other with the
// result of each product already in place for the next: no shuffles, no LDS
// and no barriers.  Indices beyond N carry zero operators.
#pragma once
#include <hip/hip_runtime.h>

#include "physics_dev.h"

namespace ice {

__device__ __forceinline__ double mm4(double a, double b, double c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// Consecutive workgroups go to the 8 XCDs in turn; this gives each XCD a
// contiguous range of workgroups, whose neighbours' coefficients its L2 holds.
__device__ __forceinline__ int xcd_contiguous(int b, int nblk) {
    const int q = nblk >> 3, r = nblk & 7, x = b & 7, k = b >> 3;
    return x * q + (x < r ? x : r) + k;
}

// Flux parameters of element e; only Burgers takes a per-element viscosity,
// the other families read the kernel argument in place.
template <class PH>
__device__ __forceinline__ decltype(auto) element_params(const typename PH::Params& p, const double* emu, int e) {
    if constexpr (PH::HAS_HOMOGENEITY) {
        typename PH::Params q = p;
        if (emu) q.mu = (typename PH::real)emu[e];
        return q;
    } else {
        return (p);
    }
}

// Per-wave maxima of the points' wave speeds and viscosities, folded by
// wave_reduce_kernel.
__device__ __forceinline__ void store_wave_maxima(double lam, double vis, int wv, double* __restrict__ part) {
    for (int off = 32; off > 0; off >>= 1) {
        lam = fmax(lam, __shfl_xor(lam, off));
        vis = fmax(vis, __shfl_xor(vis, off));
    }
    if ((threadIdx.x & 63) == 0) {
        part[2 * (size_t)wv] = lam;
        part[2 * (size_t)wv + 1] = vis;
    }
}

}  // namespace ice
