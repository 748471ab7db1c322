// Runge-Kutta stage combination formed by the kernel that computes the
// stage's increment.
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace ice {

// Optional stage combination formed by the kernel from the increment k_new
// it computes: out = base + dt (c0 k0 + c1 k1 + cn k_new) over the nprev
// earlier increments k0, k1, with the step of rk_combine_kernel (the
// stepper's dt, or the element's, none once the run is done); k_new is
// rounded to KT first, as when it is stored and read back.
template <class KT>
struct StageComb {
    KT* out = nullptr;  // null: k = M^-1 r only
    const KT* base = nullptr;
    const KT* k0 = nullptr;
    const KT* k1 = nullptr;
    int nprev = 0;
    double c0 = 0, c1 = 0, cn = 0;
    const double* dtp = nullptr;
    const double* dte = nullptr;
    const StepState* stp = nullptr;
    bool store_k = true;  // also store k_new (a later stage reads it)
    // the stage in its increment-free form (stage_advance_line)
    bool first = false;   // the stage's input is base
    double cx = 0;
};

// the combination over nprev earlier increments kk with coefficients c[0 .. nprev]
template <class KT>
inline StageComb<KT> make_stage(const KT* base, int nprev, const KT* const* kk, const double* c, const double* dtp,
                                const double* dte, const StepState* stp, KT* out, bool store_k) {
    StageComb<KT> cb;
    cb.out = out;
    cb.base = base;
    cb.k0 = nprev > 0 ? kk[0] : nullptr;
    cb.k1 = nprev > 1 ? kk[1] : nullptr;
    cb.nprev = nprev;
    cb.c0 = nprev > 0 ? c[0] : 0.0;
    cb.c1 = nprev > 1 ? c[1] : 0.0;
    cb.cn = c[nprev];
    cb.dtp = dtp;
    cb.dte = dte;
    cb.stp = stp;
    cb.store_k = store_k;
    return cb;
}

// out = base + dt (c0 k0 + c1 k1 + cn kn) over the NL contiguous values of a
// line at o, with NPV earlier increments: straight-line loads of each input
// (so they merge into wide loads), all read before out, which may be base,
// is stored; then kn itself if the stage keeps it
template <int NPV, int NL, class KT>
__device__ __forceinline__ void stage_combine_line(const StageComb<KT>& cb, KT* __restrict__ k, size_t o, double dt,
                                                   const KT* kn) {
    double sum[NL], bv[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        double acc = 0.0;
        if constexpr (NPV > 0) acc = cb.c0 * (double)cb.k0[o + i];
        if constexpr (NPV > 1) acc += cb.c1 * (double)cb.k1[o + i];
        sum[i] = acc;
        bv[i] = (double)cb.base[o + i];
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        sum[i] += cb.cn * (double)kn[i];
        cb.out[o + i] = (KT)(bv[i] + dt * sum[i]);
    }
    if (cb.store_k) {
#pragma unroll
        for (int i = 0; i < NL; ++i) k[o + i] = kn[i];
    }
}

template <int NL, class KT>
__device__ __forceinline__ void stage_combine_line(const StageComb<KT>& cb, KT* __restrict__ k, size_t o, double dt,
                                                   const KT* kn) {
    if (cb.nprev == 0) stage_combine_line<0, NL, KT>(cb, k, o, dt, kn);
    else if (cb.nprev == 1) stage_combine_line<1, NL, KT>(cb, k, o, dt, kn);
    else stage_combine_line<2, NL, KT>(cb, k, o, dt, kn);
}

// The textbook stages in the form that stores no increment: from the stage's
// input x, out = base + cx ((x - base) + dt kn) with cx = 1, 1/4, 2/3 (the
// convex combinations of ssp_rk3.hpp:164-190; x - base is exact where the
// stages lie within a factor of two).  An FP32 x would bring its own rounding
// into the combination, so FP32 states keep their increments.  It moves 8
// vectors a step instead of 11 (3D Euler P3 48^3 step 1494 -> 1084 us, the
// inputs read back from LDS).
template <int NL>
__device__ __forceinline__ void stage_advance_line(const StageComb<double>& cb, size_t o, double dt, const double* x,
                                                   const double* kn) {
    double b[NL];
    if (cb.first) {
#pragma unroll
        for (int i = 0; i < NL; ++i) b[i] = x[i];
    } else {
#pragma unroll
        for (int i = 0; i < NL; ++i) b[i] = cb.base[o + i];
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) cb.out[o + i] = b[i] + cb.cx * ((x[i] - b[i]) + dt * kn[i]);
}

// step size of element e in a stage combination
template <class KT>
__device__ __forceinline__ double stage_dt(const StageComb<KT>& cb, int e) {
    return (cb.stp && cb.stp->done) ? 0.0 : (cb.dte ? cb.dte[e] : *cb.dtp);
}

}  // namespace ice
