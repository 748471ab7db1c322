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

// step size of element e in a stage combination
template <class KT>
__device__ __forceinline__ double stage_dt(const StageComb<KT>& cb, int e) {
    return (cb.stp && cb.stp->done) ? 0.0 : (cb.dte ? cb.dte[e] : *cb.dtp);
}

}  // namespace ice
