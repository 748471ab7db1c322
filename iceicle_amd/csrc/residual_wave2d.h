// 2D residual in one launch, P1 to P3, without LDS: a wave owns four elements
// and every contraction is a v_mfma_f64_4x4x4 (four independent 4 x 4 x 4
// products, one per element).
//
// The element's N x N tensor, its N x N volume points and its 4 x N face
// points each fit its 16 (hi, lo) lanes (wave_tensor.h), one value a lane.
//
// Per wave: the volume term (interpolation, flux, test contraction), the
// traces of the own faces and of the four neighbours' facing sides
// (re-evaluated from their coefficients, so no trace or flux passes through
// memory), one numerical flux per face point and lane, its lifting, and
// optionally the inverse mass matrix with the stage combination of an
// explicit step, whose increments then never travel as a residual.
//
// Measured against the trace, flux and element launches it replaces: 2D NS
// P3 128 x 128 FP64 39.7 -> 21.1 us, mixed 131 x 97 28.3 -> 19.2 us; Burgers
// P2 32 x 32 residual 12.2 -> 7.5 us, RK3-SSP step 60 -> 22.5 us (14 launches
// -> 5).  No one unit bounds it (NS P3 128 x 128, 1011 vector and 172
// matrix instructions a wave): vector instructions are active in 39% of the SIMD
// cycles and the matrix units in 25%, waves wait in 41% of theirs, and 4096 waves
// at three a SIMD are a round and a third, 2.5 resident on average.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dg_common.h"
#include "kernels.h"
#include "physics_dev.h"
#include "stage.h"
#include "wave_tensor.h"

namespace ice {

// Bilinear map x = m + a xi0 + c xi1 + b xi0 xi1 of one element
struct Quad2 {
    double a[2], b[2], c[2];
    __device__ __forceinline__ void load(const double* __restrict__ X, int e) {
        const double* p = X + (size_t)e * 8;
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = p[k];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const double s02 = v[4 + d] - v[d], s13 = v[6 + d] - v[2 + d];
            a[d] = 0.25 * (s02 + s13);
            b[d] = 0.25 * (s13 - s02);
            c[d] = 0.25 * ((v[2 + d] - v[d]) + (v[6 + d] - v[4 + d]));
        }
    }
    // cofactors A[k][j] = det dxi_k/dx_j at (xi0, xi1); returns det J
    __device__ __forceinline__ double cof(double xi0, double xi1, double (&A)[2][2]) const {
        const double j00 = a[0] + b[0] * xi1, j10 = a[1] + b[1] * xi1;
        const double j01 = c[0] + b[0] * xi0, j11 = c[1] + b[1] * xi0;
        A[0][0] = j11;
        A[0][1] = -j01;
        A[1][0] = -j10;
        A[1][1] = j00;
        return j00 * j11 - j01 * j10;
    }
};

// An element's side of the DDG gradient at a face point from its reference
// derivatives along the face normal's axis n and the tangential axis t (g, h:
// first and second), s += cg grad u + bh (Hess u) nrm (conservation_law.hpp:
// 529-552, finite_element.hpp:328-398).  NORMAL: its component along the
// normal only, all that the scalar diffusive flux takes.
template <bool NORMAL>
struct FaceSide2 {
    double An[2], At[2], wn, wt, bn, bt, cg, bh;
    __device__ __forceinline__ void set(const Quad2& X, bool ax0, double end, double t, const double* nrm, double cg_,
                                        double bh_) {
        double A[2][2];
        double det = X.cof(ax0 ? end : t, ax0 ? t : end, A);
        det = (det == 0.0) ? 1.0 : det;
        const double idet = recip(det);
#pragma unroll
        for (int d = 0; d < 2; ++d) {  // rows of the inverse map's gradient
            An[d] = (ax0 ? A[0][d] : A[1][d]) * idet;
            At[d] = (ax0 ? A[1][d] : A[0][d]) * idet;
        }
        wn = An[0] * nrm[0] + An[1] * nrm[1];
        wt = At[0] * nrm[0] + At[1] * nrm[1];
        bn = X.b[0] * An[0] + X.b[1] * An[1];  // mixed derivative of the map against grad u
        bt = X.b[0] * At[0] + X.b[1] * At[1];
        cg = cg_;
        bh = bh_;
    }
    __device__ __forceinline__ void add(double gn, double gt, double hnn, double hnt, double htt, double* s) const {
        const double m = hnt - (gn * bn + gt * bt);
        const double yn = cg * gn + (wn * hnn + wt * m) * bh, yt = cg * gt + (wn * m + wt * htt) * bh;
        if constexpr (NORMAL) {
            s[0] += yn * wn + yt * wt;
        } else {
            s[0] += yn * An[0] + yt * At[0];
            s[1] += yn * An[1] + yt * At[1];
        }
    }
};

// Waves per SIMD the registers must allow: 3 costs NS some scratch (80 B a lane,
// 12 of the 21 MB written at 128 x 128) and measured 21.2 us against 21.2 at 2
// (mixed, 32 B: 19.2 against 20.4); 4 spills 370 B: 36 us.
#ifndef ICE_WAVE2D_MINW
#define ICE_WAVE2D_MINW 3
#endif

template <int P, class PH, class UT, bool BDY, bool STAGE>
__global__ __launch_bounds__(256, ICE_WAVE2D_MINW) void wave2d_kernel(DevSpace S, typename PH::Params ph0, DiscDev dd,
                                                     const UT* __restrict__ U, double* __restrict__ R,
                                                     UT* __restrict__ K, StageComb<UT> cb) {
    constexpr int N = P + 1, NB = N * N, M = PH::M, NT = (N + 2) * N;
    constexpr bool GRAD = !(std::is_same<PH, NavierStokes<2, false, double>>::value ||
                            std::is_same<PH, NavierStokes<2, false, float>>::value);
    constexpr bool FULL = N == 4;  // every lane holds a node and a point
    using VT = typename PH::real;
    const int lane = threadIdx.x & 63, lo = lane & 3, hi = lane >> 4, el = (lane >> 2) & 3;
    const int wv = xcd_contiguous(blockIdx.x, gridDim.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (wv * 4 >= S.nelem) return;
    const bool own = wv * 4 + el < S.nelem;
    const int e = own ? wv * 4 + el : S.nelem - 1;
    // Lanes beyond N repeat the last node or point: the operators' zero rows
    // hi >= N keep them out of every contraction, and they are not stored.
    const int lc = FULL ? lo : min(lo, N - 1), hc = FULL ? hi : min(hi, N - 1);
    const bool kin = FULL || hi < N;
    const int nd = lc * N + hc, ndT = hc * N + lc;

    // element across each face, the face row of this lane's face, the states
    int nb[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const int c = S.jcols[(size_t)e * 5 + 1 + f];
        nb[f] = c < 0 ? e : c;
    }
    const int ef = S.efaces[(size_t)e * 4 + hi];
    const int ft0 = S.ftens[(hi * S.norient + 0) * N + lc], ft1 = S.ftens[(hi * S.norient + 1) * N + lc];
    double u0[M], uT[M], un[4][M];
    const UT* Ue = U + (size_t)e * NB * M;
#pragma unroll
    for (int v = 0; v < M; ++v) {
        u0[v] = (double)Ue[nd * M + v];
        uT[v] = (double)Ue[ndT * M + v];
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const UT* Un = U + (size_t)nb[f] * NB * M + ((f & 1) ? nd : ndT) * M;
#pragma unroll
        for (int v = 0; v < M; ++v) un[f][v] = (double)Un[v];
    }
    Quad2 X;
    X.load(S.X, e);
    const int nbf = hi == 0 ? nb[0] : hi == 1 ? nb[1] : hi == 2 ? nb[2] : nb[3];
    const double* xs = S.tab;
    const double* L0 = S.tab + (N + 2);
    const double* L1 = L0 + NT;
    const double* L2 = L1 + NT;
    const double* wgl = L2 + NT;
    const double l0 = kin ? L0[nd] : 0.0, l1 = kin ? L1[nd] : 0.0;      // L[point lo][node hi]
    const double l0t = kin ? L0[ndT] : 0.0, l1t = kin ? L1[ndT] : 0.0;  // L[point hi][node lo]

    // ---- volume term: points (q0 = hi, q1 = lo), result at node (i0 = lo, i1 = hi)
    double r[M];
    double lam_w = 0.0, vis_w = 0.0;
    {
        decltype(auto) ph = element_params<PH>(ph0, dd.emu, e);
        double A[2][2];
        const double det = X.cof(xs[hc], xs[lc], A);
        const double detc = fmax(0.0, det);
        const double idet = recip((det == 0.0) ? 1.0 : det);
        VT u[M], gx[M * 2], F[M * 2];
#pragma unroll
        for (int v = 0; v < M; ++v) {
            const double t0 = mm4(u0[v], l0, 0.0);
            const double s = mm4(l0, t0, 0.0);
            u[v] = (VT)s;
            if constexpr (GRAD) {
                const double t1 = mm4(u0[v], l1, 0.0);
                const double g0 = mm4(l1, t0, 0.0) * idet, g1 = mm4(l0, t1, 0.0) * idet;
                gx[2 * v + 0] = (VT)(g0 * A[0][0] + g1 * A[1][0]);
                gx[2 * v + 1] = (VT)(g0 * A[0][1] + g1 * A[1][1]);
            } else {
                gx[2 * v] = gx[2 * v + 1] = VT(0);
            }
        }
        PH::flux(ph, u, gx, F);
        if (dd.wave) {
            lam_w = PH::wave_speed(ph, u);
            vis_w = PH::visc_at(ph, u);
            if (own && e == S.nelem - 1 && hi == N - 1 && lo == N - 1)
                dd.wave[1] = (unsigned long long)__double_as_longlong(lam_w);
        }
        const double fac = detc * (wgl[hc] * wgl[lc]) * idet;
#pragma unroll
        for (int a = 0; a < 2; ++a) A[a][0] *= fac, A[a][1] *= fac;
#pragma unroll
        for (int v = 0; v < M; ++v) {
            const double f0 = (double)F[2 * v], f1 = (double)F[2 * v + 1];
            const double G0 = f0 * A[0][0] + f1 * A[0][1];
            const double G1 = f0 * A[1][0] + f1 * A[1][1];
            const double s0 = mm4(G0, l1t, 0.0), s1 = mm4(G1, l0t, 0.0);
            r[v] = mm4(l1t, s1, mm4(l0t, s0, 0.0));
        }
    }

    // ---- face points: face hi, tangential point lo (the element's tensor
    // order), seen from this element: the normal points out of it and its
    // state is the left one, which gives each side of a face the same flux
    // with opposite signs.  Burgers keeps the face's own left and right,
    // whose order breaks its upwinding ties.
    {
        constexpr bool ORDERED = PH::HAS_HOMOGENEITY;
        constexpr bool NORMAL = M == 1;  // scalar diffusive flux
        const int row = ef >> 4;
        const bool face = ef >= 0;
        const bool interior = face && row < S.nfi;
        const bool side = (ef >> 3) & 1;
        const int q = (ef & 7) ? ft1 : ft0;  // the face row's point
        double n[2] = {1.0, 0.0}, ws = 0.0, h = 1.0;
        if (face) {
            const double* g = S.fgeo + ((size_t)row * N + q) * 4;
            const double sg = side ? -1.0 : 1.0;
            n[0] = sg * g[0];
            n[1] = sg * g[1];
            ws = g[2];
            h = g[3];
        }
        // 1D end-point rows: column lo is face lo, own end and facing end
        double eo[3], en[3];
#pragma unroll
        for (int k = 0; k < (GRAD ? 3 : 1); ++k) {
            const double* L = L0 + k * NT + hc;
            eo[k] = kin ? L[(lo < 2 ? N : N + 1) * N] : 0.0;
            en[k] = kin ? L[(lo < 2 ? N + 1 : N) * N] : 0.0;
        }
        const double l2 = (GRAD && kin) ? L2[nd] : 0.0;
        double uO[M], uN[M], gs[M * 2];
        FaceSide2<NORMAL> so, sn;
        if constexpr (GRAD) {
            const bool ax0 = (hi & 1) == 0;
            const double t = xs[lc], end = hi < 2 ? -1.0 : 1.0;
            const double bh = interior ? -(double)ph0.beta1 * h : 0.0;
            Quad2 XN;
            XN.load(S.X, nbf);
            so.set(X, ax0, end, t, n, interior ? 0.5 : 1.0, bh);
            sn.set(XN, ax0, -end, t, n, interior ? 0.5 : 0.0, -bh);
        }
#pragma unroll
        for (int v = 0; v < M; ++v) {
            double s[2] = {0.0, 0.0};
#pragma unroll
            for (int nbr = 0; nbr < 2; ++nbr) {
                double C[3] = {0.0, 0.0, 0.0};  // [derivative along the normal] at (face lo, node hi)
#pragma unroll
                for (int k = 0; k < (GRAD ? 3 : 1); ++k) {
                    if (nbr == 0) {
                        C[k] = mm4(uT[v], (lo & 1) ? 0.0 : eo[k], 0.0);
                        C[k] = mm4(u0[v], (lo & 1) ? eo[k] : 0.0, C[k]);
                    } else {
#pragma unroll
                        for (int f = 0; f < 4; ++f) C[k] = mm4(un[f][v], lo == f ? en[k] : 0.0, C[k]);
                    }
                }
                (nbr ? uN : uO)[v] = mm4(C[0], l0, 0.0);
                if constexpr (GRAD)
                    (nbr ? sn : so).add(mm4(C[1], l0, 0.0), mm4(C[0], l1, 0.0), mm4(C[2], l0, 0.0),
                                        mm4(C[1], l1, 0.0), mm4(C[0], l2, 0.0), s);
            }
            gs[2 * v] = NORMAL ? s[0] * n[0] : s[0];
            gs[2 * v + 1] = NORMAL ? s[0] * n[1] : s[1];
        }
        VT Q[M], g[M * 2];
#pragma unroll
        for (int v = 0; v < M; ++v) {
            Q[v] = VT(0);
            g[2 * v] = (VT)gs[2 * v];
            g[2 * v + 1] = (VT)gs[2 * v + 1];
        }
        const bool flip = ORDERED && side;
        if (interior) {
            VT uL[M], uR[M], jmp[M];
            const VT nv[2] = {(VT)(flip ? -n[0] : n[0]), (VT)(flip ? -n[1] : n[1])};
#pragma unroll
            for (int v = 0; v < M; ++v) {
                uL[v] = (VT)(flip ? uN[v] : uO[v]);
                uR[v] = (VT)(flip ? uO[v] : uN[v]);
                jmp[v] = (VT)(flip ? uO[v] - uN[v] : uN[v] - uO[v]);
            }
            interior_point_flux_split<2, PH>(element_params<PH>(ph0, dd.emu, side ? nbf : e), uL, uR, g, nv, (VT)h,
                                             (VT)ws, Q, jmp);
        }
        if constexpr (BDY) {
            if (face && !interior) {
                const int b = row - S.nfi;
                const int4 rec = S.fbdy[b];
                const int bctype = info_bctype(rec.y);
                const double* bvp = dd.bval + ((size_t)b * N + q) * M;
                const VT nv[2] = {(VT)n[0], (VT)n[1]};
                VT uI[M], jd[M], bv[M], uB[M];
#pragma unroll
                for (int v = 0; v < M; ++v) {
                    uI[v] = (VT)uO[v];
                    jd[v] = (VT)(bvp[v] - uO[v]);
                    bv[v] = (VT)bvp[v];
                }
                boundary_point_flux<2, PH>(element_params<PH>(ph0, dd.emu, e), bctype, rec.z, uI, g, bv, nv, (VT)h,
                                           (VT)ws, Q, uB, jd);
            }
        }
        // lifting: e_f(i0) on the faces of axis 0, e_f(i1) on those of axis 1
        const double eL = L0[N * N], eR = L0[(N + 1) * N + N - 1];
        const double ef0 = (hi == 0 && lo == 0) ? eL : (hi == 2 && lo == N - 1) ? eR : 0.0;
        const double ef1 = (hi == 1 && lo == 0) ? eL : (hi == 3 && lo == N - 1) ? eR : 0.0;
#pragma unroll
        for (int v = 0; v < M; ++v) {
            const double qv = flip ? -(double)Q[v] : (double)Q[v];
            const double w0 = mm4(qv, ef0, 0.0), w1 = mm4(qv, ef1, 0.0);
            r[v] = mm4(w1, l0t, mm4(l0t, w0, r[v]));
        }
    }
    const size_t o = ((size_t)e * NB + nd) * M;
    const bool store = own && (FULL || (lo < N && hi < N));
    if (dd.srcload) {
#pragma unroll
        for (int v = 0; v < M; ++v) r[v] -= dd.srcload[o + v];
    }
    if (dd.wave) store_wave_maxima(lam_w, vis_w, wv, dd.wave_part);
    if constexpr (!STAGE) {
        if (store) {
#pragma unroll
            for (int v = 0; v < M; ++v) R[o + v] = r[v];
        }
    } else {
        // M^-1 = B^-1 (w det)^-1 B^-T (stepper.hip), Binv[i][q]
        const double* Bi = wgl + N;
        const double bt = kin ? Bi[ndT] : 0.0, bn = kin ? Bi[nd] : 0.0;
        double A[2][2];
        const double det = X.cof(xs[hc], xs[lc], A);
        const bool sing = (__ballot(det == 0.0) & (0x000F000F000F000Full << (4 * el))) != 0;
        const double sc = recip(wgl[hc] * wgl[lc] * det);
        UT kn[M];
#pragma unroll
        for (int v = 0; v < M; ++v) {
            const double y = mm4(bt, mm4(r[v], bt, 0.0), 0.0) * sc;
            const double k = mm4(bn, mm4(y, bn, 0.0), 0.0);
            kn[v] = sing ? (UT)(1e-8 * r[v]) : (UT)k;
        }
        if (store) {
            if constexpr (std::is_same<UT, double>::value) stage_advance_line<M>(cb, o, stage_dt(cb, e), u0, kn);
            else stage_combine_line<M, UT>(cb, K, o, stage_dt(cb, e), kn);
        }
    }
}

// Meshes without boundary faces take the kernel without their branch, but not
// for Navier-Stokes: there the branch parts the code so that 6 to 14 registers
// are spilled for 36 to 39 (stages 49 for 62), which large meshes pay in memory
// traffic (periodic 320 x 320: P3 169 -> 105 us, step 618 -> 396; P1 116 -> 95).
template <class PH>
constexpr bool wave2d_branch = std::is_same<PH, NavierStokes<2, true, double>>::value ||
                               std::is_same<PH, NavierStokes<2, true, float>>::value;

template <int P, class PH, class UT>
int wave2d_launch(const DevSpace& S, const typename PH::Params& ph, const DiscDev& dd, const UT* U, double* R, UT* K,
                  const StageComb<UT>& cb, hipStream_t st) {
    const int nw = (S.nelem + 3) / 4, nblk = (nw + 3) / 4;
    auto launch = [&](auto bdy) {
        constexpr bool BDY = decltype(bdy)::value;
        if (cb.out) {  // a stage's state has the fluxes' type
            if constexpr (std::is_same<UT, typename PH::real>::value)
                wave2d_kernel<P, PH, UT, BDY, true><<<nblk, 256, 0, st>>>(S, ph, dd, U, R, K, cb);
        } else {
            wave2d_kernel<P, PH, UT, BDY, false><<<nblk, 256, 0, st>>>(S, ph, dd, U, R, K, cb);
        }
    };
    if constexpr (wave2d_branch<PH>) launch(std::true_type{});
    else if (S.nfb > 0) launch(std::true_type{});
    else launch(std::false_type{});
    if (dd.wave) launch_wave_reduce(dd.wave_part, nw, dd.wave, st);
    return (int)hipGetLastError();
}

template <class PH, class UT>
int wave2d_order(int p, const DevSpace& S, const typename PH::Params& ph, const DiscDev& dd, const UT* U, double* R,
                 UT* K, const StageComb<UT>& cb, hipStream_t st) {
    switch (p) {
    case 1: return wave2d_launch<1, PH, UT>(S, ph, dd, U, R, K, cb, st);
    case 2: return wave2d_launch<2, PH, UT>(S, ph, dd, U, R, K, cb, st);
    case 3: return wave2d_launch<3, PH, UT>(S, ph, dd, U, R, K, cb, st);
    default: return -1;
    }
}

}  // namespace ice
