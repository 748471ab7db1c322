// 2D residual of the scalar equation in one launch, four lanes to an element
// (P1 to P4), for meshes with elements enough to fill the chip.
//
// The matrix instructions of residual_wave2d.h serve a fixed 4 x 4 tensor per
// element, most of it padding at P1 and P2, and P4 does not fit.  Here a wave
// owns 16 elements and a lane one face of its element, then one line of volume
// points, then one row of the result: no padding beyond lines of five on four
// lanes.  Operators that the lanes share are scalar loads; lines and rows meet
// in LDS, through which the coefficients and the result also pass so that
// memory sees whole lines.  The neighbours' coefficients are read in place.  A
// face is a straight edge: its normal, arc length and, between two elements,
// DDG distance n . (cR - cL) are read once, not once a point.  On a boundary
// face the distance is sum_d |n_d (x_d - c_d)|, which varies along an edge that
// is oblique to the axes: read at each point.
//
// Explicit stages (residual, inverse mass, combination) over the 96 784 to
// 160 809 elements of a study's P1 to P3 and the 67 572 of its P4: 19 / 36 / 38
// us at P1 / P2 / P3 against 49 / 74 / 45 with matrix instructions, 53 us at
// P4 against 115 with the trace, flux, element and inverse mass launches.  P4
// is the faster at any size (16 x 16 step 48 for 56 us, 256 x 256 127 for 327),
// but for steps of FP32 states below 64 x 64 with boundaries (16 x 16 59 for 53,
// 48 x 48 57 for 55): one kernel for all sizes keeps a small instance's bits in
// a batch.
// Vector issue and the L1's lookups of scattered neighbour lines bound it
// about equally (each two thirds busy at P2).  FP32 states keep their increments
// (stage.h) and read them back: the same study 493 us a step to FP64's 450.
#pragma once
#include "residual_wave2d.h"

namespace ice {

// waves per SIMD the registers must allow (the same times without the bound)
constexpr int lane2d_waves(int n) { return n <= 3 ? 4 : n == 4 ? 3 : 2; }

template <int P, class PH, class UT, bool BDY, bool STAGE>
__global__ __launch_bounds__(64, lane2d_waves(P + 1)) void lane2d_kernel(DevSpace S, typename PH::Params ph0,
                                                                         DiscDev dd, const UT* __restrict__ U,
                                                                         double* __restrict__ R, UT* __restrict__ K,
                                                                         StageComb<UT> cb) {
    constexpr int N = P + 1, NB = N * N, NT = (N + 2) * N;
    constexpr int EW = 16, NL = (EW * NB + 63) / 64;  // elements, strided entries a lane
    constexpr int IT = (N + 3) / 4;                   // lines a lane
    constexpr int LU = NB | 1, LS = (2 * NB) | 1, LW = (4 * N) | 1;  // odd: elements in different banks
    static_assert(PH::M == 1 && PH::HAS_HOMOGENEITY);
    using VT = typename PH::real;
    __shared__ double su_[EW * LU];  // [i0][i1] coefficients, later the result
    __shared__ double ss_[EW * LS];  // [q1][2][i0] flux moments of a line of points
    __shared__ double sw_[EW * LW];  // [face][t] lifted fluxes
    __shared__ double sx_[EW * 9];   // vertex coordinates
    __shared__ double st_[2 * NB];   // L0, L1 at the volume points, for rows that differ by lane
    const int wv = xcd_contiguous(blockIdx.x, gridDim.x), lane = threadIdx.x, g = lane >> 2, l = lane & 3;
    const int e0 = wv * EW, cnt = min(EW, S.nelem - e0);
    const int le = min(g, cnt - 1), e = e0 + le;
    const size_t base = (size_t)e0 * NB;
    // entry i of a lane in the wave's contiguous run of coefficients (all
    // loads are issued before the first is waited for)
    auto run = [&](const UT* v, UT (&x)[NL]) {
#pragma unroll
        for (int i = 0; i < NL; ++i) x[i] = lane + 64 * i < cnt * NB ? v[base + lane + 64 * i] : UT(0);
    };
    const int ef = S.efaces[(size_t)e * 4 + l];
    const int c = S.jcols[(size_t)e * 5 + 1 + l];
    const int nbf = c < 0 ? e : c;
    for (int k = lane; k < 2 * NB; k += 64) st_[k] = S.tab[N + 2 + (k < NB ? k : NT + k - NB)];
    {
        double p[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) p[i] = lane + 64 * i < cnt * 8 ? S.X[(size_t)e0 * 8 + lane + 64 * i] : 0.0;
        UT x[NL];
        run(U, x);
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int k = lane + 64 * i;
            if (k < EW * NB) su_[k / NB * LU + k % NB] = (double)x[i];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) sx_[(lane + 64 * i) / 8 * 9 + (lane & 7)] = p[i];
    }
    __syncthreads();
    Quad2 X;
    X.load(sx_ + le * 9, 0);
    double* su = su_ + le * LU;
    double* ss = ss_ + g * LS;
    double* sw = sw_ + g * LW;
    const double* __restrict__ xs = S.tab;
    const double* __restrict__ L0 = S.tab + (N + 2);
    const double* __restrict__ L1 = L0 + NT;
    const double* __restrict__ L2 = L1 + NT;
    const double* __restrict__ wgl = L2 + NT;

    // ---- face l: axis ax, low or high end; tangential points in the
    // element's tensor order, the normal out of the element (residual_wave2d.h)
    {
        const int ax = l & 1, hi = l >> 1;
        const int row = ef >> 4;
        const bool face = ef >= 0;
        const bool interior = face && row < S.nfi;
        const bool side = (ef >> 3) & 1;
        const double* fg = S.fgeo + (size_t)row * N * 4;
        const double sg = side ? -1.0 : 1.0;
        double n[2] = {1.0, 0.0}, len = 0.0, h = 1.0;
        if (face) {
            n[0] = sg * fg[0];
            n[1] = sg * fg[1];
            len = fg[2] * recip(wgl[0]);
            h = fg[3];
        }
        const bool near = nbf >= e0 && nbf < e0 + cnt;  // the wave holds the neighbour
        Quad2 XN;
        if (near) XN.load(sx_ + (nbf - e0) * 9, 0);
        else XN.load(S.X, nbf);
        double Co[3][N], Cn[3][N];  // derivatives along the face's axis at its tangential nodes
        {
            double un[NB];
            if (near) {
                const double* Un = su_ + (nbf - e0) * LU;
#pragma unroll
                for (int i = 0; i < NB; ++i) un[i] = Un[i];
            } else {
                const UT* Un = U + (size_t)nbf * NB;
#pragma unroll
                for (int i = 0; i < NB; ++i) un[i] = (double)Un[i];
            }
            const int st = ax ? N : 1, sk = ax ? 1 : N;
#pragma unroll
            for (int t = 0; t < N; ++t)
#pragma unroll
                for (int k = 0; k < 3; ++k) Co[k][t] = Cn[k][t] = 0.0;
#pragma unroll
            for (int k = 0; k < N; ++k) {  // node k along the axis
                double o[3], f[3];  // end rows of the operators: own, facing
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const double lo = L0[d * NT + NB + k], up = L0[d * NT + NB + N + k];
                    o[d] = hi ? up : lo;
                    f[d] = hi ? lo : up;
                }
#pragma unroll
                for (int t = 0; t < N; ++t) {
                    const double uo = su[k * sk + t * st];
                    const double ua = un[k * N + t], ub = un[t * N + k], uv = ax ? ub : ua;
                    Co[0][t] += o[0] * uo;
                    Co[1][t] += o[1] * uo;
                    Co[2][t] += o[2] * uo;
                    Cn[0][t] += f[0] * uv;
                    Cn[1][t] += f[1] * uv;
                    Cn[2][t] += f[2] * uv;
                }
            }
        }
        const double end = hi ? 1.0 : -1.0, bh = interior ? -(double)ph0.beta1 * h : 0.0;
        const typename PH::Params pf = element_params<PH>(ph0, dd.emu, interior && side ? nbf : e);
        double W[N];
#pragma unroll
        for (int t = 0; t < N; ++t) W[t] = 0.0;
#pragma unroll (N <= 3 ? N : 1)
        for (int q = 0; q < N; ++q) {
            double vo[6], vn[6];  // u, u_n, u_nn, u_t, u_nt, u_tt
#pragma unroll
            for (int k = 0; k < 6; ++k) vo[k] = vn[k] = 0.0;
#pragma unroll
            for (int t = 0; t < N; ++t) {
                const double l0 = L0[q * N + t], l1 = L1[q * N + t], l2 = L2[q * N + t];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    vo[k] += l0 * Co[k][t];
                    vn[k] += l0 * Cn[k][t];
                }
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    vo[3 + k] += l1 * Co[k][t];
                    vn[3 + k] += l1 * Cn[k][t];
                }
                vo[5] += l2 * Co[0][t];
                vn[5] += l2 * Cn[0][t];
            }
            FaceSide2<true> so, sn;
            so.set(X, ax == 0, end, xs[q], n, interior ? 0.5 : 1.0, bh);
            sn.set(XN, ax == 0, -end, xs[q], n, interior ? 0.5 : 0.0, -bh);
            double s = 0.0;
            so.add(vo[1], vo[3], vo[2], vo[4], vo[5], &s);
            sn.add(vn[1], vn[3], vn[2], vn[4], vn[5], &s);
            const double uO = vo[0], uN = vn[0], ws = len * wgl[q];
            VT Q[1] = {VT(0)};
            const VT gr[2] = {(VT)(s * n[0]), (VT)(s * n[1])};
            if (interior) {  // the face's own left and right
                const VT uL[1] = {(VT)(side ? uN : uO)}, uR[1] = {(VT)(side ? uO : uN)};
                const VT jmp[1] = {(VT)(side ? uO - uN : uN - uO)};
                const VT nv[2] = {(VT)(side ? -n[0] : n[0]), (VT)(side ? -n[1] : n[1])};
                interior_point_flux_split<2, PH>(pf, uL, uR, gr, nv, (VT)h, (VT)ws, Q, jmp);
            }
            if constexpr (BDY) {
                if (face && !interior) {
                    const int b = row - S.nfi, qf = S.ftens[(l * S.norient + ((ef & 7) ? 1 : 0)) * N + q];
                    const int4 rec = S.fbdy[b];
                    const double bvp = dd.bval[(size_t)b * N + qf];
                    const VT nv[2] = {(VT)n[0], (VT)n[1]};
                    const VT uI[1] = {(VT)uO}, jd[1] = {(VT)(bvp - uO)}, bv[1] = {(VT)bvp};
                    const VT hb = (VT)fg[qf * 4 + 3];
                    VT uB[1];
                    boundary_point_flux<2, PH>(pf, info_bctype(rec.y), rec.z, uI, gr, bv, nv, hb, (VT)ws, Q, uB, jd);
                }
            }
            const double qv = side ? -(double)Q[0] : (double)Q[0];
#pragma unroll
            for (int t = 0; t < N; ++t) W[t] += L0[q * N + t] * qv;
        }
        const double eL = L0[NB], eR = L0[NB + 2 * N - 1], ew = hi ? eR : eL;  // only the end nodes carry the face's trace
#pragma unroll
        for (int t = 0; t < N; ++t) sw[l * N + t] = ew * W[t];
    }

    // ---- volume term, lines of points q1 = l, l + 4
    double lam_w = 0.0, vis_w = 0.0, lam_l = 0.0;  // maxima, and the wave speed at the lane's last point
#pragma unroll 1
    for (int q1 = l; q1 < N; q1 += 4) {
        const typename PH::Params ph = element_params<PH>(ph0, dd.emu, e);
        double a[N], b[N], s0[N], s1[N];
#pragma unroll
        for (int i = 0; i < N; ++i) a[i] = b[i] = s0[i] = s1[i] = 0.0;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double l0 = st_[q1 * N + j], l1 = st_[NB + q1 * N + j];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                a[i] += l0 * su[i * N + j];
                b[i] += l1 * su[i * N + j];
            }
        }
        const double x1 = xs[q1], w1 = wgl[q1];
#pragma unroll
        for (int q0 = 0; q0 < N; ++q0) {
            double A[2][2];
            const double det = X.cof(xs[q0], x1, A);
            const double detc = fmax(0.0, det);
            const double idet = recip((det == 0.0) ? 1.0 : det);
            double v = 0.0, g0 = 0.0, g1 = 0.0;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                v += L0[q0 * N + i] * a[i];
                g0 += L1[q0 * N + i] * a[i];
                g1 += L0[q0 * N + i] * b[i];
            }
            g0 *= idet;
            g1 *= idet;
            const VT uv[1] = {(VT)v};
            const VT gx[2] = {(VT)(g0 * A[0][0] + g1 * A[1][0]), (VT)(g0 * A[0][1] + g1 * A[1][1])};
            VT F[2];
            PH::flux(ph, uv, gx, F);
            if (dd.wave) {
                const double lam = PH::wave_speed(ph, uv);
                lam_w = fmax(lam_w, lam);
                vis_w = fmax(vis_w, (double)PH::visc_at(ph, uv));
                lam_l = lam;
            }
            const double fac = detc * (wgl[q0] * w1) * idet;
            const double f0 = (double)F[0] * fac, f1 = (double)F[1] * fac;
            const double G0 = f0 * A[0][0] + f1 * A[0][1];
            const double G1 = f0 * A[1][0] + f1 * A[1][1];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                s0[i] += L1[q0 * N + i] * G0;
                s1[i] += L0[q0 * N + i] * G1;
            }
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
            ss[(2 * q1 + 0) * N + i] = s0[i];
            ss[(2 * q1 + 1) * N + i] = s1[i];
        }
    }
    __syncthreads();

    // ---- rows i0 = l, l + 4 of the residual; its 1D inverse mass along i1
    const double* __restrict__ Bi = wgl + N;  // M^-1 = B^-1 (w det)^-1 B^-T (stepper.hip), Binv[i][q]
    su = su_ + g * LU;
    double rk[IT][N];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int i = l + 4 * it;
        double* r = rk[it];
        if (i >= N) continue;
#pragma unroll
        for (int j = 0; j < N; ++j) r[j] = 0.0;
#pragma unroll
        for (int q1 = 0; q1 < N; ++q1) {
            const double s0 = ss[(2 * q1 + 0) * N + i], s1 = ss[(2 * q1 + 1) * N + i];
#pragma unroll
            for (int j = 0; j < N; ++j) r[j] += L0[q1 * N + j] * s0 + L1[q1 * N + j] * s1;
        }
        if (i == 0)
#pragma unroll
            for (int j = 0; j < N; ++j) r[j] += sw[j];
        if (i == N - 1)
#pragma unroll
            for (int j = 0; j < N; ++j) r[j] += sw[2 * N + j];
        r[0] += sw[N + i];
        r[N - 1] += sw[3 * N + i];
        if (dd.srcload)
#pragma unroll
            for (int j = 0; j < N; ++j) r[j] -= dd.srcload[(size_t)e * NB + i * N + j];
        if constexpr (STAGE) {
#pragma unroll
            for (int q = 0; q < N; ++q) {
                double s = 0.0;
#pragma unroll
                for (int j = 0; j < N; ++j) s += r[j] * Bi[j * N + q];
                su[i * N + q] = s;
            }
        } else {
#pragma unroll
            for (int j = 0; j < N; ++j) su[i * N + j] = r[j];
        }
    }
    __syncthreads();
    if constexpr (STAGE) {
        bool sing = false;
#pragma unroll 1
        for (int q1 = l; q1 < N; q1 += 4) {  // columns
            double z[N], k[N];
            const double x1 = xs[q1], w1 = wgl[q1];
#pragma unroll
            for (int q0 = 0; q0 < N; ++q0) z[q0] = 0.0;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const double y = su[i * N + q1];
#pragma unroll
                for (int q0 = 0; q0 < N; ++q0) z[q0] += Bi[i * N + q0] * y;
            }
#pragma unroll
            for (int q0 = 0; q0 < N; ++q0) {
                double A[2][2];
                const double det = X.cof(xs[q0], x1, A);
                sing |= det == 0.0;
                z[q0] *= recip(wgl[q0] * w1 * det);
            }
#pragma unroll
            for (int i = 0; i < N; ++i) {
                k[i] = 0.0;
#pragma unroll
                for (int q0 = 0; q0 < N; ++q0) k[i] += Bi[i * N + q0] * z[q0];
                su[i * N + q1] = k[i];
            }
        }
        const bool any = (__ballot(sing) >> (lane & ~3)) & 0xF;
        __syncthreads();
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int i = l + 4 * it;
            if (i >= N) continue;
            double k[N];
#pragma unroll
            for (int j = 0; j < N; ++j) k[j] = 0.0;
#pragma unroll
            for (int q = 0; q < N; ++q) {
                const double y = su[i * N + q];
#pragma unroll
                for (int j = 0; j < N; ++j) k[j] += Bi[j * N + q] * y;
            }
#pragma unroll
            for (int j = 0; j < N; ++j) su[i * N + j] = any ? 1e-8 * rk[it][j] : +k[j];
        }
        __syncthreads();
    }

    // (the first stores of the kernel: operators loaded after a store would no
    // longer be scalar loads)
    if (dd.wave) {
        store_wave_maxima(lam_w, vis_w, wv, dd.wave_part);
        if (e0 + g == S.nelem - 1 && l == (N - 1) % 4) dd.wave[1] = (unsigned long long)__double_as_longlong(lam_l);
    }

    // ---- the result in whole lines
    double v[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int k = min(lane + 64 * i, EW * NB - 1);
        v[i] = su_[k / NB * LU + k % NB];
    }
    if constexpr (!STAGE) {
#pragma unroll
        for (int i = 0; i < NL; ++i)
            if (lane + 64 * i < cnt * NB) R[base + lane + 64 * i] = v[i];
    } else {
        // stage_advance_line, stage_combine_line over the lane's strided entries
        double dt[NL];
#pragma unroll
        for (int i = 0; i < NL; ++i) dt[i] = stage_dt(cb, e0 + min((lane + 64 * i) / NB, cnt - 1));
        UT x[NL], b[NL];
        if constexpr (std::is_same<UT, double>::value) {
            run(U, x);
            if (cb.first) {
#pragma unroll
                for (int i = 0; i < NL; ++i) b[i] = x[i];
            } else {
                run(cb.base, b);
            }
#pragma unroll
            for (int i = 0; i < NL; ++i)
                if (lane + 64 * i < cnt * NB)
                    cb.out[base + lane + 64 * i] = b[i] + cb.cx * ((x[i] - b[i]) + dt[i] * v[i]);
        } else {
            double sum[NL];
            run(cb.base, b);
#pragma unroll
            for (int i = 0; i < NL; ++i) sum[i] = 0.0;
            if (cb.nprev > 0) {
                run(cb.k0, x);
#pragma unroll
                for (int i = 0; i < NL; ++i) sum[i] = cb.c0 * (double)x[i];
            }
            if (cb.nprev > 1) {
                run(cb.k1, x);
#pragma unroll
                for (int i = 0; i < NL; ++i) sum[i] += cb.c1 * (double)x[i];
            }
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const UT kn = (UT)v[i];
                if (lane + 64 * i >= cnt * NB) continue;
                cb.out[base + lane + 64 * i] = (UT)((double)b[i] + dt[i] * (sum[i] + cb.cn * (double)kn));
                if (cb.store_k) K[base + lane + 64 * i] = kn;
            }
        }
    }
}

template <int P, class PH, class UT>
int lane2d_launch(const DevSpace& S, const typename PH::Params& ph, const DiscDev& dd, const UT* U, double* R, UT* K,
                  const StageComb<UT>& cb, hipStream_t st) {
    const int nblk = (S.nelem + 15) / 16;
    if (cb.out) {  // a stage's state has the fluxes' type
        if constexpr (std::is_same<UT, typename PH::real>::value) {
            if (S.nfb > 0) lane2d_kernel<P, PH, UT, true, true><<<nblk, 64, 0, st>>>(S, ph, dd, U, R, K, cb);
            else lane2d_kernel<P, PH, UT, false, true><<<nblk, 64, 0, st>>>(S, ph, dd, U, R, K, cb);
        }
    } else {
        if (S.nfb > 0) lane2d_kernel<P, PH, UT, true, false><<<nblk, 64, 0, st>>>(S, ph, dd, U, R, K, cb);
        else lane2d_kernel<P, PH, UT, false, false><<<nblk, 64, 0, st>>>(S, ph, dd, U, R, K, cb);
    }
    if (dd.wave) launch_wave_reduce(dd.wave_part, nblk, dd.wave, st);
    return (int)hipGetLastError();
}

}  // namespace ice
