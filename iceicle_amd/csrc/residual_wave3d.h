// 3D residual of fluxes without a gradient (Euler) in one launch, P2 and P3: a
// wave owns four elements, axes 0 and 2 of their tensors lie in the lanes
// (wave_tensor.h) and axis 1 in registers.  Contractions along the lane axes
// are FP64 matrix instructions, along axis 1 plain FMAs; the own nodes of a
// face of axis 0 or 2 come from other lanes through the wave's part of LDS
// (51 KB a workgroup at P3, no barriers).  Layouts (hi, lo): nodes (i0, i2), volume
// points (q2, q0), points of the faces of axis 0 (q2, q1), axis 1 (q2, q0),
// axis 2 (q0, q1).
//
// Each face's flux is evaluated by both its elements, from the own face
// nodes and the neighbour's (only the nodes on the face contribute to the
// face's values: the others' basis functions vanish there).  The normal points out of the
// own element, whose state is the left one; the Van Leer splitting gives the
// two sides the same flux with opposite signs.  Optionally the inverse mass
// matrix and the stage combination of an explicit step follow in registers.
//
// Measured against the trace, flux and element launches it replaces (Euler
// P3): 64^3 FP64 2.05 -> 0.57 ms, mixed 47 x 41 x 37 425 -> 165 us, 48^3
// RK3-SSP step 3.74 -> 1.08 ms.  It reads 1.7 and writes 0.67 GB at 64^3
// (0.67 and 0.67 compulsory); vector issue takes 50% and the matrix units 32%
// of the SIMD cycles at two waves per SIMD, what 250 registers allow.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "dg_common.h"
#include "kernels.h"
#include "physics_dev.h"
#include "stage.h"
#include "wave_tensor.h"

namespace ice {

// Trilinear map x = sum c[a b c] xi0^a xi1^b xi2^c of one element (index
// 4 a + 2 b + c)
struct Hex3 {
    double c[8][3];
    __device__ __forceinline__ void load(const double* __restrict__ X, int e) {
        const double* p = X + (size_t)e * 24;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            double t[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) t[k] = p[k * 3 + d];
#pragma unroll
            for (int s = 1; s < 8; s <<= 1)
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (!(k & s)) {
                        const double a = t[k], b = t[k | s];
                        t[k] = a + b;
                        t[k | s] = b - a;
                    }
#pragma unroll
            for (int k = 1; k < 8; ++k) c[k][d] = 0.125 * t[k];
        }
    }
    // derivative along axis A at the point whose other coordinates are s (the
    // lower axis) and t
    template <int A>
    __device__ __forceinline__ void column(double s, double t, double (&J)[3]) const {
        constexpr int a = 4 >> A, b = A == 0 ? 2 : 4, g = A == 2 ? 2 : 1;
#pragma unroll
        for (int d = 0; d < 3; ++d) J[d] = (c[a][d] + c[a | b][d] * s) + (c[a | g][d] + c[7][d] * s) * t;
    }
};

__device__ __forceinline__ void cross3(const double (&a)[3], const double (&b)[3], double (&o)[3]) {
    o[0] = a[1] * b[2] - a[2] * b[1];
    o[1] = a[2] * b[0] - a[0] * b[2];
    o[2] = a[0] * b[1] - a[1] * b[0];
}

// Order of the workgroups (16 consecutive elements each) of a mesh of nz
// layers: strips of `strip` workgroups per layer, layer by layer within a
// strip, so that the neighbours across layers are in flight or recently read
// (a layer of 64 x 64 P3 elements is 10 MB, an XCD's L2 4 MB): 2.8 -> 1.1 GB
// read at 64^3, 697 -> 647 us; strips of 8, 32 and 64 measured 660, 640 and
// 657 us, 48^3 steps 1.3, 0.8 and 2% slower than 16.  Layer z is
// workgroups z n / nz .. (z + 1) n / nz; returns -1 for a slot beyond it.
// Layers within a strip are in order by themselves, and no slots are left empty
// then: of thin columns' slots one in sixteen held work, on a few of the CUs
// (1 x 1 x 5000 P2 45 us, 20 in order; the three launches 41).
#ifndef ICE_WAVE3D_STRIP
#define ICE_WAVE3D_STRIP 16
#endif
constexpr unsigned WAVE3D_STRIP = ICE_WAVE3D_STRIP;
__host__ __device__ inline unsigned strip_layers(unsigned n, int nel2) {
    const unsigned nz = nel2 > 1 ? nel2 : 1;
    return (n + nz - 1) / nz > WAVE3D_STRIP ? nz : 1;
}
inline int strip_slots(int n, int nz) { return nz * ((n + nz - 1) / nz); }
__device__ __forceinline__ int strip_order(unsigned slot, unsigned n, unsigned nz) {
    const unsigned per = (n + nz - 1) / nz;  // workgroups of the largest layer
    const unsigned s = slot / (WAVE3D_STRIP * nz), rem = slot - s * (WAVE3D_STRIP * nz);
    const unsigned width = min(WAVE3D_STRIP, per - s * WAVE3D_STRIP);
    const unsigned z = rem / width, j = s * WAVE3D_STRIP + (rem - z * width);
    const unsigned b = (unsigned)((unsigned long long)z * n / nz), b1 = (unsigned)((unsigned long long)(z + 1) * n / nz);
    return b + j < b1 ? (int)(b + j) : -1;
}

// Waves per SIMD the registers must allow: at 1 the 64^3 residual took 967 us
// against 697, at 3 it spills 330 B: 1640 us.
#ifndef ICE_WAVE3D_MINW
#define ICE_WAVE3D_MINW 2
#endif

template <int P, class PH, class UT, bool BDY, bool STAGE>
__global__ __launch_bounds__(256, ICE_WAVE3D_MINW) void wave3d_kernel(DevSpace S, typename PH::Params ph, DiscDev dd,
                                                                      const UT* __restrict__ U,
                                                                      double* __restrict__ R, UT* __restrict__ K,
                                                                      StageComb<UT> cb) {
    constexpr int N = P + 1, NN = N * N, NB = NN * N, M = PH::M, NT = (N + 2) * N;
    constexpr bool FULL = N == 4;
    using VT = typename PH::real;
    const int lane = threadIdx.x & 63, lo = lane & 3, hi = lane >> 4, el = (lane >> 2) & 3;
    const unsigned nwg = ((S.nelem + 3) / 4 + 3) / 4;
    const int wg = strip_order(xcd_contiguous(blockIdx.x, gridDim.x), nwg, strip_layers(nwg, S.nel[2]));
    const int wv = wg * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (wg < 0 || wv * 4 >= S.nelem) return;
    const bool own = wv * 4 + el < S.nelem;
    const int e = own ? wv * 4 + el : S.nelem - 1;
    // lanes beyond N repeat the last index; the operators' zero rows hi >= N
    // keep them out of every contraction, and they are not stored
    const int lc = FULL ? lo : min(lo, N - 1), hc = FULL ? hi : min(hi, N - 1);
    const bool kin = FULL || hi < N;
    const double* xs = S.tab;
    const double* L0 = S.tab + (N + 2);
    const double* L1 = L0 + NT;
    const double* wgl = L1 + 2 * NT;
    const double l0 = kin ? L0[lc * N + hc] : 0.0;                                     // L[point lo][node hi]
    const double l0t = kin ? L0[hc * N + lc] : 0.0, l1t = kin ? L1[hc * N + lc] : 0.0;  // L[point hi][node lo]
    const double xlo = xs[lc], xhi = xs[hc], wq2 = wgl[lc] * wgl[hc];
    const UT* Ue = U + (size_t)e * NB * M;

    // coefficients at (hi = k0, k1, lo = k2), kept in the wave's part of LDS
    // too: the own nodes of the faces of axes 0 and 2, and a stage's input,
    // are read back from there
    constexpr int RS = 80;  // row stride: a face read's rows fall on other banks
    __shared__ double stash[4][M * N * RS];
    double* const own_u = stash[threadIdx.x >> 6];
    double u[M][N];
#pragma unroll
    for (int k1 = 0; k1 < N; ++k1)
#pragma unroll
        for (int v = 0; v < M; ++v) {
            u[v][k1] = (double)Ue[(hc * NN + k1 * N + lc) * M + v];
            own_u[(v * N + k1) * RS + lane] = u[v][k1];
        }
    Hex3 X;
    X.load(S.X, e);

    double r[M][N];  // residual at (hi = i0, i1, lo = i2)
#pragma unroll
    for (int v = 0; v < M; ++v)
#pragma unroll
        for (int i = 0; i < N; ++i) r[v][i] = 0.0;
    double lam_w = 0.0, vis_w = 0.0;

    // ---- volume term, one plane q1 of points (q2 = hi, q0 = lo) at a time
    {
        // the Jacobian's columns along the plane's normal: J0 = p0 + xi1 r0, J2 = p2 + xi1 r2, J1 fixed
        double p0[3], r0[3], p2[3], r2[3], J1[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            p0[d] = X.c[4][d] + X.c[5][d] * xhi;
            r0[d] = X.c[6][d] + X.c[7][d] * xhi;
            p2[d] = X.c[1][d] + X.c[5][d] * xlo;
            r2[d] = X.c[3][d] + X.c[7][d] * xlo;
        }
        X.column<1>(xlo, xhi, J1);
#pragma unroll 1
        for (int q1 = 0; q1 < N; ++q1) {
            const double* La = L0 + q1 * N;
            const double* Lb = L1 + q1 * N;
            VT us[M], gx[M * 3] = {}, F[M * 3];
#pragma unroll
            for (int v = 0; v < M; ++v) {
                double t = La[0] * u[v][0];
#pragma unroll
                for (int k = 1; k < N; ++k) t += La[k] * u[v][k];
                us[v] = (VT)mm4(l0, mm4(t, l0, 0.0), 0.0);
            }
            const double x1 = xs[q1];
            double J0[3], J2[3], A[3][3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                J0[d] = p0[d] + x1 * r0[d];
                J2[d] = p2[d] + x1 * r2[d];
            }
            cross3(J1, J2, A[0]);
            cross3(J2, J0, A[1]);
            cross3(J0, J1, A[2]);
            const double det = J0[0] * A[0][0] + J0[1] * A[0][1] + J0[2] * A[0][2];
            const double fac = det > 0.0 ? wq2 * wgl[q1] : 0.0;  // w max(0, det) / det
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int d = 0; d < 3; ++d) A[a][d] *= fac;
            PH::flux(ph, us, gx, F);
            if (dd.wave) {
                const double lam = PH::wave_speed(ph, us);
                lam_w = fmax(lam_w, lam);
                vis_w = fmax(vis_w, (double)PH::visc_at(ph, us));
                if (own && e == S.nelem - 1 && q1 == N - 1 && hi == N - 1 && lo == N - 1)
                    dd.wave[1] = (unsigned long long)__double_as_longlong(lam);
            }
#pragma unroll
            for (int v = 0; v < M; ++v) {
                const double f0 = (double)F[3 * v], f1 = (double)F[3 * v + 1], f2 = (double)F[3 * v + 2];
                const double G0 = f0 * A[0][0] + f1 * A[0][1] + f2 * A[0][2];
                const double G1 = f0 * A[1][0] + f1 * A[1][1] + f2 * A[1][2];
                const double G2 = f0 * A[2][0] + f1 * A[2][1] + f2 * A[2][2];
                const double x = mm4(l1t, mm4(G0, l0t, 0.0), mm4(l0t, mm4(G2, l1t, 0.0), 0.0));
                const double y = mm4(l0t, mm4(G1, l0t, 0.0), 0.0);
#pragma unroll
                for (int i = 0; i < N; ++i) r[v][i] += La[i] * x + Lb[i] * y;
            }
        }
    }

    // ---- faces
    // (the faces read coefficients that other lanes of the wave stashed)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    double lt[N];  // L0[point hi][node i]: the lifting operators along axis 1
#pragma unroll
    for (int i = 0; i < N; ++i) lt[i] = kin ? L0[hc * N + i] : 0.0;
    // nodes of a face, own and facing: (hi, lo) = (k1, k2), (k0, k2), (k1, k0)
    double nd[2][2 * M];
    auto fetch = [&](auto fc, double* t) {
        constexpr int F = decltype(fc)::value, AX = F % 3, END = F / 3;
        constexpr int SK = AX == 0 ? NN : AX == 1 ? N : 1;
        const int nbr = S.jcols[(size_t)e * 7 + 1 + F];
        const int base = AX == 0 ? hc * N + lc : AX == 1 ? hc * NN + lc : lc * NN + hc * N;
        const UT* Un = U + ((size_t)(nbr < 0 ? e : nbr) * NB + base + (END ? 0 : N - 1) * SK) * M;
        constexpr int kO = END ? N - 1 : 0;
        const double* Uo = own_u + hc * RS + 4 * el + (AX == 0 ? lc + 16 * kO : kO + 16 * lc);
#pragma unroll
        for (int v = 0; v < M; ++v) {
            t[M + v] = (double)Un[v];
            t[v] = AX == 1 ? u[v][kO] : Uo[v * N * RS];
        }
    };
    auto face = [&](auto fc, const double* t) {
        constexpr int F = decltype(fc)::value, AX = F % 3, END = F / 3;
        VT uO[M], uN[M], nv[3], Q[M];
#pragma unroll
        for (int v = 0; v < M; ++v) {
            uO[v] = (VT)mm4(l0, mm4(t[v], l0, 0.0), 0.0);
            uN[v] = (VT)mm4(l0, mm4(t[M + v], l0, 0.0), 0.0);
        }
        double n[3], Ja[3], Jb[3];
        const double x = END ? 1.0 : -1.0;
        if constexpr (AX == 0) {
            X.template column<1>(x, xhi, Ja);
            X.template column<2>(x, xlo, Jb);
        } else if constexpr (AX == 1) {
            X.template column<2>(xlo, x, Ja);
            X.template column<0>(x, xhi, Jb);
        } else {
            X.template column<0>(xlo, x, Ja);
            X.template column<1>(xhi, x, Jb);
        }
        cross3(Ja, Jb, n);
        double area, inv;
        sqrt_recip(n[0] * n[0] + n[1] * n[1] + n[2] * n[2], area, inv);
#pragma unroll
        for (int d = 0; d < 3; ++d) nv[d] = (VT)(END ? n[d] * inv : -n[d] * inv);
        const VT ws = (VT)(wq2 * area);
        PH::conv(ph, uO, uN, nv, Q);
        // (boundary faces follow below)
        const VT wsi = (!BDY || S.jcols[(size_t)e * 7 + 1 + F] >= 0) ? -ws : VT(0);
#pragma unroll
        for (int v = 0; v < M; ++v) Q[v] *= wsi;
        const double en = END ? L0[(N + 1) * N + N - 1] : L0[N * N];  // the face nodes' basis value on the face
#pragma unroll
        for (int v = 0; v < M; ++v) {
            const double w = mm4((double)Q[v] * en, l0t, 0.0);
            if constexpr (AX == 1) {
                r[v][END ? N - 1 : 0] = mm4(l0t, w, r[v][END ? N - 1 : 0]);
            } else {
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const double op = lo == (END ? N - 1 : 0) ? lt[i] : 0.0;
                    r[v][i] = AX == 0 ? mm4(op, w, r[v][i]) : mm4(w, op, r[v][i]);
                }
            }
        }
    };
    // one face ahead, axis 1 first: its own nodes are the last use of u (each
    // face's loads at its start: 647 us at 64^3 against 578)
    using std::integral_constant;
    fetch(integral_constant<int, 1>{}, nd[0]);
    fetch(integral_constant<int, 4>{}, nd[1]);
    face(integral_constant<int, 1>{}, nd[0]);
    fetch(integral_constant<int, 0>{}, nd[0]);
    face(integral_constant<int, 4>{}, nd[1]);
    fetch(integral_constant<int, 3>{}, nd[1]);
    face(integral_constant<int, 0>{}, nd[0]);
    fetch(integral_constant<int, 2>{}, nd[0]);
    face(integral_constant<int, 3>{}, nd[1]);
    fetch(integral_constant<int, 5>{}, nd[1]);
    face(integral_constant<int, 2>{}, nd[0]);
    face(integral_constant<int, 5>{}, nd[1]);

    if constexpr (BDY) {
        // boundary faces, one at a time by the waves that hold any
#pragma unroll 1
        for (int f = 0; f < 6; ++f) {
            const int ef = S.efaces[(size_t)e * 6 + f];
            const bool bdy = ef >= 0 && (ef >> 4) >= S.nfi;
            if (!__any(bdy)) continue;
            const int ax = f % 3, kO = f < 3 ? 0 : N - 1;
            const int base = ax == 0 ? hc * N + lc + kO * NN : ax == 1 ? hc * NN + lc + kO * N : lc * NN + hc * N + kO;
            VT uO[M], Q[M];
#pragma unroll
            for (int v = 0; v < M; ++v) {
                uO[v] = (VT)mm4(l0, mm4((double)Ue[base * M + v], l0, 0.0), 0.0);
                Q[v] = VT(0);
            }
            if (bdy) {
                const double x = f < 3 ? -1.0 : 1.0;
                const double x0 = ax == 0 ? x : ax == 1 ? xlo : xhi, x1 = ax == 1 ? x : xlo, x2 = ax == 2 ? x : xhi;
                double J[3][3], n[3];
                X.template column<0>(x1, x2, J[0]);
                X.template column<1>(x0, x2, J[1]);
                X.template column<2>(x0, x1, J[2]);
                double Ja[3], Jb[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    Ja[d] = ax == 0 ? J[1][d] : ax == 1 ? J[2][d] : J[0][d];
                    Jb[d] = ax == 0 ? J[2][d] : ax == 1 ? J[0][d] : J[1][d];
                }
                cross3(Ja, Jb, n);
                double area, inv;
                sqrt_recip(n[0] * n[0] + n[1] * n[1] + n[2] * n[2], area, inv);
                const VT nv[3] = {(VT)(n[0] * inv * x), (VT)(n[1] * inv * x), (VT)(n[2] * inv * x)};
                const int b = (ef >> 4) - S.nfi;
                const int4 rec = S.fbdy[b];
                // the face's point at this lane's tensor index (a face's own order is a mirror of it)
                const int q = S.ftens[(size_t)f * S.norient * NN + (ax == 2 ? hc * N + lc : lc * N + hc)];
                const double* bvp = dd.bval + ((size_t)b * NN + q) * M;
                VT g[M * 3] = {}, bv[M], uB[M];
#pragma unroll
                for (int v = 0; v < M; ++v) bv[v] = (VT)bvp[v];
                boundary_point_flux<3, PH>(ph, info_bctype(rec.y), rec.z, uO, g, bv, nv, VT(1), (VT)(wq2 * area), Q, uB);
            }
            const double en = f < 3 ? L0[N * N] : L0[(N + 1) * N + N - 1];
#pragma unroll
            for (int v = 0; v < M; ++v) {
                const double w = mm4((double)Q[v] * en, l0t, 0.0);
                if (ax == 1) {
                    const double z = mm4(l0t, w, 0.0);
                    r[v][0] += f < 3 ? z : 0.0;
                    r[v][N - 1] += f < 3 ? 0.0 : z;
                } else {
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        const double op = lo == kO ? lt[i] : 0.0;
                        r[v][i] = ax == 0 ? mm4(op, w, r[v][i]) : mm4(w, op, r[v][i]);
                    }
                }
            }
        }
    }

    const size_t o = ((size_t)e * NB + hc * NN + lc) * M;
    const bool store = own && (FULL || (lo < N && hi < N));
    if (dd.srcload) {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int v = 0; v < M; ++v) r[v][i] -= dd.srcload[o + i * N * M + v];
    }
    if (dd.wave) store_wave_maxima(lam_w, vis_w, wv, dd.wave_part);
    if constexpr (!STAGE) {
        if (store) {
#pragma unroll
            for (int i = 0; i < N; ++i)
#pragma unroll
                for (int v = 0; v < M; ++v) R[o + i * N * M + v] = r[v][i];
        }
    } else {
        // M^-1 = B^-1 (w det)^-1 B^-T (stepper.hip), Binv[i][q]; k at (hi = i0, i1, lo = i2)
        const double* Bi = wgl + N;
        const double bt = kin ? Bi[hc * N + lc] : 0.0, bn = kin ? Bi[lc * N + hc] : 0.0;
        double k[M][N];
#pragma unroll
        for (int v = 0; v < M; ++v)
#pragma unroll
            for (int i = 0; i < N; ++i) k[v][i] = 0.0;
        bool zero = false;
        double J1[3];
        X.column<1>(xlo, xhi, J1);
#pragma unroll 1
        for (int q1 = 0; q1 < N; ++q1) {
            double J0[3], J2[3], A0[3];
            X.column<0>(xs[q1], xhi, J0);
            X.column<2>(xlo, xs[q1], J2);
            cross3(J1, J2, A0);
            const double det = J0[0] * A0[0] + J0[1] * A0[1] + J0[2] * A0[2];
            zero = zero || det == 0.0;
            const double sc = recip(wq2 * wgl[q1] * det);
#pragma unroll
            for (int v = 0; v < M; ++v) {
                double t = Bi[q1] * r[v][0];
#pragma unroll
                for (int i = 1; i < N; ++i) t += Bi[i * N + q1] * r[v][i];
                const double z = mm4(bt, mm4(t, bt, 0.0), 0.0) * sc;
                const double y = mm4(bn, mm4(z, bn, 0.0), 0.0);
#pragma unroll
                for (int i = 0; i < N; ++i) k[v][i] += Bi[i * N + q1] * y;
            }
        }
        const bool sing = (__ballot(zero) & (0x000F000F000F000Full << (4 * el))) != 0;
        const double dt = stage_dt(cb, e);
        if (store) {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                UT kn[M];
#pragma unroll
                for (int v = 0; v < M; ++v) kn[v] = sing ? (UT)(1e-8 * r[v][i]) : (UT)k[v][i];
                if constexpr (std::is_same<UT, double>::value) {
                    double x[M];
#pragma unroll
                    for (int v = 0; v < M; ++v) x[v] = own_u[(v * N + i) * RS + lane];
                    stage_advance_line<M>(cb, o + i * N * M, dt, x, kn);
                } else {
                    stage_combine_line<M, UT>(cb, K, o + i * N * M, dt, kn);
                }
            }
        }
    }
}

template <int P, class PH, class UT>
int wave3d_launch(const DevSpace& S, const typename PH::Params& ph, const DiscDev& dd, const UT* U, double* R, UT* K,
                  const StageComb<UT>& cb, hipStream_t st) {
    const int nw = (S.nelem + 3) / 4, nwg = (nw + 3) / 4, nblk = strip_slots(nwg, strip_layers(nwg, S.nel[2]));
    if (cb.out) {  // a stage's state has the fluxes' type
        if constexpr (std::is_same<UT, typename PH::real>::value) {
            if (S.nfb > 0) wave3d_kernel<P, PH, UT, true, true><<<nblk, 256, 0, st>>>(S, ph, dd, U, R, K, cb);
            else wave3d_kernel<P, PH, UT, false, true><<<nblk, 256, 0, st>>>(S, ph, dd, U, R, K, cb);
        }
    } else {
        if (S.nfb > 0) wave3d_kernel<P, PH, UT, true, false><<<nblk, 256, 0, st>>>(S, ph, dd, U, R, K, cb);
        else wave3d_kernel<P, PH, UT, false, false><<<nblk, 256, 0, st>>>(S, ph, dd, U, R, K, cb);
    }
    if (dd.wave) launch_wave_reduce(dd.wave_part, nw, dd.wave, st);
    return (int)hipGetLastError();
}

}  // namespace ice
