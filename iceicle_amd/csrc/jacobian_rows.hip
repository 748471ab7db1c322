// Element-block Jacobian in 1D and 2D (without DDGIC vectors), one workgroup
// per element writing its whole block row once (form_petsc_jacobian.hpp:
// 55-317, conservation_law.hpp:316-432; storage as jacobian.hip).
//
// A coefficient enters the flux at a point only through the point's states
// and DDG gradient, linearly: u += phi_j, g += the basis function's share
// G_j of the gradient (interior_point_flux_split).  So the flux is
// differenced once per point and argument, not once per coefficient: by
// forward differences in the states with the reference's step, and exactly in
// the gradient, in which every viscous flux is linear.  With
//   Z_q[v][j, w] = dQ_v/du_w phi_j + sum_d dQ_v/dg_wd G_jd
// a block is sum_q phi_i Z_q over face points (the rows of the face's nodes)
// plus sum_q w grad phi_i . Z_q over volume points: matrix products over
// points, taken on the matrix cores (v_mfma_f64_16x16x4, rows = nodes of one
// variable, columns = 16 coefficients) with Z formed in registers.
//
// Perturbing every coefficient took 2 nb m fluxes a face point against
// 2 m + m d here, and face colour by face colour the diagonal blocks were read
// back: 2D NS P3 64 x 64 1446 us with the residual, 201 us now (the 671 MB of
// blocks at 3.3 TB/s; a fill of that size reaches 6.5), and a tenth of the
// differencing error.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dg_common.h"
#include "kernels.h"
#include "physics_dev.h"

namespace ice {

namespace {

typedef double doublex4 __attribute__((ext_vector_type(4)));

constexpr double SQRT_EPS = 1.4901161193847656e-08;  // sqrt(DBL_EPSILON)

// Step of the gradient arguments.  The flux is linear in them, so a step has
// no truncation error whatever its size, and a large one leaves the total
// flux's rounding behind: with a unit step in SI units (air, energy flux 4e7,
// viscosity 1.8e-5) entries that are viscous only were up to 2e-4 off.
constexpr double GRAD_STEP = 0x1p40, INV_GRAD_STEP = 0x1p-40;

template <int D, int P, class PH>
struct RowShape {
    static constexpr int N = P + 1, NB = Pow<N, D>::value, NFQ = Pow<N, D - 1>::value, M = PH::M, NBM = NB * M;
    static constexpr int NF = 2 * D, FP = NF * NFQ;         // faces, face points
    static constexpr int CT = (NBM + 15) / 16;              // column tiles
    static constexpr int RT = (NB + 15) / 16;               // row tiles of one variable
    static constexpr int WAVES = CT < 4 ? CT : 4;
    static constexpr int THREADS = 64 * WAVES;
};

// values, gradients and (HESS) normal Hessian terms of basis function j at
// the table rows pt in the element with vertices X
template <int D, int N, bool HESS>
__device__ __forceinline__ void basis_phys(const double* tab, const double* X, const int* pt, int j, const double* nrm,
                                           double& phi, double* gx, double* hn) {
    const double* L0 = tab + (N + 2);
    const double* L1 = L0 + (N + 2) * N;
    const double* L2 = L1 + (N + 2) * N;
    double Xv[1 << D][D], xi[D], a0[D], a1[D], a2[D];
    {
        int r = j;
#pragma unroll
        for (int d = D - 1; d >= 0; --d) {
            const int id = pt[d] * N + r % N;
            r /= N;
            xi[d] = tab[pt[d]];
            a0[d] = L0[id];
            a1[d] = L1[id];
            a2[d] = HESS ? L2[id] : 0.0;
        }
    }
#pragma unroll
    for (int k = 0; k < (1 << D); ++k)
#pragma unroll
        for (int d = 0; d < D; ++d) Xv[k][d] = X[k * D + d];
    double J[D][D], Hm[D][D][D], A[D][D];
    q1_map<D>(Xv, xi, nullptr, J, Hm);
    double det = det_adj<D>(J, A);
    det = (det == 0.0) ? 1.0 : det;
    const double idet = 1.0 / det;
    double gr[D];
    phi = 1.0;
#pragma unroll
    for (int d = 0; d < D; ++d) phi *= a0[d];
#pragma unroll
    for (int a = 0; a < D; ++a) {
        double t = 1.0;
#pragma unroll
        for (int d = 0; d < D; ++d) t *= (d == a) ? a1[d] : a0[d];
        gr[a] = t;
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
        double s = 0;
#pragma unroll
        for (int k = 0; k < D; ++k) s += gr[k] * A[k][d];
        gx[d] = s * idet;
    }
    if constexpr (HESS) {
        double w[D], y[D];  // inverse map's gradient along the normal, (Hess phi) against it
#pragma unroll
        for (int l = 0; l < D; ++l) {
            double s = 0;
#pragma unroll
            for (int d = 0; d < D; ++d) s += A[l][d] * nrm[d];
            w[l] = s * idet;
            y[l] = 0.0;
        }
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
            for (int b = 0; b < D; ++b) {
                double t = 1.0;
#pragma unroll
                for (int d = 0; d < D; ++d)
                    t *= (a == b) ? (d == a ? a2[d] : a0[d]) : ((d == a || d == b) ? a1[d] : a0[d]);
#pragma unroll
                for (int k = 0; k < D; ++k) t -= Hm[k][a][b] * gx[k];
                y[b] += w[a] * t;
            }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            double s = 0;
#pragma unroll
            for (int k = 0; k < D; ++k) s += y[k] * A[k][d];
            hn[d] = s * idet;
        }
    }
}

}  // namespace

template <int D, int P, class PH>
__global__ __launch_bounds__((RowShape<D, P, PH>::THREADS), 2) void jac_row_kernel(DevSpace S, PhysParams ph,
                                                                               const double* __restrict__ bval,
                                                                               const double* __restrict__ U,
                                                                               double* __restrict__ J) {
    using T = RowShape<D, P, PH>;
    constexpr int N = T::N, NB = T::NB, NFQ = T::NFQ, M = T::M, NBM = T::NBM, NF = T::NF, FP = T::FP;
    constexpr int THREADS = T::THREADS, MD = M * D, NX = (1 << D) * D;
    constexpr int NPF = 2 * M + MD, NPV = M + MD;  // perturbed arguments of a face and a volume point
    __shared__ double sU[(NF + 1) * NBM], sX[(NF + 1) * NX];                          // own element, then the neighbours
    __shared__ int snb[NF], sef[NF];                                                  // neighbour (-1), face row word
    __shared__ double sn[FP][D], sws[FP], sh[FP];                                     // normal of the face's left, w sqrt(g), h
    __shared__ double bphi[2][FP][NB], bG[2][FP][NB][D];                              // own and facing basis at face points
    __shared__ double vphi[NB][NB], vg[NB][NB][D], sdw[NB];                           // basis and weight at volume points
    __shared__ double fu[2][FP][M], fg[FP][MD], fQ[FP][M], fres[FP * M];              // face states, DDG gradient share sum, flux
    __shared__ double dA[2][FP][M][M], dB[FP][M][MD];                                 // flux derivatives (own, facing; gradient)
    __shared__ double vu[NB][M], vgr[NB][MD], vF[NB][MD], veps[NB];
    __shared__ double dFu[NB][M][D][M], dFg[NB][M][D][MD];
    const int e = blockIdx.x, tid = threadIdx.x;
    constexpr int bslots = NF + 1;
    if (tid < NF) {
        snb[tid] = S.jcols[(size_t)e * bslots + 1 + tid];
        sef[tid] = S.efaces[(size_t)e * NF + tid];
    }
    __syncthreads();
    for (int t = tid; t < (NF + 1) * NBM; t += THREADS) {
        const int k = t / NBM, nb = k ? snb[k - 1] : e;
        sU[t] = U[(size_t)(nb < 0 ? e : nb) * NBM + t % NBM];
    }
    for (int t = tid; t < (NF + 1) * NX; t += THREADS) {
        const int k = t / NX, nb = k ? snb[k - 1] : e;
        sX[t] = S.X[(size_t)(nb < 0 ? e : nb) * NX + t % NX];
    }
    // face points in the element's tensor order s; the face row's point is its mirror (ftens)
    if (tid < FP) {
        const int f = tid / NFQ, s = tid % NFQ, ef = sef[f];
        double g[D + 2];
#pragma unroll
        for (int k = 0; k < D + 2; ++k) g[k] = k == D + 1 ? 1.0 : 0.0;
        if (ef >= 0) {
            const int q = S.ftens[(f * S.norient + (ef & 7)) * NFQ + s];
            const double* gp = S.fgeo + ((size_t)(ef >> 4) * NFQ + q) * (D + 2);
#pragma unroll
            for (int k = 0; k < D + 2; ++k) g[k] = gp[k];
        }
#pragma unroll
        for (int d = 0; d < D; ++d) sn[tid][d] = g[d];
        sws[tid] = g[D];
        sh[tid] = g[D + 1];
    }
    __syncthreads();
    // basis values and gradient shares at the face points (each side's
    // (grad phi)/2 -+ beta1 h (Hess phi) n; grad phi on boundary faces), and
    // at the volume points
    for (int t = tid; t < 2 * FP * NB; t += THREADS) {
        const int nbr = t / (FP * NB), fq = (t / NB) % FP, j = t % NB;
        const int f = fq / NFQ, s = fq % NFQ;
        const bool left = ((sef[f] >> 3) & 1) == nbr;  // this basis lives on the face's left element
        int pt[D];
#pragma unroll
        for (int d = 0; d < D; ++d) pt[d] = s;  // one tangential axis at most
        pt[f % D] = (f < D) != (nbr == 1) ? N : N + 1;
        double phi, gx[D], hn[D];
        basis_phys<D, N, true>(S.tab, sX + (nbr ? 1 + f : 0) * NX, pt, j, sn[fq], phi, gx, hn);
        // only the nodes on the face have a trace there
        int kd = j;
#pragma unroll
        for (int d = D - 1; d > f % D; --d) kd /= N;
        const bool on = kd % N == (pt[f % D] == N ? 0 : N - 1);
        bphi[nbr][fq][j] = on ? phi : 0.0;
        const bool bdy = snb[f] < 0;
        const double cg = bdy ? (nbr ? 0.0 : 1.0) : 0.5, ch = bdy ? 0.0 : (left ? -ph.beta1 : ph.beta1) * sh[fq];
#pragma unroll
        for (int d = 0; d < D; ++d) bG[nbr][fq][j][d] = cg * gx[d] + ch * hn[d];
    }
    for (int t = tid; t < NB * NB; t += THREADS) {
        const int q = t / NB, j = t % NB;
        int pt[D];
        int r = q;
#pragma unroll
        for (int d = D - 1; d >= 0; --d) { pt[d] = r % N; r /= N; }
        double phi, gx[D];
        basis_phys<D, N, false>(S.tab, sX, pt, j, nullptr, phi, gx, nullptr);
        vphi[q][j] = phi;
#pragma unroll
        for (int d = 0; d < D; ++d) vg[q][j][d] = gx[d];
        if (j == 0) {
            double Xv[1 << D][D], xi[D], Jm[D][D], Hm[D][D][D], A[D][D], wq = 1.0;
            const double* wgl = S.tab + (N + 2) + 3 * (N + 2) * N;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                xi[d] = S.tab[pt[d]];
                wq *= wgl[pt[d]];
            }
#pragma unroll
            for (int k = 0; k < (1 << D); ++k)
#pragma unroll
                for (int d = 0; d < D; ++d) Xv[k][d] = sX[k * D + d];
            q1_map<D>(Xv, xi, nullptr, Jm, Hm);
            sdw[q] = fmax(0.0, det_adj<D>(Jm, A)) * wq;
        }
    }
    __syncthreads();
    // states and gradients at the face and volume points
    for (int t = tid; t < (FP + NB) * M; t += THREADS) {
        const int p = t / M, v = t % M;
        if (p < FP) {
            double g[D] = {};
#pragma unroll
            for (int nbr = 0; nbr < 2; ++nbr) {
                const double* Un = sU + (nbr ? 1 + p / NFQ : 0) * NBM + v;
                double u = 0;
                for (int j = 0; j < NB; ++j) {
                    const double c = Un[j * M];
                    u += c * bphi[nbr][p][j];
#pragma unroll
                    for (int d = 0; d < D; ++d) g[d] += c * bG[nbr][p][j][d];
                }
                fu[nbr][p][v] = u;
            }
#pragma unroll
            for (int d = 0; d < D; ++d) fg[p][v * D + d] = g[d];
        } else {
            const int q = p - FP;
            double u = 0, g[D] = {};
            for (int j = 0; j < NB; ++j) {
                const double c = sU[j * M + v];
                u += c * vphi[q][j];
#pragma unroll
                for (int d = 0; d < D; ++d) g[d] += c * vg[q][j][d];
            }
            vu[q][v] = u;
#pragma unroll
            for (int d = 0; d < D; ++d) vgr[q][v * D + d] = g[d];
        }
    }
    __syncthreads();
    // the flux out of this element at face point p from its own state uO, the
    // facing state uN and the gradient g (0 where the face carries none)
    auto face_flux = [&](int p, const double* uO, const double* uN, const double* g, double* Q) {
        const int f = p / NFQ, ef = sef[f];
        double nrm[D];
#pragma unroll
        for (int d = 0; d < D; ++d) nrm[d] = sn[p][d];
#pragma unroll
        for (int v = 0; v < M; ++v) Q[v] = 0.0;
        if (ef < 0) return;
        if (snb[f] >= 0) {
            const bool side = (ef >> 3) & 1;
            double uL[M], uR[M];
#pragma unroll
            for (int v = 0; v < M; ++v) {
                uL[v] = side ? uN[v] : uO[v];
                uR[v] = side ? uO[v] : uN[v];
            }
            interior_point_flux_split<D, PH>(ph, uL, uR, g, nrm, sh[p], sws[p], Q);
#pragma unroll
            for (int v = 0; v < M; ++v) Q[v] = side ? -Q[v] : Q[v];
        } else {
            const int b = (ef >> 4) - S.nfi;
            const int4 rec = S.fbdy[b];
            const int bctype = info_bctype(rec.y);
            const bool general = !(bctype == ICE_BC_DIRICHLET || bctype == ICE_BC_NEUMANN ||
                                   bctype == ICE_BC_EXTRAPOLATION || bctype == ICE_BC_SPACETIME_FUTURE);
            if (bctype == ICE_BC_NEUMANN || (general && !PH::IMPLEMENTS_BCS)) return;  // no dependence on u
            const int q = S.ftens[f * S.norient * NFQ + p % NFQ];
            double bv[M], uB[M];
#pragma unroll
            for (int v = 0; v < M; ++v) bv[v] = bval[((size_t)b * NFQ + q) * M + v];
            boundary_point_flux<D, PH>(ph, bctype, rec.z, uO, g, bv, nrm, sh[p], sws[p], Q, uB);
        }
    };
    for (int p = tid; p < FP + NB; p += THREADS) {
        if (p < FP) {
            double Q[M];
            face_flux(p, fu[0][p], fu[1][p], fg[p], Q);
#pragma unroll
            for (int v = 0; v < M; ++v) fQ[p][v] = Q[v];
        } else {
            const int q = p - FP;
            double F[MD], fro = 0;
            PH::flux(ph, vu[q], vgr[q], F);
#pragma unroll
            for (int k = 0; k < MD; ++k) {
                vF[q][k] = F[k];
                fro += F[k] * F[k];
            }
            veps[q] = fmax(SQRT_EPS, SQRT_EPS * sqrt(fro));  // conservation_law.hpp:366-369
        }
    }
    __syncthreads();
    // squares of the face residuals, the lifted fluxes of the face's nodes
    for (int t = tid; t < FP * M; t += THREADS) {
        const int p = t / M, v = t % M, f = p / NFQ, a = p % NFQ;  // the face's node with tangential index a
        const int kn = f < D ? 0 : N - 1;
        const int node = D == 1 ? kn : (f % D == 0 ? kn * N + a : a * N + kn);
        double s = 0;
        for (int q = 0; q < NFQ; ++q) s += fQ[f * NFQ + q][v] * bphi[0][f * NFQ + q][node];
        fres[t] = s * s;
    }
    __syncthreads();
    for (int t = tid; t < FP * NPF + NB * NPV; t += THREADS) {
        if (t < FP * NPF) {
            const int p = t / NPF, k = t % NPF, f = p / NFQ;
            double uO[M], uN[M], g[MD], Q[M];
            if (k < 2 * M) {
                // eps = max(sqrt eps, sqrt eps |res|) (form_petsc_jacobian.hpp:122, :191;
                // the two elements' face residuals are the same up to sign)
                double r2 = 0;
                for (int i = 0; i < NFQ * M; ++i) r2 += fres[f * NFQ * M + i];
                const double eps = fmax(SQRT_EPS, SQRT_EPS * sqrt(r2)), ieps = 1.0 / eps;
#pragma unroll
                for (int v = 0; v < M; ++v) {
                    uO[v] = fu[0][p][v] + (k == v ? eps : 0.0);
                    uN[v] = fu[1][p][v] + (k == M + v ? eps : 0.0);
                }
#pragma unroll
                for (int i = 0; i < MD; ++i) g[i] = fg[p][i];
                face_flux(p, uO, uN, g, Q);
                const int w = k % M;
#pragma unroll
                for (int v = 0; v < M; ++v) dA[k / M][p][v][w] = (Q[v] - fQ[p][v]) * ieps;
            } else {
                // linear in the gradient: exact to rounding
#pragma unroll
                for (int v = 0; v < M; ++v) {
                    uO[v] = fu[0][p][v];
                    uN[v] = fu[1][p][v];
                }
#pragma unroll
                for (int i = 0; i < MD; ++i) g[i] = fg[p][i] + (k - 2 * M == i ? GRAD_STEP : 0.0);
                face_flux(p, uO, uN, g, Q);
#pragma unroll
                for (int v = 0; v < M; ++v) dB[p][v][k - 2 * M] = (Q[v] - fQ[p][v]) * INV_GRAD_STEP;
            }
        } else {
            const int s = t - FP * NPF, q = s / NPV, k = s % NPV;
            double u[M], g[MD], F[MD];
            const double eps = veps[q], ieps = 1.0 / eps;
#pragma unroll
            for (int v = 0; v < M; ++v) u[v] = vu[q][v] + (k == v ? eps : 0.0);
#pragma unroll
            for (int i = 0; i < MD; ++i) g[i] = vgr[q][i] + (k - M == i ? GRAD_STEP : 0.0);
            PH::flux(ph, u, g, F);
#pragma unroll
            for (int v = 0; v < M; ++v)
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const double df = F[v * D + d] - vF[q][v * D + d];
                    if (k < M) dFu[q][v][d][k] = df * ieps;
                    else dFg[q][v][d][k - M] = df * INV_GRAD_STEP;
                }
        }
    }
    __syncthreads();
    // blocks: A operand rows i, B operand columns c of Z, k = 4 points a step;
    // D register r of a lane holds row (lane / 16) + 4 r of column lane % 16
    const int lane = tid & 63, n = lane & 15, k4 = lane >> 4;
    double* Je = J + (size_t)e * bslots * NBM * NBM;
    for (int ct = tid >> 6; ct < T::CT; ct += T::WAVES) {
        const int col = ct * 16 + n, c = col < NBM ? col : 0, j = c / M, w = c % M;
        auto store = [&](int slot, const doublex4 (&acc)[T::RT][M]) {
            if (col >= NBM) return;
            double* Js = Je + (size_t)slot * NBM * NBM + col;
#pragma unroll
            for (int rt = 0; rt < T::RT; ++rt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = rt * 16 + k4 + 4 * r;
                    if (i >= NB) continue;
#pragma unroll
                    for (int v = 0; v < M; ++v) Js[(size_t)(i * M + v) * NBM] = acc[rt][v][r];
                }
        };
        doublex4 acc[T::RT][M];
#pragma unroll
        for (int rt = 0; rt < T::RT; ++rt)
#pragma unroll
            for (int v = 0; v < M; ++v) acc[rt][v] = doublex4{0, 0, 0, 0};
#pragma unroll 1
        for (int ks = 0; ks < (NB * D + 3) / 4; ++ks) {
            const int kk = ks * 4 + k4;
            const bool on = kk < NB * D;
            const int q = on ? kk / D : 0, d = on ? kk % D : 0;
            double a[T::RT];
#pragma unroll
            for (int rt = 0; rt < T::RT; ++rt) {
                const int i = rt * 16 + n;
                a[rt] = (on && i < NB) ? sdw[q] * vg[q][i < NB ? i : 0][d] : 0.0;
            }
            const double pj = vphi[q][j];
            double gj[D];
#pragma unroll
            for (int x = 0; x < D; ++x) gj[x] = vg[q][j][x];
#pragma unroll
            for (int v = 0; v < M; ++v) {
                double z = dFu[q][v][d][w] * pj;
#pragma unroll
                for (int x = 0; x < D; ++x) z += dFg[q][v][d][w * D + x] * gj[x];
#pragma unroll
                for (int rt = 0; rt < T::RT; ++rt)
                    acc[rt][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rt], z, acc[rt][v], 0, 0, 0);
            }
        }
#pragma unroll 1
        for (int f = 0; f < NF; ++f) {
            doublex4 off[T::RT][M];
#pragma unroll
            for (int rt = 0; rt < T::RT; ++rt)
#pragma unroll
                for (int v = 0; v < M; ++v) off[rt][v] = doublex4{0, 0, 0, 0};
            const bool coupled = snb[f] >= 0;
#pragma unroll 1
            for (int ks = 0; ks < (NFQ + 3) / 4; ++ks) {
                const int s = ks * 4 + k4;
                const bool on = s < NFQ;
                const int p = f * NFQ + (on ? s : 0);
                double a[T::RT];
#pragma unroll
                for (int rt = 0; rt < T::RT; ++rt) {
                    const int i = rt * 16 + n;
                    a[rt] = (on && i < NB) ? bphi[0][p][i < NB ? i : 0] : 0.0;
                }
#pragma unroll
                for (int nbr = 0; nbr < 2; ++nbr) {
                    if (nbr && !coupled) continue;
                    const double pj = bphi[nbr][p][j];
                    double gj[D];
#pragma unroll
                    for (int x = 0; x < D; ++x) gj[x] = bG[nbr][p][j][x];
#pragma unroll
                    for (int v = 0; v < M; ++v) {
                        double z = dA[nbr][p][v][w] * pj;
#pragma unroll
                        for (int x = 0; x < D; ++x) z += dB[p][v][w * D + x] * gj[x];
#pragma unroll
                        for (int rt = 0; rt < T::RT; ++rt) {
                            if (nbr) off[rt][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rt], z, off[rt][v], 0, 0, 0);
                            else acc[rt][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rt], z, acc[rt][v], 0, 0, 0);
                        }
                    }
                }
            }
            store(1 + f, off);  // zero where there is no neighbour: the block products multiply it by zero
        }
        store(0, acc);
    }
}

template <int D, int P, class PH>
int launch_rows(const DevSpace& S, const PhysParams& ph, const DiscDev& dd, const double* U, double* J, hipStream_t st) {
    jac_row_kernel<D, P, PH><<<S.nelem, RowShape<D, P, PH>::THREADS, 0, st>>>(S, ph, dd.bval, U, J);
    return (int)hipGetLastError();
}

template <class PH, int D>
int rows_order(int p, const DevSpace& S, const PhysParams& ph, const DiscDev& dd, const double* U, double* J,
               hipStream_t st) {
    switch (p) {
    case 1: return launch_rows<D, 1, PH>(S, ph, dd, U, J, st);
    case 2: return launch_rows<D, 2, PH>(S, ph, dd, U, J, st);
    case 3: return launch_rows<D, 3, PH>(S, ph, dd, U, J, st);
    case 4: return launch_rows<D, 4, PH>(S, ph, dd, U, J, st);
    default: return -1;
    }
}

template <int D>
static int rows_flux(int p, int flux, const DevSpace& S, const PhysParams& ph, const DiscDev& dd, const double* U,
                     double* J, hipStream_t st) {
    if (flux == ICE_FLUX_BURGERS) return rows_order<Burgers<D>, D>(p, S, ph, dd, U, J, st);
    if (flux == ICE_FLUX_NAVIER_STOKES) return rows_order<NavierStokes<D, true>, D>(p, S, ph, dd, U, J, st);
    if (flux == ICE_FLUX_EULER) return rows_order<NavierStokes<D, false>, D>(p, S, ph, dd, U, J, st);
    return -1;
}

int jacobian_rows(int ndim, int p, int flux, const DevSpace& S, const PhysParams& ph, const DiscDev& dd,
                  const double* U, double* J, hipStream_t st) {
    if (ndim == 1) return rows_flux<1>(p, flux, S, ph, dd, U, J, st);
    if (ndim == 2) return rows_flux<2>(p, flux, S, ph, dd, U, J, st);
    return -2;
}

}  // namespace ice
