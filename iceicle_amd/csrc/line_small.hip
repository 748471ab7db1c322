// Line preconditioner of chains of small blocks (bs <= 5, e.g. scalar 1D
// problems): block tridiagonal factorisation and solve.
//
// chain_*: elimination along the chain by one lane with everything in
// registers.  A chain of n dependent small inverses and products, whatever
// the card: 709 us to factor and 214 us to solve 256 blocks of 4 x 4.
//
// pcr_*: parallel cyclic reduction in one workgroup, rows to threads.  Every
// row eliminates its neighbours s = 1, 2, 4, .. rows away in each of
// ceil(log2 n) steps,
//   A = L_e D_{e-s}^-1, C = U_e D_{e+s}^-1
//   D' = D - A U_{e-s} - C L_{e+s},  L' = -A L_{e-s},  U' = -C U_{e+s}
//   b' = b - A b_{e-s} - C b_{e+s}
// until the rows stand alone, x = D^-1 b; A and C of every step are kept for
// the solves.  log2 n times the arithmetic, but a chain of 8 steps for 256
// rows: 80 us to factor, 28 us to solve.  Where the
// elimination along the chain would meet regular blocks, reduction can meet a
// singular one (a zero diagonal block); a block conditioned worse than 1e10
// sends the factorisation, and its solves, along the chain instead.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "line_small.h"

namespace ice {

namespace {

constexpr int PCR_THREADS = 256, PCR_MAX_ROWS = 1024;
constexpr int PCR_HEAD = 16;  // doubles before the workspace's arrays: [0] nonzero = factored along the chain

// I = M^-1 by Gauss-Jordan in place with partial pivoting (largest |I[i][k]|,
// lowest row on ties); rows are exchanged, and the columns back at the end,
// by selects, so that no register array is indexed at run time; false and the
// identity if singular
template <int BS>
__device__ __forceinline__ bool small_inverse(const double (&M)[BS * BS], double (&I)[BS * BS]) {
    int piv[BS];
    bool bad = false;
#pragma unroll
    for (int k = 0; k < BS * BS; ++k) I[k] = M[k];
#pragma unroll
    for (int k = 0; k < BS; ++k) {
        piv[k] = k;
        double best = fabs(I[k * BS + k]);
#pragma unroll
        for (int i = k + 1; i < BS; ++i) {
            const double a = fabs(I[i * BS + k]);
            if (a > best) {
                best = a;
                piv[k] = i;
            }
        }
        if (!(best > 0.0)) bad = true;
#pragma unroll
        for (int i = k + 1; i < BS; ++i)
#pragma unroll
            for (int c = 0; c < BS; ++c) {
                const double tk = I[k * BS + c], ti = I[i * BS + c];
                I[k * BS + c] = (piv[k] == i) ? ti : tk;
                I[i * BS + c] = (piv[k] == i) ? tk : ti;
            }
        const double ip = 1.0 / I[k * BS + k];
        I[k * BS + k] = 1.0;
#pragma unroll
        for (int c = 0; c < BS; ++c) I[k * BS + c] *= ip;
#pragma unroll
        for (int i = 0; i < BS; ++i) {
            if (i == k) continue;
            const double f = I[i * BS + k];
            I[i * BS + k] = 0.0;
#pragma unroll
            for (int c = 0; c < BS; ++c) I[i * BS + c] -= f * I[k * BS + c];
        }
    }
#pragma unroll
    for (int k = BS - 1; k >= 0; --k)
#pragma unroll
        for (int j = k + 1; j < BS; ++j)
#pragma unroll
            for (int i = 0; i < BS; ++i) {
                const double tk = I[i * BS + k], tj = I[i * BS + j];
                I[i * BS + k] = (piv[k] == j) ? tj : tk;
                I[i * BS + j] = (piv[k] == j) ? tk : tj;
            }
    if (bad)
#pragma unroll
        for (int k = 0; k < BS * BS; ++k) I[k] = k % (BS + 1) == 0 ? 1.0 : 0.0;
    return !bad;
}

template <int BS>
__device__ __forceinline__ void mul(const double (&A)[BS * BS], const double (&B)[BS * BS], double (&C)[BS * BS]) {
#pragma unroll
    for (int i = 0; i < BS; ++i)
#pragma unroll
        for (int c = 0; c < BS; ++c) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < BS; ++k) s += A[i * BS + k] * B[k * BS + c];
            C[i * BS + c] = s;
        }
}

template <int BS>
__device__ __forceinline__ void get(const double* p, int n, int e, double (&M)[BS * BS]) {
#pragma unroll
    for (int k = 0; k < BS * BS; ++k) M[k] = p[(size_t)k * n + e];
}
template <int BS>
__device__ __forceinline__ void put(double* p, int n, int e, const double (&M)[BS * BS]) {
#pragma unroll
    for (int k = 0; k < BS * BS; ++k) p[(size_t)k * n + e] = M[k];
}

// (the next element's blocks are loaded a step ahead)
template <int BS>
__device__ void chain_factor(int nelem, int nslots, const double* J, double* Sinv, double* W, int* nsingular) {
    constexpr int BB = BS * BS;
    double Wp[BB] = {};
    double cD[BB], cL[BB], cU[BB], nD[BB], nL[BB], nU[BB];
    auto load = [&](int e, double (&d)[BB], double (&l)[BB], double (&u)[BB]) {
        const double* Je = J + (size_t)e * nslots * BB;
#pragma unroll
        for (int k = 0; k < BB; ++k) {
            d[k] = Je[k];
            l[k] = Je[BB + k];
            u[k] = Je[2 * BB + k];
        }
    };
    load(0, cD, cL, cU);
    for (int e = 0; e < nelem; ++e) {
        if (e + 1 < nelem) load(e + 1, nD, nL, nU);
        double S[BB], I[BB];
#pragma unroll
        for (int i = 0; i < BS; ++i)
#pragma unroll
            for (int c = 0; c < BS; ++c) {
                double sacc = cD[i * BS + c];
                if (e > 0)
#pragma unroll
                    for (int k = 0; k < BS; ++k) sacc -= cL[i * BS + k] * Wp[k * BS + c];
                S[i * BS + c] = sacc;
            }
        if (!small_inverse<BS>(S, I)) atomicAdd(nsingular, 1);
        double* So = Sinv + (size_t)e * BB;
#pragma unroll
        for (int k = 0; k < BB; ++k) So[k] = I[k];
        if (e + 1 < nelem) {
            double* Wo = W + (size_t)e * BB;
#pragma unroll
            for (int i = 0; i < BS; ++i)
#pragma unroll
                for (int c = 0; c < BS; ++c) {
                    double sacc = 0.0;
#pragma unroll
                    for (int k = 0; k < BS; ++k) sacc += I[i * BS + k] * cU[k * BS + c];
                    Wp[i * BS + c] = sacc;
                    Wo[i * BS + c] = sacc;
                }
#pragma unroll
            for (int k = 0; k < BB; ++k) {
                cD[k] = nD[k];
                cL[k] = nL[k];
                cU[k] = nU[k];
            }
        }
    }
}

template <int BS>
__device__ void chain_solve(int nelem, int nslots, const double* J, const double* Sinv, const double* W,
                            const double* b, double* x) {
    constexpr int BB = BS * BS;
    double yp[BS] = {};
    double cL[BB], cS[BB], cb[BS], nL[BB], nS[BB], nb[BS];
    auto load = [&](int e, double (&l)[BB], double (&si)[BB], double (&bv)[BS]) {
        const double* L = J + ((size_t)e * nslots + 1) * BB;
#pragma unroll
        for (int k = 0; k < BB; ++k) {
            l[k] = L[k];
            si[k] = Sinv[(size_t)e * BB + k];
        }
#pragma unroll
        for (int k = 0; k < BS; ++k) bv[k] = b[(size_t)e * BS + k];
    };
    load(0, cL, cS, cb);
    for (int e = 0; e < nelem; ++e) {
        if (e + 1 < nelem) load(e + 1, nL, nS, nb);
        double t[BS];
#pragma unroll
        for (int i = 0; i < BS; ++i) {
            double sacc = cb[i];
            if (e > 0)
#pragma unroll
                for (int k = 0; k < BS; ++k) sacc -= cL[i * BS + k] * yp[k];
            t[i] = sacc;
        }
#pragma unroll
        for (int i = 0; i < BS; ++i) {
            double sacc = 0.0;
#pragma unroll
            for (int k = 0; k < BS; ++k) sacc += cS[i * BS + k] * t[k];
            yp[i] = sacc;
            x[(size_t)e * BS + i] = sacc;
        }
#pragma unroll
        for (int k = 0; k < BB; ++k) {
            cL[k] = nL[k];
            cS[k] = nS[k];
        }
#pragma unroll
        for (int k = 0; k < BS; ++k) cb[k] = nb[k];
    }
    // backward: x_e = y_e - W_e x_{e+1}; yp holds x_{n-1}
    double cW[BB], cy[BS], nW[BB], ny[BS];
    auto loadb = [&](int e, double (&w)[BB], double (&yv)[BS]) {
#pragma unroll
        for (int k = 0; k < BB; ++k) w[k] = W[(size_t)e * BB + k];
#pragma unroll
        for (int k = 0; k < BS; ++k) yv[k] = x[(size_t)e * BS + k];
    };
    if (nelem >= 2) loadb(nelem - 2, cW, cy);
    for (int e = nelem - 2; e >= 0; --e) {
        if (e >= 1) loadb(e - 1, nW, ny);
        double xe[BS];
#pragma unroll
        for (int i = 0; i < BS; ++i) {
            double sacc = cy[i];
#pragma unroll
            for (int k = 0; k < BS; ++k) sacc -= cW[i * BS + k] * yp[k];
            xe[i] = sacc;
        }
#pragma unroll
        for (int i = 0; i < BS; ++i) {
            yp[i] = xe[i];
            x[(size_t)e * BS + i] = xe[i];
        }
#pragma unroll
        for (int k = 0; k < BB; ++k) cW[k] = nW[k];
#pragma unroll
        for (int k = 0; k < BS; ++k) cy[k] = ny[k];
    }
}

template <int BS>
__global__ __launch_bounds__(64) void chain_factor_kernel(int n, int nslots, const double* J, double* Sinv, double* W,
                                                          int* nsingular) {
    if (threadIdx.x == 0) chain_factor<BS>(n, nslots, J, Sinv, W, nsingular);
}

template <int BS>
__global__ __launch_bounds__(64) void chain_solve_kernel(int n, int nslots, const double* J, const double* Sinv,
                                                         const double* W, const double* b, double* x) {
    if (threadIdx.x == 0) chain_solve<BS>(n, nslots, J, Sinv, W, b, x);
}

template <int BS>
__device__ __forceinline__ double largest(const double (&M)[BS * BS]) {
    double a = 0.0;
#pragma unroll
    for (int k = 0; k < BS * BS; ++k) a = fmax(a, fabs(M[k]));
    return a;
}

// workspace: head, D^-1 [entries][n], two sets of D, L, U, then A and C of each step
template <int BS>
__global__ __launch_bounds__(PCR_THREADS) void pcr_factor_kernel(int n, int nslots, const double* J, double* Sinv,
                                                                 double* work, int* nsingular) {
    constexpr int BB = BS * BS;
    __shared__ int chain;
    __shared__ double size[PCR_MAX_ROWS];  // largest entry a row's diagonal block had or lost (the row's thread's own)
    const size_t blk = (size_t)BB * n;
    double *I = work + PCR_HEAD, *cur = I + blk, *nxt = cur + 3 * blk, *AC = nxt + 3 * blk;
    const int tid = threadIdx.x;
    if (tid == 0) chain = 0;
    for (int e = tid; e < n; e += PCR_THREADS) {
        const double* Je = J + (size_t)e * nslots * BB;
#pragma unroll
        for (int k = 0; k < BB; ++k) {
            cur[(size_t)k * n + e] = Je[k];
            cur[blk + (size_t)k * n + e] = e > 0 ? Je[BB + k] : 0.0;
            cur[2 * blk + (size_t)k * n + e] = e + 1 < n ? Je[2 * BB + k] : 0.0;
        }
        size[e] = 0.0;
    }
    __syncthreads();
    for (int s = 1;; s <<= 1) {
        for (int e = tid; e < n; e += PCR_THREADS) {
            double M[BB], Inv[BB];
            get<BS>(cur, n, e, M);
            const bool ok = small_inverse<BS>(M, Inv);
            size[e] = fmax(size[e], largest<BS>(M));
            if (!ok || !(size[e] * largest<BS>(Inv) <= 1e10)) chain = 1;
            put<BS>(s < n ? I : Sinv, n, e, Inv);
        }
        __syncthreads();
        if (s >= n || chain) break;
        for (int e = tid; e < n; e += PCR_THREADS) {
            double X[BB], Y[BB], A[BB], T[BB], nD[BB], nO[BB];
            auto eliminate = [&](bool has, int f, int off, int other) {  // off: L or U of this row, other: of row f
#pragma unroll
                for (int k = 0; k < BB; ++k) A[k] = nO[k] = 0.0;
                if (!has) return;
                get<BS>(cur + off * blk, n, e, X);
                get<BS>(I, n, f, Y);
                mul<BS>(X, Y, A);
                get<BS>(cur + other * blk, n, f, X);
                mul<BS>(A, X, T);
#pragma unroll
                for (int k = 0; k < BB; ++k) nD[k] -= T[k];
                size[e] = fmax(size[e], largest<BS>(T));
                get<BS>(cur + off * blk, n, f, X);
                mul<BS>(A, X, T);
#pragma unroll
                for (int k = 0; k < BB; ++k) nO[k] = -T[k];
            };
            get<BS>(cur, n, e, nD);
            eliminate(e - s >= 0, e - s, 1, 2);
            put<BS>(AC, n, e, A);
            put<BS>(nxt + blk, n, e, nO);
            eliminate(e + s < n, e + s, 2, 1);
            put<BS>(AC + blk, n, e, A);
            put<BS>(nxt + 2 * blk, n, e, nO);
            put<BS>(nxt, n, e, nD);
        }
        __syncthreads();
        double* h = cur;
        cur = nxt;
        nxt = h;
        AC += 2 * blk;
    }
    if (tid == 0) {
        work[0] = chain;
        if (chain) chain_factor<BS>(n, nslots, J, Sinv, work + PCR_HEAD, nsingular);
    }
}

// A row a thread (512 threads leave a thread the registers of both blocks):
// bound by the latency of a step's loads of A and C and of one exchange
// through LDS.  The reduced blocks lose digits with the rows they span
// (residual 3e-13 of b at 256 rows, 4e-12 at 1024, along the chain 4e-16); a
// second pass on the residual of the first restores them.
template <int BS, int THREADS>
__global__ __launch_bounds__(THREADS) void pcr_solve_kernel(int n, int nslots, const double* J,
                                                                 const double* Sinv, const double* work,
                                                                 const double* b, double* x) {
    constexpr int BB = BS * BS;
    extern __shared__ double sb[];  // right-hand side [BS][n]
    if (work[0] != 0.0) {
        if (threadIdx.x == 0) chain_solve<BS>(n, nslots, J, Sinv, work + PCR_HEAD, b, x);
        return;
    }
    const int e = threadIdx.x;
    const bool row = e < n;
    const size_t blk = (size_t)BB * n;
    double t[BS], xe[BS];
#pragma unroll
    for (int i = 0; i < BS; ++i) {
        t[i] = row ? b[(size_t)e * BS + i] : 0.0;
        xe[i] = 0.0;
    }
    for (int pass = 0;; ++pass) {
        const double* AC = work + PCR_HEAD + 7 * blk;
        for (int s = 1; s < n; s <<= 1) {
            double A[BB], C[BB];
            if (row) {
#pragma unroll
                for (int i = 0; i < BS; ++i) sb[i * n + e] = t[i];
                get<BS>(AC, n, e, A);
                get<BS>(AC + blk, n, e, C);
            }
            __syncthreads();
            if (row) {
                const int m = e - s >= 0 ? e - s : e, p = e + s < n ? e + s : e;  // (A, C are zero there)
#pragma unroll
                for (int k = 0; k < BS; ++k) {
                    const double bm = sb[k * n + m], bp = sb[k * n + p];
#pragma unroll
                    for (int i = 0; i < BS; ++i) t[i] -= A[i * BS + k] * bm + C[i * BS + k] * bp;
                }
            }
            __syncthreads();
            AC += 2 * blk;
        }
        if (row) {
            double I[BB];
            get<BS>(Sinv, n, e, I);
#pragma unroll
            for (int i = 0; i < BS; ++i)
#pragma unroll
                for (int k = 0; k < BS; ++k) xe[i] += I[i * BS + k] * t[k];
        }
        if (pass == 1) break;
        // the residual of the first solve is the right-hand side of the second
        if (row) {
#pragma unroll
            for (int i = 0; i < BS; ++i) sb[i * n + e] = xe[i];
        }
        __syncthreads();
        if (row) {
#pragma unroll
            for (int i = 0; i < BS; ++i) t[i] = b[(size_t)e * BS + i];
#pragma unroll
            for (int slot = 0; slot < 3; ++slot) {
                const int f = slot == 0 ? e : slot == 1 ? e - 1 : e + 1;
                if (f < 0 || f >= n) continue;
                const double* Js = J + ((size_t)e * nslots + slot) * BB;
#pragma unroll
                for (int k = 0; k < BS; ++k) {
                    const double v = sb[k * n + f];
#pragma unroll
                    for (int i = 0; i < BS; ++i) t[i] -= Js[i * BS + k] * v;
                }
            }
        }
        __syncthreads();
    }
    if (row)
#pragma unroll
        for (int i = 0; i < BS; ++i) x[(size_t)e * BS + i] = xe[i];
}

// f(block size as a constant)
template <class F>
int with_size(int bs, F f) {
    using std::integral_constant;
    switch (bs) {
    case 1: f(integral_constant<int, 1>{}); break;
    case 2: f(integral_constant<int, 2>{}); break;
    case 3: f(integral_constant<int, 3>{}); break;
    case 4: f(integral_constant<int, 4>{}); break;
    case 5: f(integral_constant<int, 5>{}); break;
    default: return -1;
    }
    return (int)hipGetLastError();
}

// the solve has a row a thread in one workgroup.  Against the chain the gain
// grows with the rows (256 of 4 x 4: 80 for 709 us and 28 for 214 us), with four
// or fewer the chain is as short.
bool reduces(int nelem) { return nelem > 4 && nelem <= PCR_MAX_ROWS; }

}  // namespace

size_t line_small_work(int nelem, int bs) {
    const size_t blk = (size_t)bs * bs * nelem;
    if (!reduces(nelem)) return blk;
    size_t steps = 0;
    for (int s = 1; s < nelem; s <<= 1) ++steps;
    return PCR_HEAD + (7 + 2 * steps) * blk;
}

int line_small_factor(int nelem, int nslots, int bs, const double* J, double* Sinv, double* work, int* nsingular,
                      hipStream_t st) {
    return with_size(bs, [&](auto BS) {
        if (reduces(nelem))
            pcr_factor_kernel<BS()><<<1, PCR_THREADS, 0, st>>>(nelem, nslots, J, Sinv, work, nsingular);
        else
            chain_factor_kernel<BS()><<<1, 64, 0, st>>>(nelem, nslots, J, Sinv, work, nsingular);
    });
}

int line_small_solve(int nelem, int nslots, int bs, const double* J, const double* Sinv, const double* work,
                     const double* b, double* x, hipStream_t st) {
    return with_size(bs, [&](auto BS) {
        const int threads = (nelem + 63) & ~63;
        const size_t sh = (size_t)nelem * bs * sizeof(double);
        if (!reduces(nelem))
            chain_solve_kernel<BS()><<<1, 64, 0, st>>>(nelem, nslots, J, Sinv, work, b, x);
        else if (threads <= 512)
            pcr_solve_kernel<BS(), 512><<<1, threads, sh, st>>>(nelem, nslots, J, Sinv, work, b, x);
        else
            pcr_solve_kernel<BS(), PCR_MAX_ROWS><<<1, threads, sh, st>>>(nelem, nslots, J, Sinv, work, b, x);
    });
}

}  // namespace ice
