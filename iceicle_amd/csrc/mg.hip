// V-cycle of the agglomeration multigrid (preconditioner of the Newton solve).
//
// A level's cells have m x m blocks (m = 1..5) and few neighbours, so a
// pass over a coarse level is a launch of a few microseconds of latency
// whatever its size; what counts is how many passes and launches there are.
//  - Levels of a few thousand cells: a group of lanes owns a cell (one lane
//    a row, vectors exchanged by lane shuffles); the first two colours of a
//    forward sweep, the residual with its restriction, and the prolongation
//    with the next residual are one launch each.
//  - The levels that fit one workgroup's LDS (up to about 1300 cells in all
//    at m = 4) run to the bottom and back in one launch, vectors in LDS.
//  - After a symmetric sweep the rows of colour 0, solved last, have no
//    residual (unless a cell is its own neighbour, in a periodic direction of
//    one cell: the sweep leaves that coupling out, and the residual is formed
//    on every row); on the fine level that halves the residual, and after the
//    coarse correction x += P xc the residual is updated with the precomputed
//    J P (a sixteenth of the bytes at 16 nodes an element) instead of formed again.
// 2D NS P3 64 x 64, an iteration of GMRES with its operator: 710 -> 460 us
// (launches 60 -> 27; FP32 operator and FP16 fine sweeps, 5.2 TB/s, 180 us
// of it; tail 74 us, the levels above it 60 us).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mg.h"

namespace ice {
namespace {

template <int M>
constexpr int GROUP = M == 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : 8;  // lanes of a cell

// Cells of levels numbered colour by colour carry no colour arrays: cell k of
// a colour's list is k itself and colours compare as the offsets do, which
// leaves a pass one load (the neighbours' list) ahead of its data.
__device__ __forceinline__ int cell_of(const MGCells& L, int k) { return L.celems ? L.celems[k] : k; }
__device__ __forceinline__ bool before(const MGCells& L, int col, int colour) {
    return L.ecolor ? L.ecolor[col] < colour : col < L.coff[colour];
}
__device__ __forceinline__ bool after(const MGCells& L, int col, int colour) {
    return L.ecolor ? L.ecolor[col] > colour : col >= L.coff[colour + 1];
}

// sum over the columns of D of entry t held by the group's lane c
// (D: row r of the block's first column, the next columns n m entries on)
template <int M>
__device__ __forceinline__ double diag_mul(const MGCells& L, const float* __restrict__ D, double t) {
    constexpr int G = GROUP<M>;
    const int base = (threadIdx.x & 63) & ~(G - 1);
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < M; ++c) s += (double)D[(size_t)c * L.n * M] * __shfl(t, base + c);
    return s;
}

// row r of A_e,col y over the neighbours the filter admits
template <int M, int NS, class F, class Y>
__device__ __forceinline__ double row_sum(const MGCells& L, int e, int r, F admit, Y value) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int col = L.cols[(size_t)e * NS + k];
        if (col < 0 || !admit(k, col)) continue;
        const size_t a = ((size_t)k * M * L.n + e) * M + r, stride = (size_t)L.n * M;
#pragma unroll
        for (int c = 0; c < M; ++c) s += (double)L.A[a + c * stride] * value(col, c);
    }
    return s;
}

// one forward (y = D^-1 (rhs - L y)) or backward (y -= D^-1 U y) colour pass
template <int M, int NS, bool FWD>
__device__ __forceinline__ void colour_row(const MGCells& L, int colour, int e, int r, bool row, const double* rhs,
                                           double* y) {
    const int rr = row ? r : 0;
    const double s = (FWD && colour == 0)
                         ? 0.0
                         : row_sum<M, NS>(
                               L, e, rr,
                               [&](int k, int col) { return k > 0 && (FWD ? before(L, col, colour) : after(L, col, colour)); },
                               [&](int col, int c) { return y[(size_t)col * M + c]; });
    const size_t i = (size_t)e * M + rr;
    const double d = diag_mul<M>(L, L.Dinv + i, FWD ? rhs[i] - s : s);
    if (row) y[i] = FWD ? d : y[i] - d;
}

template <int M, int NS>
__global__ __launch_bounds__(256) void forward2_kernel(MGCells L, const double* __restrict__ rhs, double* __restrict__ y) {
    constexpr int G = GROUP<M>;
    const int idx = blockIdx.x * (256 / G) + threadIdx.x / G, r = threadIdx.x % G;
    if (idx >= L.coff[2]) return;
    const int e = cell_of(L, idx), rr = r < M ? r : 0;
    const size_t i = (size_t)e * M + rr;
    double t = rhs[i];
    if (idx >= L.coff[1]) {
        // colour 1: its colour-0 neighbours' values, formed again here
#pragma unroll
        for (int k = 1; k < NS; ++k) {
            const int col = L.cols[(size_t)e * NS + k];
            if (col < 0 || !before(L, col, 1)) continue;
            const size_t j = (size_t)col * M + rr;
            const double z = diag_mul<M>(L, L.Dinv + j, rhs[j]);
            t -= diag_mul<M>(L, L.A + ((size_t)k * M * L.n + e) * M + rr, z);
        }
    }
    const double d = diag_mul<M>(L, L.Dinv + i, t);
    if (r < M) y[i] = d;
}

template <int M, int NS, bool FWD>
__global__ __launch_bounds__(256) void colour_kernel(MGCells L, int colour, const double* __restrict__ rhs, double* y) {
    constexpr int G = GROUP<M>;
    const int idx = L.coff[colour] + blockIdx.x * (256 / G) + threadIdx.x / G, r = threadIdx.x % G;
    if (idx >= L.coff[colour + 1]) return;
    colour_row<M, NS, FWD>(L, colour, cell_of(L, idx), r, r < M, rhs, y);
}

template <int M, int NS>
__global__ __launch_bounds__(256) void residual_restrict_kernel(MGCells L, MGCells C, const double* __restrict__ b,
                                                                const double* __restrict__ x, double* __restrict__ bc) {
    constexpr int G = GROUP<M>;
    const int P = blockIdx.x * (256 / G) + threadIdx.x / G, r = threadIdx.x % G;
    if (P >= C.n || r >= M) return;
    double s = 0.0;
    for (int k = 0; k < 8; ++k) {
        const int e = C.children[(size_t)P * 8 + k];
        if (e < 0 || (L.settled && before(L, e, 1))) continue;
        s += b[(size_t)e * M + r] - row_sum<M, NS>(
                                        L, e, r, [](int, int) { return true; },
                                        [&](int col, int c) { return x[(size_t)col * M + c]; });
    }
    bc[(size_t)P * M + r] = s;
}

template <int M, int NS>
__global__ __launch_bounds__(256) void prolong_residual_kernel(MGCells L, const double* __restrict__ b,
                                                               const double* __restrict__ x,
                                                               const double* __restrict__ xc, double* __restrict__ r_) {
    constexpr int G = GROUP<M>;
    const int e = blockIdx.x * (256 / G) + threadIdx.x / G, r = threadIdx.x % G;
    if (e >= L.n || r >= M) return;
    r_[(size_t)e * M + r] = b[(size_t)e * M + r] -
                            row_sum<M, NS>(
                                L, e, r, [](int, int) { return true; },
                                [&](int col, int c) { return x[(size_t)col * M + c] + xc[(size_t)L.parent[col] * M + c]; });
}

__global__ void prolong_add_kernel(MGCells L, int m, const double* __restrict__ xc, const double* __restrict__ t,
                                   double* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= L.n * m) return;
    const int e = i / m, v = i - e * m;
    x[i] += xc[(size_t)L.parent[e] * m + v] + t[i];
}

// A64 [n][nslots][m][m] row-major -> A [nslots][m][n][m], D [n][m][m]
// column-major -> Dinv [m][n][m]
__global__ void pack_kernel(int n, int nslots, int m, const double* __restrict__ A64, const float* __restrict__ D,
                            float* __restrict__ A, float* __restrict__ Dinv) {
    const size_t row = (size_t)n * m, na = row * nslots * m, nd = row * m;
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < na + nd; t += (size_t)gridDim.x * blockDim.x) {
        const size_t u = t < na ? t : t - na;
        const int r = (int)(u % m), e = (int)(u / m % n), c = (int)(u / row % m), s = (int)(u / (row * m));
        if (t < na) A[t] = (float)A64[(((size_t)e * nslots + s) * m + r) * m + c];
        else Dinv[u] = D[((size_t)e * m + c) * m + r];
    }
}

constexpr int TAIL_THREADS = MG_DIRECT;

// The V-cycle of T's levels in one workgroup, three vectors a level in LDS:
// solution, right-hand side (later the correction), residual.
template <int M, int NS>
__global__ __launch_bounds__(TAIL_THREADS) void tail_kernel(MGTail T, const double* __restrict__ bin,
                                                            double* __restrict__ xout) {
    extern __shared__ double lds[];
    constexpr int G = GROUP<M>, CELLS = TAIL_THREADS / G;
    __shared__ double part[TAIL_THREADS];
    const int tid = threadIdx.x, g = tid / G, r = tid % G;
    const bool row = r < M;
    auto sweep = [&](const MGCells& L, const double* rhs, double* y) {
        for (int c = 0; c < L.ncol; ++c) {
            for (int k = L.coff[c] + g; k < L.coff[c + 1]; k += CELLS)
                colour_row<M, NS, true>(L, c, cell_of(L, k), r, row, rhs, y);
            __syncthreads();
        }
        for (int c = L.ncol - 2; c >= 0; --c) {
            for (int k = L.coff[c] + g; k < L.coff[c + 1]; k += CELLS)
                colour_row<M, NS, false>(L, c, cell_of(L, k), r, row, nullptr, y);
            __syncthreads();
        }
    };
    auto residual = [&](const MGCells& L, const double* b, const double* x, double* out, bool swept) {
        for (int e = g; e < L.n; e += CELLS) {
            if (!row) continue;
            out[e * M + r] = (swept && before(L, e, 1))
                                 ? 0.0
                                 : b[e * M + r] - row_sum<M, NS>(
                                                      L, e, r, [](int, int) { return true; },
                                                      [&](int col, int c) { return x[col * M + c]; });
        }
        __syncthreads();
    };
    double* x = lds;  // this level's vectors; the next level's follow
    for (int i = tid; i < T.lev[0].n * M; i += TAIL_THREADS) x[T.lev[0].n * M + i] = bin[i];
    __syncthreads();
    int l = 0;
    for (; l + 1 < T.nlev; ++l) {
        const MGCells& L = T.lev[l];
        const MGCells& C = T.lev[l + 1];
        double *b = x + L.n * M, *t = b + L.n * M, *xn = t + L.n * M;
        sweep(L, b, x);
        residual(L, b, x, t, L.settled);
        for (int i = tid; i < C.n * M; i += TAIL_THREADS) {
            const int P = i / M, v = i - P * M;
            double s = 0.0;
            for (int k = 0; k < 8; ++k) {
                const int c = C.children[(size_t)P * 8 + k];
                if (c >= 0) s += t[c * M + v];
            }
            xn[C.n * M + i] = s;
        }
        __syncthreads();
        x = xn;
    }
    {
        const MGCells& L = T.lev[l];
        const int n = L.n * M;
        double *b = x + n, *t = b + n;
        if (T.inv) {
            // rows in the threads' low part, columns split over the rest
            const int nr = (n + 63) & ~63, np = TAIL_THREADS / nr, i = tid % nr, p = tid / nr;
            double s = 0.0;
            if (p < np && i < n) {
#pragma unroll 16
                for (int j = p; j < n; j += np) s += T.inv[(size_t)j * n + i] * b[j];
            }
            part[tid] = s;
            __syncthreads();
            if (tid < n) {
                s = 0.0;
                for (int k = 0; k < np; ++k) s += part[k * nr + tid];
                x[tid] = s;
            }
            __syncthreads();
        } else {
            // no exact solve: eight more symmetric sweeps
            double* z = t + n;
            sweep(L, b, x);
            for (int it = 0; it < 8; ++it) {
                residual(L, b, x, t, false);
                sweep(L, t, z);
                for (int i = tid; i < n; i += TAIL_THREADS) x[i] += z[i];
                __syncthreads();
            }
        }
    }
    for (--l; l >= 0; --l) {
        const MGCells& L = T.lev[l];
        const double* xc = x;
        x -= 3 * L.n * M;
        double *b = x + L.n * M, *t = b + L.n * M;
        for (int i = tid; i < L.n * M; i += TAIL_THREADS) x[i] += xc[L.parent[i / M] * M + i % M];
        __syncthreads();
        residual(L, b, x, t, false);
        sweep(L, t, b);
        for (int i = tid; i < L.n * M; i += TAIL_THREADS) x[i] += b[i];
        __syncthreads();
    }
    for (int i = tid; i < T.lev[0].n * M; i += TAIL_THREADS) xout[i] = x[i];
}

// r = v - J x on the rows of elements of colour > 0, 0 on colour 0, with the
// rows' sums over the nodes b0[e][v]; one wave per element, blocks read as
// bsrT_wave_kernel
template <class T, int NS>
__global__ __launch_bounds__(256) void fine_residual_kernel(int nelem, int bs, int m, int lrg,
                                                            const int* __restrict__ cols,
                                                            const int* __restrict__ ecolor, const T* __restrict__ JT,
                                                            const double* __restrict__ x, const double* __restrict__ v,
                                                            double* __restrict__ r, double* __restrict__ b0) {
    constexpr int VEC = 16 / (int)sizeof(T);
    typedef T vec_t __attribute__((ext_vector_type(VEC)));
    const int lane = threadIdx.x & 63;
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= nelem) return;  // uniform across the wave
    const int rg = lane & ((1 << lrg) - 1), cg = lane >> lrg, CG = 64 >> lrg;
    double acc[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) acc[k] = 0.0;
    const bool live = ecolor[e] != 0;
    if (live) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int col = cols[(size_t)e * NS + s];
            if (col < 0) continue;
            const T* Jb = JT + ((size_t)e * NS + s) * bs * bs + rg * VEC;
            const double* xv = x + (size_t)col * bs;
#pragma unroll 4
            for (int c = cg; c < bs; c += CG) {
                const double xc = xv[c];
                const vec_t jv = *reinterpret_cast<const vec_t*>(Jb + (size_t)c * bs);
#pragma unroll
                for (int k = 0; k < VEC; ++k) acc[k] += (double)jv[k] * xc;
            }
        }
        for (int off = 1 << lrg; off < 64; off <<= 1)
#pragma unroll
            for (int k = 0; k < VEC; ++k) acc[k] += __shfl_xor(acc[k], off);
        const size_t g = (size_t)e * bs + rg * VEC;
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[k] = v[g + k] - acc[k];
    }
    if (cg == 0) {
        const size_t g = (size_t)e * bs + rg * VEC;
#pragma unroll
        for (int k = 0; k < VEC; ++k) r[g + k] = acc[k];
    }
    // entries k of a lane belong to variable k % m (m divides VEC)
    for (int w = 0; w < m; ++w) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < VEC; ++k) s += (k % m == w) ? acc[k] : 0.0;
        for (int off = 1; off < (1 << lrg); off <<= 1) s += __shfl_xor(s, off);
        if (lane == 0) b0[(size_t)e * m + w] = s;
    }
}

// out += P x0, r -= (J P) x0
template <int M, int NS>
__global__ __launch_bounds__(256) void fine_correct_kernel(int ntot, int bs, const int* __restrict__ cols,
                                                           const float* __restrict__ ap, const double* __restrict__ x0,
                                                           double* __restrict__ out, double* __restrict__ r) {
    const int g = blockIdx.x * 256 + threadIdx.x;
    if (g >= ntot) return;
    const int e = g / bs, i = g - e * bs;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int col = cols[(size_t)e * NS + k];
        if (col < 0) continue;
        const float* a = ap + ((size_t)e * NS + k) * bs * M + i;
#pragma unroll
        for (int w = 0; w < M; ++w) s += (double)a[(size_t)w * bs] * x0[(size_t)col * M + w];
    }
    r[g] -= s;
    out[g] += x0[(size_t)e * M + i % M];
}

// (nslots, m) of the discretizations: Burgers, and the systems of 1D, 2D, 3D
template <class F>
int dispatch(int nslots, int m, F f) {
    using std::integral_constant;
    if (nslots == 3 && m == 1) return f(integral_constant<int, 1>{}, integral_constant<int, 3>{});
    if (nslots == 3 && m == 3) return f(integral_constant<int, 3>{}, integral_constant<int, 3>{});
    if (nslots == 5 && m == 1) return f(integral_constant<int, 1>{}, integral_constant<int, 5>{});
    if (nslots == 5 && m == 4) return f(integral_constant<int, 4>{}, integral_constant<int, 5>{});
    if (nslots == 7 && m == 1) return f(integral_constant<int, 1>{}, integral_constant<int, 7>{});
    if (nslots == 7 && m == 5) return f(integral_constant<int, 5>{}, integral_constant<int, 7>{});
    return -1;
}

template <int M>
int group_grid(int cells) { return (cells * GROUP<M> + 255) / 256; }

}  // namespace

int mg_tail_bytes(int nlev, const int* cells, int m) {
    int s = cells[nlev - 1];  // the last level's sweeps without an exact solve take a fourth vector
    for (int l = 0; l < nlev; ++l) s += 3 * cells[l];
    return s * m * (int)sizeof(double);
}

int mg_tail_cycle(int nslots, int m, const MGTail& T, const double* b, double* x, hipStream_t st) {
    int cells[MG_MAX_LEVELS];
    for (int l = 0; l < T.nlev; ++l) cells[l] = T.lev[l].n;
    const int sh = mg_tail_bytes(T.nlev, cells, m);
    return dispatch(nslots, m, [&](auto M, auto NS) {
        tail_kernel<M(), NS()><<<1, TAIL_THREADS, sh, st>>>(T, b, x);
        return (int)hipGetLastError();
    });
}

int mg_pack(int n, int nslots, int m, const double* A64, const float* D, float* A, float* Dinv, hipStream_t st) {
    const size_t total = (size_t)n * m * m * (nslots + 1);
    pack_kernel<<<(unsigned)std::min<size_t>((total + 255) / 256, 4096), 256, 0, st>>>(n, nslots, m, A64, D, A, Dinv);
    return (int)hipGetLastError();
}

int mg_forward2(int nslots, int m, const MGCells& L, const double* rhs, double* y, hipStream_t st) {
    return dispatch(nslots, m, [&](auto M, auto NS) {
        forward2_kernel<M(), NS()><<<group_grid<M()>(L.coff[2]), 256, 0, st>>>(L, rhs, y);
        return (int)hipGetLastError();
    });
}

int mg_forward(int nslots, int m, const MGCells& L, int colour, const double* rhs, double* y, hipStream_t st) {
    return dispatch(nslots, m, [&](auto M, auto NS) {
        colour_kernel<M(), NS(), true>
            <<<group_grid<M()>(L.coff[colour + 1] - L.coff[colour]), 256, 0, st>>>(L, colour, rhs, y);
        return (int)hipGetLastError();
    });
}

int mg_backward(int nslots, int m, const MGCells& L, int colour, double* y, hipStream_t st) {
    return dispatch(nslots, m, [&](auto M, auto NS) {
        colour_kernel<M(), NS(), false>
            <<<group_grid<M()>(L.coff[colour + 1] - L.coff[colour]), 256, 0, st>>>(L, colour, nullptr, y);
        return (int)hipGetLastError();
    });
}

int mg_residual_restrict(int nslots, int m, const MGCells& L, const MGCells& C, const double* b, const double* x,
                         double* bc, hipStream_t st) {
    return dispatch(nslots, m, [&](auto M, auto NS) {
        residual_restrict_kernel<M(), NS()><<<group_grid<M()>(C.n), 256, 0, st>>>(L, C, b, x, bc);
        return (int)hipGetLastError();
    });
}

int mg_prolong_residual(int nslots, int m, const MGCells& L, const double* b, const double* x, const double* xc,
                        double* r, hipStream_t st) {
    return dispatch(nslots, m, [&](auto M, auto NS) {
        prolong_residual_kernel<M(), NS()><<<group_grid<M()>(L.n), 256, 0, st>>>(L, b, x, xc, r);
        return (int)hipGetLastError();
    });
}

int mg_prolong_add(int m, const MGCells& L, const double* xc, const double* t, double* x, hipStream_t st) {
    prolong_add_kernel<<<(L.n * m + 255) / 256, 256, 0, st>>>(L, m, xc, t, x);
    return (int)hipGetLastError();
}

bool mg_fine_covers(int bs, int m, int entry_bytes) {
    const int vec = 16 / entry_bytes, rg = bs / vec;
    return bs >= 16 && bs % vec == 0 && rg <= 64 && (rg & (rg - 1)) == 0 && vec % m == 0;
}

template <class T>
int mg_fine_residual(int nelem, int nslots, int bs, int m, const int* cols, const int* ecolor, const T* JT,
                     const double* x, const double* v, double* r, double* b0, hipStream_t st) {
    const int lrg = __builtin_ctz(bs / (16 / (int)sizeof(T))), grid = (nelem + 3) / 4;
    switch (nslots) {
    case 3: fine_residual_kernel<T, 3><<<grid, 256, 0, st>>>(nelem, bs, m, lrg, cols, ecolor, JT, x, v, r, b0); break;
    case 5: fine_residual_kernel<T, 5><<<grid, 256, 0, st>>>(nelem, bs, m, lrg, cols, ecolor, JT, x, v, r, b0); break;
    case 7: fine_residual_kernel<T, 7><<<grid, 256, 0, st>>>(nelem, bs, m, lrg, cols, ecolor, JT, x, v, r, b0); break;
    default: return -1;
    }
    return (int)hipGetLastError();
}
template int mg_fine_residual<float>(int, int, int, int, const int*, const int*, const float*, const double*,
                                     const double*, double*, double*, hipStream_t);
template int mg_fine_residual<_Float16>(int, int, int, int, const int*, const int*, const _Float16*, const double*,
                                        const double*, double*, double*, hipStream_t);

int mg_fine_correct(int nelem, int nslots, int bs, int m, const int* cols, const float* ap, const double* x0,
                    double* out, double* r, hipStream_t st) {
    const int ntot = nelem * bs, grid = (ntot + 255) / 256;
    return dispatch(nslots, m, [&](auto M, auto NS) {
        fine_correct_kernel<M(), NS()><<<grid, 256, 0, st>>>(ntot, bs, cols, ap, x0, out, r);
        return (int)hipGetLastError();
    });
}

}  // namespace ice
