// Multigrid levels as the device kernels see them.
#pragma once
#include <hip/hip_runtime.h>

namespace ice {

constexpr int MG_MAX_LEVELS = 16, MG_MAX_COLOURS = 8;
constexpr int MG_DIRECT = 1024;  // unknowns of a last level solved exactly, at most: one a thread of the tail

// n cells with m x m blocks in the Jacobian's slots (slot 0 the cell itself),
// blocks and factored diagonals FP32 with the cells' rows contiguous, so that
// consecutive lanes read consecutive entries
struct MGCells {
    int n, ncol;
    const int* cols;      // [n][nslots]
    const float* A;       // [nslots][m columns][n][m rows]
    const float* Dinv;    // [m columns][n][m rows]
    const int* ecolor;    // colours, and cells grouped by colour; null on levels
    const int* celems;    // whose cells are numbered colour by colour
    int coff[MG_MAX_COLOURS + 1];
    const int* children;  // [n][8] cells of the finer level
    const int* parent;    // [n] cell of the coarser level
    bool settled;         // a symmetric sweep leaves colour 0 no residual (no cell is its own neighbour)
};

// The levels one workgroup takes through a V-cycle
struct MGTail {
    int nlev;
    MGCells lev[MG_MAX_LEVELS];
    const double* inv;    // dense inverse of the last level (column-major, up to MG_DIRECT unknowns), or null
};

// the blocks' FP32 copies in that layout, from row-major FP64 blocks and
// column-major factored diagonals
int mg_pack(int n, int nslots, int m, const double* A64, const float* D, float* A, float* Dinv, hipStream_t st);
int mg_tail_bytes(int nlev, const int* cells, int m);  // LDS of a tail with these levels
int mg_tail_cycle(int nslots, int m, const MGTail& T, const double* b, double* x, hipStream_t st);
// y = the first two colours of a forward sweep
int mg_forward2(int nslots, int m, const MGCells& L, const double* rhs, double* y, hipStream_t st);
// y: one colour's forward value, one colour's backward update
int mg_forward(int nslots, int m, const MGCells& L, int colour, const double* rhs, double* y, hipStream_t st);
int mg_backward(int nslots, int m, const MGCells& L, int colour, double* y, hipStream_t st);
// coarse right-hand side: the residual b - A x of a completed sweep, restricted
int mg_residual_restrict(int nslots, int m, const MGCells& L, const MGCells& C, const double* b, const double* x,
                         double* bc, hipStream_t st);
// r = b - A (x + P xc)
int mg_prolong_residual(int nslots, int m, const MGCells& L, const double* b, const double* x, const double* xc,
                        double* r, hipStream_t st);
// x += P xc + t
int mg_prolong_add(int m, const MGCells& L, const double* xc, const double* t, double* x, hipStream_t st);
// fine level: r = v - J x of a completed sweep that leaves colour 0 no residual
// (it is not formed there) and its element sums b0; then out += P x0,
// r -= (J P) x0
template <class T>
int mg_fine_residual(int nelem, int nslots, int bs, int m, const int* cols, const int* ecolor, const T* JT,
                     const double* x, const double* v, double* r, double* b0, hipStream_t st);
int mg_fine_correct(int nelem, int nslots, int bs, int m, const int* cols, const float* ap, const double* x0,
                    double* out, double* r, hipStream_t st);
bool mg_fine_covers(int bs, int m, int entry_bytes);

}  // namespace ice
