// Block tridiagonal factorisation and solve for blocks of up to LINE_SMALL
// rows (line preconditioner)
#pragma once
#include <hip/hip_runtime.h>

namespace ice {

constexpr int LINE_SMALL = 5;

size_t line_small_work(int nelem, int bs);  // doubles of `work`
int line_small_factor(int nelem, int nslots, int bs, const double* J, double* Sinv, double* work, int* nsingular,
                      hipStream_t st);
int line_small_solve(int nelem, int nslots, int bs, const double* J, const double* Sinv, const double* work,
                     const double* b, double* x, hipStream_t st);

}  // namespace ice
