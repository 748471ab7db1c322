// One-launch 2D residual (residual_wave2d.h): compressible Navier-Stokes.
#include "residual_wave2d.h"

namespace ice {

int wave2d_ns(int p, const DevSpace& S, const PhysT<double>& ph, const DiscDev& dd, const double* U, double* R,
              double* K, const StageComb<double>& cb, hipStream_t st) {
    return wave2d_order<NavierStokes<2, true, double>, double>(p, S, ph, dd, U, R, K, cb, st);
}

int wave2d_ns(int p, const DevSpace& S, const PhysT<float>& ph, const DiscDev& dd, const double* U, double* R,
              hipStream_t st) {
    return wave2d_order<NavierStokes<2, true, float>, double>(p, S, ph, dd, U, R, nullptr, StageComb<double>{}, st);
}

int wave2d_ns(int p, const DevSpace& S, const PhysT<float>& ph, const DiscDev& dd, const float* U, double* R,
              float* K, const StageComb<float>& cb, hipStream_t st) {
    return wave2d_order<NavierStokes<2, true, float>, float>(p, S, ph, dd, U, R, K, cb, st);
}

}  // namespace ice
