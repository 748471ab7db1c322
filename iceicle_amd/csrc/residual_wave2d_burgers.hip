// One-launch 2D residual (residual_wave2d.h): viscous Burgers.
#include "residual_wave2d.h"

namespace ice {

int wave2d_burgers(int p, const DevSpace& S, const PhysT<double>& ph, const DiscDev& dd, const double* U, double* R,
                   double* K, const StageComb<double>& cb, hipStream_t st) {
    return wave2d_order<Burgers<2, double>, double>(p, S, ph, dd, U, R, K, cb, st);
}

int wave2d_burgers(int p, const DevSpace& S, const PhysT<float>& ph, const DiscDev& dd, const double* U, double* R,
                   hipStream_t st) {
    return wave2d_order<Burgers<2, float>, double>(p, S, ph, dd, U, R, nullptr, StageComb<double>{}, st);
}

int wave2d_burgers(int p, const DevSpace& S, const PhysT<float>& ph, const DiscDev& dd, const float* U, double* R,
                   float* K, const StageComb<float>& cb, hipStream_t st) {
    return wave2d_order<Burgers<2, float>, float>(p, S, ph, dd, U, R, K, cb, st);
}

}  // namespace ice
