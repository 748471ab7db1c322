// One-launch 3D residual (residual_wave3d.h): Euler.
#include "residual_wave3d.h"

namespace ice {

template <class PH, class UT>
static int order3(int p, const DevSpace& S, const typename PH::Params& ph, const DiscDev& dd, const UT* U, double* R,
                  UT* K, const StageComb<UT>& cb, hipStream_t st) {
    switch (p) {
    case 2: return wave3d_launch<2, PH, UT>(S, ph, dd, U, R, K, cb, st);
    case 3: return wave3d_launch<3, PH, UT>(S, ph, dd, U, R, K, cb, st);
    default: return -1;
    }
}

int wave3d_euler(int p, const DevSpace& S, const PhysT<double>& ph, const DiscDev& dd, const double* U, double* R,
                 double* K, const StageComb<double>& cb, hipStream_t st) {
    return order3<NavierStokes<3, false, double>, double>(p, S, ph, dd, U, R, K, cb, st);
}

int wave3d_euler(int p, const DevSpace& S, const PhysT<float>& ph, const DiscDev& dd, const double* U, double* R,
                 hipStream_t st) {
    return order3<NavierStokes<3, false, float>, double>(p, S, ph, dd, U, R, nullptr, StageComb<double>{}, st);
}

int wave3d_euler(int p, const DevSpace& S, const PhysT<float>& ph, const DiscDev& dd, const float* U, double* R,
                 float* K, const StageComb<float>& cb, hipStream_t st) {
    return order3<NavierStokes<3, false, float>, float>(p, S, ph, dd, U, R, K, cb, st);
}

}  // namespace ice
