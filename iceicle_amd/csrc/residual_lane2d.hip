// One-launch 2D residual by lanes (residual_lane2d.h): viscous Burgers.
#include "residual_lane2d.h"

namespace ice {

namespace {
template <class PH, class UT>
int order(int p, const DevSpace& S, const typename PH::Params& ph, const DiscDev& dd, const UT* U, double* R, UT* K,
          const StageComb<UT>& cb, hipStream_t st) {
    switch (p) {
    case 1: return lane2d_launch<1, PH, UT>(S, ph, dd, U, R, K, cb, st);
    case 2: return lane2d_launch<2, PH, UT>(S, ph, dd, U, R, K, cb, st);
    case 3: return lane2d_launch<3, PH, UT>(S, ph, dd, U, R, K, cb, st);
    case 4: return lane2d_launch<4, PH, UT>(S, ph, dd, U, R, K, cb, st);
    default: return -1;
    }
}
}  // namespace

int lane2d_burgers(int p, const DevSpace& S, const PhysT<double>& ph, const DiscDev& dd, const double* U, double* R,
                   double* K, const StageComb<double>& cb, hipStream_t st) {
    return order<Burgers<2, double>, double>(p, S, ph, dd, U, R, K, cb, st);
}

int lane2d_burgers(int p, const DevSpace& S, const PhysT<float>& ph, const DiscDev& dd, const double* U, double* R,
                   hipStream_t st) {
    return order<Burgers<2, float>, double>(p, S, ph, dd, U, R, nullptr, StageComb<double>{}, st);
}

int lane2d_burgers(int p, const DevSpace& S, const PhysT<float>& ph, const DiscDev& dd, const float* U, double* R,
                   float* K, const StageComb<float>& cb, hipStream_t st) {
    return order<Burgers<2, float>, float>(p, S, ph, dd, U, R, K, cb, st);
}

}  // namespace ice
