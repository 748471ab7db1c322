// Flux parameters shared by the host engine and the device kernels.
#pragma once
#include "../../include/iceicle_amd.h"

namespace ice {

// Parameters of every flux family, flattened for a kernel argument, in the
// arithmetic type R of the kernels that use them.
template <class R>
struct PhysT {
    // Burgers (BurgersCoefficients, burgers.hpp:14-40)
    R mu;
    R a[3];
    R b[3];
    // Navier-Stokes (Physics + CaloricallyPerfectEoS + Nondimensionalization)
    R gamma;
    R Pr;
    R Re, Eu, e_coeff;
    R T_coeff;           // cp * ref.T * ref.rho / ref.p
    int visc_kind;
    R visc_mu;
    R mu_ratio, T0r, Tsr;  // DimensionlessSutherlands ratios
    R isoT[ICE_MAX_BCFLAG];
    R fs_rho, fs_u, fs_dir[3], fs_T;
    int textbook_energy;
    // ConservationLawDDG
    R sigma_ic;
    R sigma_face, sigma_bdy;  // DDGIC factors per interior side and on Dirichlet faces
    int ic_mirror;            // DDGIC test gradients averaged with the mirror point's
    R beta0, beta1, beta0_bdy;
    // parameter-only factors of the flux formulas, computed once on the host
    // (set_derived) so the pointwise fluxes multiply instead of divide
    R p_fac;        // (gamma - 1) / (e_coeff Eu): p = p_fac rho e
    R T_fac;        // gamma / ((gamma - 1) T_coeff): T = T_fac p / rho
    R inv_e_coeff;  // 1 / e_coeff
    R g_over_Pr;    // gamma / Pr
    R inv_Re;       // 1 / Re
    R inv_gamma;    // 1 / gamma
    R vl_fac;       // 1 / (2 (gamma^2 - 1)), VanLeer energy split
};
using PhysParams = PhysT<double>;

// fill the derived factors from the primary parameters
inline void set_derived(PhysParams& p) {
    p.p_fac = (p.gamma - 1) / (p.e_coeff * p.Eu);
    p.T_fac = p.gamma / ((p.gamma - 1) * p.T_coeff);
    p.inv_e_coeff = 1.0 / p.e_coeff;
    p.g_over_Pr = p.gamma / p.Pr;
    p.inv_Re = 1.0 / p.Re;
    p.inv_gamma = 1.0 / p.gamma;
    p.vl_fac = 1.0 / (2 * (p.gamma * p.gamma - 1));
}

// the same parameters rounded to another arithmetic type
template <class R>
inline PhysT<R> phys_cast(const PhysParams& p) {
    PhysT<R> q;
    q.mu = (R)p.mu;
    for (int k = 0; k < 3; ++k) {
        q.a[k] = (R)p.a[k];
        q.b[k] = (R)p.b[k];
        q.fs_dir[k] = (R)p.fs_dir[k];
    }
    q.gamma = (R)p.gamma;
    q.Pr = (R)p.Pr;
    q.Re = (R)p.Re;
    q.Eu = (R)p.Eu;
    q.e_coeff = (R)p.e_coeff;
    q.T_coeff = (R)p.T_coeff;
    q.visc_kind = p.visc_kind;
    q.visc_mu = (R)p.visc_mu;
    q.mu_ratio = (R)p.mu_ratio;
    q.T0r = (R)p.T0r;
    q.Tsr = (R)p.Tsr;
    for (int k = 0; k < ICE_MAX_BCFLAG; ++k) q.isoT[k] = (R)p.isoT[k];
    q.fs_rho = (R)p.fs_rho;
    q.fs_u = (R)p.fs_u;
    q.fs_T = (R)p.fs_T;
    q.textbook_energy = p.textbook_energy;
    q.sigma_ic = (R)p.sigma_ic;
    q.sigma_face = (R)p.sigma_face;
    q.sigma_bdy = (R)p.sigma_bdy;
    q.ic_mirror = p.ic_mirror;
    q.beta0 = (R)p.beta0;
    q.beta1 = (R)p.beta1;
    q.beta0_bdy = (R)p.beta0_bdy;
    q.p_fac = (R)p.p_fac;
    q.T_fac = (R)p.T_fac;
    q.inv_e_coeff = (R)p.inv_e_coeff;
    q.g_over_Pr = (R)p.g_over_Pr;
    q.inv_Re = (R)p.inv_Re;
    q.inv_gamma = (R)p.inv_gamma;
    q.vl_fac = (R)p.vl_fac;
    return q;
}

}  // namespace ice
