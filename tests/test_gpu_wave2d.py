"""One-launch 2D residual (P1-P3): element counts that leave a wave's four
elements partly empty, meshes one element wide, against the CPU oracle; and
the fused Runge-Kutta stages against the residual and inverse mass entry
points.  Tolerance 1e-12 of the largest entry, the FP64 parity bar of the
residual path; a step adds rounding of the stage sums only (1e-13)."""
import numpy as np
import pytest

from iceicle_amd import abi
from tests import cases

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

BCT = ["DIRICHLET", "SLIP_WALL", "EXTRAPOLATION", "NO_SLIP_ISOTHERMAL"]


def _params(flux):
    if flux == abi.FLUX_BURGERS:
        return cases.burgers_params(2, a=(0.3, -0.2, 0))
    return cases.ns_params(2, flux=flux)


def _mesh(nel, flux, periodic):
    bct = ["PERIODIC"] * 4 if periodic else (BCT if flux != abi.FLUX_BURGERS else ["DIRICHLET", "NEUMANN",
                                                                                   "EXTRAPOLATION", "DIRICHLET"])
    mode = abi.PERIODIC_COUPLED if periodic else abi.PERIODIC_REFERENCE
    m = abi.mesh_desc(2, nel, [0.0, 0.0], [1.0, 1.0], bct, periodic_mode=mode)
    c = cases.perturbed_coords(m, 0.15, 5)
    return abi.mesh_desc(2, nel, [0.0, 0.0], [1.0, 1.0], bct, periodic_mode=mode, coord=c)


@pytest.mark.parametrize("flux", [abi.FLUX_BURGERS, abi.FLUX_NAVIER_STOKES, abi.FLUX_EULER])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("nel,periodic", [([1, 1], False), ([1, 3], True), ([5, 1], True), ([3, 7], False),
                                          ([9, 2], True)])
def test_residual_element_remainders(flux, order, nel, periodic):
    from iceicle_amd import engine
    from oracle.oracle import Oracle
    m, p = _mesh(nel, flux, periodic), _params(flux)
    o = Oracle(m, abi.space_desc(order), p)
    u = cases.random_state(flux, 2, o.nelem, o.nbasis, 7)
    ref = o.residual(u)
    space = engine.FESpace(m, order)
    disc = engine.ConservationLawDDG(space, p)
    ud = torch.from_numpy(u).cuda()
    r = torch.full((u.size + 64,), float("nan"), dtype=torch.float64, device="cuda")
    engine.form_residual(space, disc, ud, r[:u.size])
    assert cases.rel_inf(r[:u.size].cpu().numpy(), ref) <= 1e-12
    assert bool(torch.isnan(r[u.size:]).all())  # nothing stored beyond the last element
    # mixed: FP32 fluxes of FP64 states and jumps, 2e-5 as the other mixed tests
    engine.form_residual(space, disc, ud, r[:u.size], precision="mixed")
    assert cases.rel_inf(r[:u.size].cpu().numpy(), ref) <= 2e-5


@pytest.mark.parametrize("flux", [abi.FLUX_BURGERS, abi.FLUX_NAVIER_STOKES])
@pytest.mark.parametrize("order", [1, 2, 3])
def test_fused_stages(flux, order):
    from iceicle_amd import engine
    m, p = _mesh([7, 3], flux, True), _params(flux)
    space = engine.FESpace(m, order)
    disc = engine.ConservationLawDDG(space, p)
    u0 = torch.from_numpy(cases.random_state(flux, 2, space.nelem, space.nbasis, 3)).cuda()
    dt = 1e-4
    for fp32 in (False, True):
        u = u0.float() if fp32 else u0.clone()
        st = engine.ExplicitStepper(disc, abi.stepper_desc(abi.STEP_RK3_SSP, dt=dt, ntime=10))
        st.step(u)
        r, k = torch.empty_like(u0), [torch.empty_like(u0) for _ in range(3)]
        x0 = u0.float().double() if fp32 else u0
        x = x0
        for s, c in enumerate(([1.0], [0.25, 0.25], [1 / 6, 1 / 6, 2 / 3])):
            engine.form_residual(space, disc, x.float() if fp32 else x, r, precision="mixed" if fp32 else "fp64")
            engine.mass_inverse_apply(disc, r, k[s])
            if fp32:
                k[s] = k[s].float().double()
            x = x0 + dt * sum(ci * ki for ci, ki in zip(c, k))
            x = x.float().double() if fp32 else x
        # FP32 states: at most two roundings of a stage's increments apart
        tol = 4 * 2.0 ** -24 if fp32 else 1e-13
        err = float((u.double() - x).abs().max() / x.abs().max())
        assert err <= tol, err


@pytest.mark.parametrize("nel", [[157, 152], [161, 150], [190, 189], [191, 189]])
def test_ns_p1_on_many_elements(nel):
    """P1 Navier-Stokes on both sides of the element counts from which its
    stages (24000) and its residual (36000) take three launches: residuals and
    in-place residuals against the oracle, an FP64 step against the oracle's,
    an FP32 step within two roundings of a stage's increments of it."""
    from iceicle_amd import engine
    from oracle.oracle import Oracle
    m, p = _mesh(nel, abi.FLUX_NAVIER_STOKES, False), _params(abi.FLUX_NAVIER_STOKES)
    o = Oracle(m, abi.space_desc(1), p)
    u = cases.random_state(abi.FLUX_NAVIER_STOKES, 2, o.nelem, 4, 7).astype(np.float32).astype(np.float64)
    ref = o.residual_parallel(u)
    space = engine.FESpace(m, 1)
    disc = engine.ConservationLawDDG(space, p)
    ud = torch.from_numpy(u).cuda()
    for precision, tol in (("fp64", 1e-12), ("mixed", 2e-5)):
        r, w = torch.full_like(ud, float("nan")), ud.clone()
        engine.form_residual(space, disc, ud, r, precision=precision)
        engine.form_residual(space, disc, w, w, precision=precision)
        err = cases.rel_inf(r.cpu().numpy(), ref)
        print(f"{nel} {precision}: {err:.1e}", flush=True)
        assert err <= tol and torch.equal(r, w)
    dt = 1e-6
    v = o.rk_solve(u, kind=0, dt=dt, ntime=1)[0]
    for x, tol in ((ud.clone(), 1e-13), (ud.float(), 4 * 2.0 ** -24)):
        engine.ExplicitStepper(disc, abi.stepper_desc(abi.STEP_RK3_SSP, dt=dt, ntime=1)).step(x)
        err = cases.rel_inf(x.double().cpu().numpy(), v)
        print(f"{nel} {x.dtype} step: {err:.1e}", flush=True)
        assert err <= tol
