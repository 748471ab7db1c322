"""One-launch 3D Euler residual (P2, P3): element counts that leave a wave's
four elements partly empty, layers that divide unevenly into workgroups,
meshes one element wide, boundaries of every Euler type, against the CPU
oracle; and the fused Runge-Kutta stages against the residual and inverse
mass entry points.  Tolerance 1e-12 of the largest entry, the FP64 parity bar
of the residual path (a step adds rounding of the stage sums only: 1e-13)."""
import pytest

from iceicle_amd import abi
from tests import cases

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

WALLS = ["SLIP_WALL", "RIEMANN", "DIRICHLET", "EXTRAPOLATION", "SLIP_WALL", "DIRICHLET"]
MIXED_BCT = ["PERIODIC", "SLIP_WALL", "PERIODIC", "PERIODIC", "RIEMANN", "PERIODIC"]


def _mesh(nel, bct):
    mode = abi.PERIODIC_COUPLED if "PERIODIC" in bct else abi.PERIODIC_REFERENCE
    m = abi.mesh_desc(3, nel, [0.0] * 3, [1.0, 1.2, 0.9], bct, periodic_mode=mode)
    c = cases.perturbed_coords(m, 0.12, 5)
    return abi.mesh_desc(3, nel, [0.0] * 3, [1.0, 1.2, 0.9], bct, periodic_mode=mode, coord=c)


@pytest.mark.parametrize("order", [2, 3])
@pytest.mark.parametrize("nel,bct", [([1, 1, 1], WALLS), ([1, 1, 1], ["PERIODIC"] * 6), ([3, 1, 2], ["PERIODIC"] * 6),
                                     ([5, 3, 3], MIXED_BCT), ([2, 3, 5], WALLS), ([7, 6, 5], ["PERIODIC"] * 6)])
def test_residual_element_remainders(order, nel, bct):
    from iceicle_amd import engine
    from oracle.oracle import Oracle
    m, p = _mesh(nel, bct), cases.ns_params(3, flux=abi.FLUX_EULER)
    o = Oracle(m, abi.space_desc(order), p)
    u = cases.random_state(abi.FLUX_EULER, 3, o.nelem, o.nbasis, 7)
    ref = o.residual(u)
    space = engine.FESpace(m, order)
    disc = engine.ConservationLawDDG(space, p)
    ud = torch.from_numpy(u).cuda()
    r = torch.full((u.size + 64,), float("nan"), dtype=torch.float64, device="cuda")
    engine.form_residual(space, disc, ud, r[:u.size])
    assert cases.rel_inf(r[:u.size].cpu().numpy(), ref) <= 1e-12
    assert bool(torch.isnan(r[u.size:]).all())  # nothing stored beyond the last element
    # mixed: FP32 fluxes of FP64 states, 2e-5 as the other mixed tests
    engine.form_residual(space, disc, ud, r[:u.size], precision="mixed")
    assert cases.rel_inf(r[:u.size].cpu().numpy(), ref) <= 2e-5


@pytest.mark.parametrize("order", [2, 3])
@pytest.mark.parametrize("nel,bct", [([18, 17, 3], MIXED_BCT), ([16, 16, 4], ["PERIODIC"] * 6), ([17, 31, 2], WALLS),
                                     ([1, 1, 333], ["PERIODIC"] * 6), ([2, 3, 150], WALLS)])
def test_layers_and_columns(order, nel, bct):
    """Layers of more than one strip of 16 workgroups (the last one narrower,
    layers that do not start at a workgroup) and of exactly one, thin columns."""
    from iceicle_amd import engine
    from oracle.oracle import Oracle
    m, p = _mesh(nel, bct), cases.ns_params(3, flux=abi.FLUX_EULER)
    o = Oracle(m, abi.space_desc(order), p)
    u = cases.random_state(abi.FLUX_EULER, 3, o.nelem, o.nbasis, 7)
    ref = o.residual_parallel(u)
    space = engine.FESpace(m, order)
    disc = engine.ConservationLawDDG(space, p)
    r = torch.full((u.size,), float("nan"), dtype=torch.float64, device="cuda")
    engine.form_residual(space, disc, torch.from_numpy(u).cuda(), r)
    assert cases.rel_inf(r.cpu().numpy(), ref) <= 1e-12


@pytest.mark.parametrize("order", [2, 3])
@pytest.mark.parametrize("bct", [["PERIODIC"] * 6, MIXED_BCT])
def test_fused_stages(order, bct):
    from iceicle_amd import engine
    m, p = _mesh([5, 3, 3], bct), cases.ns_params(3, flux=abi.FLUX_EULER)
    space = engine.FESpace(m, order)
    disc = engine.ConservationLawDDG(space, p)
    u0 = torch.from_numpy(cases.random_state(abi.FLUX_EULER, 3, space.nelem, space.nbasis, 3)).cuda()
    dt = 1e-4
    for fp32 in (False, True):
        u = u0.float() if fp32 else u0.clone()
        st = engine.ExplicitStepper(disc, abi.stepper_desc(abi.STEP_RK3_SSP, dt=dt, ntime=1))
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
        done = u.clone()
        st.step(u)  # the run is over: nothing moves
        assert torch.equal(u, done)
