"""Scalar 2D residual by lanes, taken for many elements, against the wave
kernel taken for few (P4, which the lanes always take: in other places of a
wave): a space of copies of one small mesh has the small mesh's residual in
every copy.

The two differ in the order of sums only: FP64 within 1e-12 of the largest
entry, and so with FP32 fluxes but for an FP32 rounding of the point values
(1e-5); a stage likewise.

And the lanes at every order against the CPU oracle: oblique boundary edges, a
source term, a viscosity of each instance, steps at a CFL number."""
import numpy as np
import pytest

from iceicle_amd import abi
from tests import cases

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

D, P, N = "DIRICHLET", "PERIODIC", "NEUMANN"
MIN = {1: 6400, 2: 9216, 3: 25600, 4: 1000}  # elements from which the lanes are taken


def _spaces(order, nel, bc, copies):
    from iceicle_amd import engine
    m = abi.mesh_desc(2, nel, [0.0, 0.0], [1.0, 0.8], bc, bcflag=[0, 1, 1, 0], periodic_mode=abi.PERIODIC_COUPLED)
    m = abi.mesh_desc(2, nel, [0.0, 0.0], [1.0, 0.8], bc, bcflag=[0, 1, 1, 0], periodic_mode=abi.PERIODIC_COUPLED,
                      coord=cases.perturbed_coords(m, 0.1, 3))
    return [(engine.FESpace([m] * k, order), k) for k in (1, copies)]


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("nel,bc", [([13, 9], [P, P, P, P]), ([8, 16], [D, N, N, D]), ([5, 7], [P, D, P, N])])
def test_copies(order, nel, bc):
    from iceicle_amd import engine
    ne = nel[0] * nel[1]
    prm = cases.burgers_params(2, mu=0.02, a=(0.3, -0.2, 0.0), b=(1.0, 0.7, 0.0))
    rng = np.random.default_rng(order)
    u1 = rng.uniform(-1.0, 1.0, ne * (order + 1) ** 2)
    out = {}
    for space, k in _spaces(order, nel, bc, -(-MIN[order] // ne)):
        assert (space.nelem >= MIN[order]) == (k > 1)
        disc = engine.ConservationLawDDG(space, prm)
        u = torch.from_numpy(np.tile(u1, k)).cuda()
        r = torch.full_like(u, float("nan"))
        rm = torch.full_like(u, float("nan"))
        engine.form_residual(space, disc, u, r)
        engine.form_residual(space, disc, u, rm, precision="mixed")
        v = u.clone()
        st = engine.ExplicitStepper(disc, abi.stepper_desc(abi.STEP_RK3_SSP, dt=1e-3, ntime=2))
        w = u.float()
        for _ in range(2):
            st.step(v)
            st.step(w)
        out[k] = [x.view(k, -1).cpu().numpy() for x in (r, rm, v, w)]
    (small, big) = out[1], out[max(out)]
    for a, b, tol in zip(small, big, (1e-12, 1e-5, 1e-12, 1e-5)):
        err = np.abs(b - a).max() / np.abs(a).max()
        print(f"P{order} {nel} {bc}: {err:.1e}", flush=True)
        assert err <= tol


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("bc", [[D, D, D, D], [N, D, "EXTRAPOLATION", D]])
def test_oblique_sides(order, bc):
    """A tapered, sheared domain: on an oblique boundary edge the DDG distance
    varies from point to point.  Every copy against the CPU oracle of one, at
    the bars of the other residual tests (1e-12; FP32 fluxes 2e-5)."""
    from iceicle_amd import engine
    from oracle.oracle import Oracle
    nel = [7, 5]
    m = abi.mesh_desc(2, nel, [0.0, 0.0], [1.0, 0.8], bc)
    x, y = cases.perturbed_coords(m, 0.1, 3).T
    coord = np.ascontiguousarray(np.stack([x + 0.3 * y + 0.2 * x * y, y - 0.4 * x + 0.3 * x * y], axis=1))
    m = abi.mesh_desc(2, nel, [0.0, 0.0], [1.0, 0.8], bc, bcflag=[0, 1, 1, 0], coord=coord)
    prm = cases.burgers_params(2, mu=0.05, a=(0.3, -0.2, 0.0), b=(1.0, 0.7, 0.0))
    o = Oracle(m, abi.space_desc(order), prm)
    u1 = np.random.default_rng(order).uniform(-1.0, 1.0, o.size)
    ref = o.residual(u1)
    copies = -(-MIN[order] // 35) if order < 4 else 3
    disc = engine.ConservationLawDDG(engine.FESpace([m] * copies, order), prm)
    u = torch.from_numpy(np.tile(u1, copies)).cuda()
    for precision, tol in (("fp64", 1e-12), ("mixed", 2e-5)):
        r = torch.full_like(u, float("nan"))
        engine.form_residual(disc.space, disc, u, r, precision=precision)
        err = np.abs(r.view(copies, -1).cpu().numpy() - ref).max() / np.abs(ref).max()
        print(f"P{order} {bc} {precision}: {err:.1e}", flush=True)
        assert err <= tol


@pytest.mark.parametrize("order", [1, 2, 3, 4])
def test_source_and_element_viscosity(order):
    """A source term and a viscosity of each copy, every copy against the CPU
    oracle with its viscosity; an odd element count leaves a wave's 16 partly
    empty."""
    from iceicle_amd import engine
    from oracle.oracle import Oracle
    nel, bc = [5, 3], [D, P, N, P]
    m = abi.mesh_desc(2, nel, [0.0, 0.0], [1.0, 0.8], bc, periodic_mode=abi.PERIODIC_COUPLED)
    coord = cases.perturbed_coords(m, 0.15, 3)
    m = abi.mesh_desc(2, nel, [0.0, 0.0], [1.0, 0.8], bc, bcflag=[0, 1, 1, 0], periodic_mode=abi.PERIODIC_COUPLED,
                      coord=coord)
    copies = -(-MIN[order] // 15) | 1
    mu = [0.005, 0.03, 0.2]
    prm = cases.burgers_params(2, a=(0.3, -0.2, 0.0), b=(1.0, 0.7, 0.0))
    prm.source = abi.Field.make("SINUSOIDS", [2, 3.0, 1, 2, 0, -2.0, 2, 1, 0])
    u1 = np.random.default_rng(order).uniform(-1.0, 1.0, 15 * (order + 1) ** 2)
    ref = []
    for v in mu:
        prm.mu = v
        ref.append(Oracle(m, abi.space_desc(order), prm).residual(u1))
    disc = engine.ConservationLawDDG(engine.FESpace([m] * copies, order), prm)
    which = np.arange(copies) % 3
    disc.set_element_viscosity(np.repeat(np.array(mu)[which], 15))
    u = torch.from_numpy(np.tile(u1, copies)).cuda()
    for precision, tol in (("fp64", 1e-12), ("mixed", 2e-5)):
        r = torch.full_like(u, float("nan"))
        engine.form_residual(disc.space, disc, u, r, precision=precision)
        got = r.view(copies, -1).cpu().numpy()
        err = max(np.abs(got[which == k] - ref[k]).max() / np.abs(ref[k]).max() for k in range(3))
        print(f"P{order} {precision}: {err:.1e}", flush=True)
        assert err <= tol


@pytest.mark.parametrize("order,nel", [(1, [83, 79]), (2, [101, 93]), (3, [161, 160]), (4, [13, 9])])
def test_cfl_steps(order, nel):
    """Steps whose size comes from the wave speeds the lanes find, against the
    oracle's: the same times to rounding and states to 1e-12."""
    from iceicle_amd import engine
    from oracle.oracle import Oracle
    assert nel[0] * nel[1] >= MIN[order] or order == 4
    m = abi.mesh_desc(2, nel, [0.0, 0.0], [1.0, 1.0], [P] * 4, periodic_mode=abi.PERIODIC_COUPLED)
    prm = cases.burgers_params(2, mu=1e-3, a=(0.3, -0.2, 0.0), b=(1.0, 0.7, 0.0))
    o = Oracle(m, abi.space_desc(order), prm)
    u0 = o.project(abi.Field.make("SINUSOIDS", [2, 0.7, 1, 0, 0, -0.4, 1, 1, 0]))
    ref, n_ref, t_ref = o.rk_solve(u0, kind=0, cfl=0.2, ntime=4)
    u = torch.from_numpy(u0).cuda()
    disc = engine.ConservationLawDDG(engine.FESpace(m, order), prm)
    n, t = engine.ExplicitStepper(disc, abi.stepper_desc(abi.STEP_RK3_SSP, cfl=0.2, ntime=4)).solve(u)
    err = cases.rel_inf(u.cpu().numpy(), ref)
    print(f"P{order}: t {t:.6e} ({t_ref:.6e}) err {err:.1e}", flush=True)
    assert n == n_ref == 4 and abs(t - t_ref) <= 1e-13 * t_ref and err <= 1e-12
