"""Block rows in one launch: the tile edges of its matrix products (orders
whose nodes, columns or face points are not multiples of 16 and 4) against
the oracle's finite-difference blocks, with the bar of test_gpu_jacobian."""
import numpy as np
import pytest

from iceicle_amd import abi
from tests import cases
from tests.test_gpu_jacobian import _compare, _mesh

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flux", [abi.FLUX_BURGERS, abi.FLUX_NAVIER_STOKES, abi.FLUX_EULER])
@pytest.mark.parametrize("order", [1, 4])
def test_2d_tile_edges(flux, order):
    p = cases.burgers_params(2, mu=0.05, a=(0.3, -0.2, 0)) if flux == abi.FLUX_BURGERS else cases.ns_params(2, flux=flux)
    bct = ["DIRICHLET", "NEUMANN", "EXTRAPOLATION", "DIRICHLET"] if flux == abi.FLUX_BURGERS else \
        ["RIEMANN", "SLIP_WALL", "DIRICHLET", "EXTRAPOLATION"]
    m, keep = _mesh(2, [3, 2], bct, 0.15, 4, bcflag=[0, 1, 0, 0])
    _compare(m, order, p, cases.random_state(flux, 2, 6, (order + 1) ** 2, 11))


@pytest.mark.parametrize("flux", [abi.FLUX_NAVIER_STOKES, abi.FLUX_EULER])
@pytest.mark.parametrize("order", [1, 2, 4])
def test_1d_systems(flux, order):
    p = cases.ns_params(1, flux=flux)
    m, keep = _mesh(1, [5], ["RIEMANN", "EXTRAPOLATION"], 0.2, 3)
    _compare(m, order, p, cases.random_state(flux, 1, 5, order + 1, 12))


@pytest.mark.parametrize("dim,order", [(1, 2), (1, 4), (2, 2), (2, 3)])
def test_viscous_entries_of_dimensional_air(dim, order):
    """Blocks of nodes off the shared face couple through the gradient alone,
    so they scale with a constant viscosity: air in SI units (energy flux
    4e7 W/m^2 and viscosity 1.8e-5 Pa s, twelve decades apart) against the same
    state with 2^30 times the viscosity, whose entries the convective flux
    does not blur.  A few roundings of the quantities of one entry: 1e-12."""
    from iceicle_amd import engine
    out = []
    for scale in (1.0, 2.0 ** 30):
        p = cases.ns_params(dim, mu=1.8e-5 * scale)
        p.dirichlet[0] = abi.Field.make("CONSTANT", [1.2, 120.0] + [0.0] * (dim - 1) + [2.5e5])
        m = abi.mesh_desc(dim, [3] * dim, [0.0] * dim, [0.02] * dim, ["DIRICHLET"] * (2 * dim))
        disc = engine.ConservationLawDDG(engine.FESpace(m, order), p)
        n, nb, v = order + 1, (order + 1) ** dim, dim + 2
        rng = np.random.default_rng(5)
        u = np.tile([1.2, 120.0] + [40.0] * (dim - 1) + [2.5e5], (disc.size // v, 1))
        u *= 1.0 + 0.02 * rng.uniform(-1.0, 1.0, u.shape)
        jac = engine.BlockJacobian(disc)
        jac.assemble(torch.from_numpy(u.ravel()).cuda())
        blk = jac.blocks.cpu().numpy().reshape(jac.cols.shape + (nb, v, nb, v))
        rows = []
        for e, s in zip(*np.nonzero(jac.cols[:, 1:] >= 0)):
            node = np.arange(nb) // n ** (dim - 1 - s % dim) % n  # index along the face's axis
            off = node != (n - 1 if s < dim else 0)               # the neighbour's nodes off the face
            rows.append(blk[e, 1 + s][:, :, off] / scale)
        out.append(np.stack(rows))
    # entry by entry of (row variable, column variable)
    for i in range(v):
        for j in range(v):
            a, b = (x[:, :, i, :, j] for x in out)
            err = np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)
            print(f"{dim}D P{order} ({i},{j}): {err:.1e} of {np.abs(b).max():.1e}", flush=True)
            assert err <= 1e-12, (i, j)
