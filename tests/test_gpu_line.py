"""Line preconditioner (block tridiagonal solve) of 1D problems: cyclic
reduction with a row a thread and elimination along the chain, at the row
counts where the number of steps, the threads and the rule between the two
change, for every small block size; the way back from a reduction that meets
a singular block to elimination along the chain, and singular blocks there;
and a norm's sizes on both sides of one workgroup's 16384 entries.

With the preconditioner an exact inverse, J x = b is solved in one iteration
(two, should the first leave a residual above the tolerance asked); x is held
to 1e-9, the condition of the viscous operator times the rounding of FP64."""
import ctypes as C

import numpy as np
import pytest

from iceicle_amd import abi
from tests import cases

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,nelem", [(3, 2), (3, 4), (1, 5), (3, 5), (2, 8), (3, 63), (4, 64), (1, 65), (2, 129), (3, 255),
                                         (3, 256), (4, 257), (3, 300), (2, 511), (4, 512), (3, 513), (4, 1023),
                                         (1, 1024), (4, 1024), (3, 1025),
                                         (3, 4096), (3, 4097)])
def test_line_solve(order, nelem):
    from iceicle_amd import engine
    p = cases.burgers_params(1, mu=0.02, a=(0.5, 0, 0))
    m = abi.mesh_desc(1, [nelem], [0.0], [1.0], ["DIRICHLET"] * 2)
    disc = engine.ConservationLawDDG(engine.FESpace(m, order), p)
    rng = np.random.default_rng(nelem)
    u = torch.from_numpy(rng.uniform(-0.5, 0.5, disc.size)).cuda()
    jac = engine.BlockJacobian(disc)
    jac.assemble(u)
    x_true = torch.from_numpy(rng.normal(size=disc.size)).cuda()
    b = torch.empty_like(u)
    jac.apply(x_true, b)
    solver = engine.PetscNewton(disc, jacobian_precision=abi.PREC_FP64, preconditioner=abi.PC_LINE, linear_rtol=1e-12)
    x = torch.full_like(u, float("nan"))
    its, rel = solver.linear_solve(b, x, u=u)
    err = float((x - x_true).norm() / x_true.norm())
    print(f"P{order} {nelem}: {its} iterations, rel {rel:.2e}, x err {err:.2e}", flush=True)
    assert its <= 2 and rel <= 1e-12 and err <= 1e-9


def _chain_reference(D, L, U, b):
    """Elimination along the chain, singular blocks replaced by the identity: x and their number."""
    n, bs = b.shape
    W, y, bad = np.zeros((bs, bs)), np.zeros(bs), 0
    Ws, ys = [], []
    for e in range(n):
        S = D[e] - L[e] @ W
        try:
            inv = np.linalg.inv(S)
        except np.linalg.LinAlgError:
            inv, bad = np.eye(bs), bad + 1
        W, y = inv @ U[e], inv @ (b[e] - L[e] @ y)
        Ws.append(W)
        ys.append(y)
    for e in range(n - 2, -1, -1):
        ys[e] = ys[e] - Ws[e] @ ys[e + 1]
    return np.stack(ys), bad


class _Line:
    """The block tridiagonal solver on matrices of the test's choice."""

    def __init__(self, n, bs):
        from iceicle_amd import engine
        lib = engine.lib()
        work = lib._ZN3ice15line_small_workEii
        work.restype, work.argtypes = C.c_size_t, [C.c_int] * 2
        self.factor_ = lib._ZN3ice17line_small_factorEiiiPKdPdS2_PiP12ihipStream_t
        self.solve_ = lib._ZN3ice16line_small_solveEiiiPKdS1_S1_S1_PdP12ihipStream_t
        for f, k in ((self.factor_, 5), (self.solve_, 6)):
            f.restype, f.argtypes = C.c_int, [C.c_int] * 3 + [C.c_void_p] * k
        self.n, self.bs = n, bs
        self.sinv = torch.full((n * bs * bs,), float("nan"), dtype=torch.float64, device="cuda")
        self.work = torch.full((work(n, bs),), float("nan"), dtype=torch.float64, device="cuda")

    def solve(self, D, L, U, b):
        J = torch.from_numpy(np.ascontiguousarray(np.stack([D, L, U], axis=1))).cuda()
        bd, bad = torch.from_numpy(b).cuda(), torch.zeros(1, dtype=torch.int32, device="cuda")
        x = torch.full_like(bd, float("nan"))
        st = torch.cuda.current_stream().cuda_stream
        a = (self.n, 3, self.bs, J.data_ptr(), self.sinv.data_ptr(), self.work.data_ptr())
        assert self.factor_(*a, bad.data_ptr(), st) == 0
        assert self.solve_(*a, bd.data_ptr(), x.data_ptr(), st) == 0
        torch.cuda.synchronize()
        return x.cpu().numpy(), int(bad)


def _product(D, L, U, x):
    y = np.einsum("eij,ej->ei", D, x)
    y[1:] += np.einsum("eij,ej->ei", L[1:], x[:-1])
    y[:-1] += np.einsum("eij,ej->ei", U[:-1], x[1:])
    return y


@pytest.mark.parametrize("kind,n", [(k, n) for k in ("cancelled", "zero", "defective", "late") for n in (5, 9, 64, 300, 1024)
                                    if n > 5 or k != "late"])
@pytest.mark.parametrize("bs", [2, 3, 4, 5])
def test_reduction_that_meets_a_singular_block(kind, bs, n):
    """Blocks regular along the chain, but a diagonal block that is singular,
    or that reduction cancels: D = L D'^-1 U + U D'^-1 L at one row leaves it
    rounding only, in one step or (late) in the second.  The solve then goes
    along the chain, residual ten times that of the same elimination in numpy,
    or 1e-13.  A regular matrix on the same buffers afterwards is solved to
    1e-13."""
    rng = np.random.default_rng(100 * n + bs)
    D, L, U = (a * np.eye(bs) + 0.2 * rng.normal(size=(n, bs, bs)) for a in (4.0, 1.0, 1.0))
    L[0], U[-1] = 0.0, 0.0
    good = D.copy()
    e = n // 2
    inv = np.linalg.inv
    if kind == "cancelled":
        D[e] = L[e] @ inv(D[e - 1]) @ U[e - 1] + U[e] @ inv(D[e + 1]) @ L[e + 1]
    elif kind == "zero":
        D[e] = 0.0
    elif kind == "defective":
        D[e][:, -1] = D[e][:, 0]
    else:  # the second step eliminates rows two away, reduced once
        def once(k):
            d, l, u = D[k].copy(), np.zeros((bs, bs)), np.zeros((bs, bs))
            if k > 0:
                a = L[k] @ inv(D[k - 1])
                d, l = d - a @ U[k - 1], -a @ L[k - 1]
            if k + 1 < n:
                c = U[k] @ inv(D[k + 1])
                d, u = d - c @ L[k + 1], -c @ U[k + 1]
            return d, l, u
        (d, l, u), lo, hi = once(e), once(e - 2), once(e + 2)
        D[e] = D[e] - d + l @ inv(lo[0]) @ lo[2] + u @ inv(hi[0]) @ hi[1]
    solver = _Line(n, bs)
    b = rng.normal(size=(n, bs))
    x, bad = solver.solve(D, L, U, b)
    ref = _chain_reference(D, L, U, b)[0]
    err = [np.linalg.norm(_product(D, L, U, v) - b) / np.linalg.norm(b) for v in (x, ref)]
    x, bad2 = solver.solve(good, L, U, b)
    err.append(np.linalg.norm(_product(good, L, U, x) - b) / np.linalg.norm(b))
    print(f"{kind} {bs} {n}: {err[0]:.1e} (numpy {err[1]:.1e}), regular {err[2]:.1e}", flush=True)
    assert err[0] <= max(10.0 * err[1], 1e-13) and bad == 0
    assert err[2] <= 1e-13 and bad2 == 0


@pytest.mark.parametrize("n", [4, 5, 64, 1024, 1025])
@pytest.mark.parametrize("bs", [1, 3, 5])
def test_singular_chain(bs, n):
    """A block singular along the chain too is replaced by the identity and counted."""
    rng = np.random.default_rng(n + bs)
    D = rng.normal(size=(n, bs, bs)) + (3.0 + 2.0 * bs) * np.eye(bs)
    L, U = rng.normal(size=(n, bs, bs)), rng.normal(size=(n, bs, bs))
    D[0] = 0.0
    b = rng.normal(size=(n, bs))
    x, bad = _Line(n, bs).solve(D, L, U, b)
    ref, want = _chain_reference(D, L, U, b)
    err = np.abs(x - ref).max() / np.abs(ref).max()
    print(f"{bs} {n}: {err:.1e}", flush=True)
    assert bad == want == 1 and err <= 1e-10
