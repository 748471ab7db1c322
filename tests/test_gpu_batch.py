"""Batched instances: a batched space evaluates every instance exactly as
its own space does (bit for bit where both take the same kernel, as here: see
test_gpu_lane2d for a space of elements enough for the lanes against one that
has not), per-element viscosities and step sizes
reproduce per-instance runs, HIP-graph replay reproduces eager stepping,
and every element-kernel tile gives the same residual."""
import numpy as np
import pytest

from iceicle_amd import abi, batch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

INSTS = [dict(N=3, p=2, nu=0.02, amp=np.array([0.5, -0.3, 0.2, 0.1])),
         dict(N=5, p=2, nu=0.003, amp=np.array([-0.7, 0.1, 0.4, -0.2])),
         dict(N=4, p=2, nu=0.08, amp=np.array([0.2, 0.9, -0.5, 0.3]))]


def _single(inst):
    from iceicle_amd import engine
    space = engine.FESpace(batch.mesh(inst["N"]), inst["p"])
    disc = engine.ConservationLawDDG(space, batch.params(inst["nu"]))
    xn = space.node_coords()
    u0 = batch.initial_condition(xn[..., 0], xn[..., 1], inst["amp"]).ravel()
    return space, disc, torch.from_numpy(u0).cuda()


def test_batched_residual_equals_per_instance():
    from iceicle_amd import engine
    g = batch.Group(INSTS, 2)
    r = torch.empty_like(g.u)
    engine.form_residual(g.space, g.disc, g.u, r)
    for k, inst in enumerate(INSTS):
        space, disc, u = _single(inst)
        assert torch.equal(g.u[g.instance_slice(k)], u)
        rk = torch.empty_like(u)
        engine.form_residual(space, disc, u, rk)
        assert torch.equal(r[g.instance_slice(k)], rk), k
    # the mixed-precision residual on the batch against the FP64 one
    r32 = torch.empty_like(r)
    engine.form_residual(g.space, g.disc, g.u, r32, precision="mixed")
    err = float((r32 - r).abs().max() / r.abs().max())
    print(f"batched mixed residual rel err {err:.2e}", flush=True)
    assert err <= 2e-5


def test_batched_steps_equal_per_instance_steps():
    """Element step sizes: each instance advances with its own CFL step,
    exactly as a separate stepper with that step."""
    from iceicle_amd import engine
    g = batch.Group(INSTS, 2)
    for _ in range(3):
        g.stepper.step(g.u)
    for k, inst in enumerate(INSTS):
        space, disc, u = _single(inst)
        st = engine.ExplicitStepper(disc, abi.stepper_desc(abi.STEP_RK3_SSP, dt=float(g.dt[k]), ntime=10))
        for _ in range(3):
            st.step(u)
        assert torch.equal(g.u[g.instance_slice(k)], u), k


def test_step_graph_replays_equal_eager_steps():
    insts = batch.sample_instances(10, seed=7)
    for i, inst in enumerate(insts):  # keep it small
        inst["N"] = 3 + i % 4
    b_eager = batch.Batch(insts)
    b_graph = batch.Batch(insts)
    graph = b_graph.graph(2)
    for rep in range(3):
        for _ in range(2):
            b_eager.step()
        graph.launch()
        torch.cuda.synchronize()
        # eager work between replays
        scratch = torch.ones(1000, device="cuda").sum()
        for ge, gg in zip(b_eager.groups, b_graph.groups):
            assert torch.equal(ge.u, gg.u), (rep, ge.order)
    assert all(bool(torch.isfinite(g.u).all()) for g in b_graph.groups)


def test_tiles_give_identical_residuals():
    from iceicle_amd import engine
    for order in (1, 3, 4):
        g = batch.Group([dict(INSTS[0], p=order), dict(INSTS[1], p=order)], order)
        rs = []
        for tile in (0, 1, 2):
            g.disc.set_tile(tile)
            r = torch.empty_like(g.u)
            engine.form_residual(g.space, g.disc, g.u, r)
            rs.append(r)
        assert torch.equal(rs[0], rs[1]) and torch.equal(rs[0], rs[2])
        best, ms = g.disc.autotune(g.u, torch.empty_like(g.u), reps=3)
        print(f"p={order} tile times {ms} best {best}", flush=True)
        assert best in (0, 1, 2)


def test_batched_space_rejections():
    from iceicle_amd import engine
    with pytest.raises(engine.IceError, match="share ndim"):
        engine.FESpace([batch.mesh(3), abi.mesh_desc(1, [4], [0], [1], ["PERIODIC"] * 2,
                                                     periodic_mode=abi.PERIODIC_COUPLED)], 1)
    g = batch.Group(INSTS, 2)
    with pytest.raises(engine.IceError):
        engine.PetscNewton(g.disc)  # no device Jacobian with per-element viscosity


def test_stiffest_members_stay_stable():
    """The most viscous, highest-order, finest members of the family over
    100 steps at their CFL step."""
    insts = [dict(N=96, p=4, nu=0.1, amp=np.array([1.0, -1.0, 1.0, -1.0])),
             dict(N=16, p=4, nu=1e-3, amp=np.array([1.0, 1.0, 1.0, 1.0])),
             dict(N=96, p=1, nu=0.1, amp=np.array([-1.0, 1.0, 0.5, 1.0]))]
    b = batch.Batch(insts)
    for _ in range(100):
        b.step()
    torch.cuda.synchronize()
    for g in b.groups:
        assert bool(torch.isfinite(g.u).all())
        assert float(g.u.abs().max()) <= 4.0 + 1e-9  # |u0| <= 4 and the solution does not grow


def test_full_batch_of_512_instances():
    """The batched workload at full size: 512 instances (N ~ U{16..96},
    p ~ U{1..4}, nu log-uniform on [1e-3, 1e-1]), about 24 M unknowns in four
    order groups.  Properties checked: every residual finite, the mixed
    residual close to the FP64 one (bound from FP32 rounding of the DDG jump
    terms), and 10 RK3-SSP steps at each instance's CFL step keep every
    state finite and inside the initial range (the viscous Burgers maximum
    principle, up to a 5% DG overshoot)."""
    from iceicle_amd import engine, workloads
    insts = batch.sample_instances(512, seed=workloads.SEED0 + 3)
    bt = batch.Batch(insts)
    assert len(bt.insts) == 512 and sum(len(g.insts) for g in bt.groups) == 512
    print(f"512 instances, {bt.size} unknowns, groups {[len(g.insts) for g in bt.groups]}", flush=True)
    r64 = [torch.empty_like(g.u) for g in bt.groups]
    r32 = [torch.empty_like(g.u) for g in bt.groups]
    bt.residual(r64)
    bt.residual(r32, precision="mixed")
    torch.cuda.synchronize()
    for g, a, b in zip(bt.groups, r64, r32):
        assert bool(torch.isfinite(a).all()) and bool(torch.isfinite(b).all()), g.order
        err = float((a - b).abs().max() / a.abs().max())
        print(f"p={g.order}: mixed vs FP64 residual {err:.2e}", flush=True)
        assert err < 2e-4, (g.order, err)
    umax0 = [float(g.u.abs().max()) for g in bt.groups]
    for _ in range(10):
        bt.step()
    torch.cuda.synchronize()
    for g, m0 in zip(bt.groups, umax0):
        assert bool(torch.isfinite(g.u).all()), g.order
        assert float(g.u.abs().max()) <= 1.05 * m0, (g.order, float(g.u.abs().max()), m0)


@pytest.mark.parametrize("order,one_launch", [(2, True), (4, False)])
def test_autotune_of_one_shape(order, one_launch):
    """A residual of one launch has one shape: tile 0 and one time, reported
    for all three; the three launches (Euler P4) are timed one tile at a time."""
    from iceicle_amd import engine
    m = abi.mesh_desc(2, [9, 8], [0.0, 0.0], [1.0, 1.0], ["EXTRAPOLATION"] * 4)
    disc = engine.ConservationLawDDG(engine.FESpace(m, order), abi.default_params(abi.FLUX_EULER))
    u = torch.from_numpy(np.tile([1.0, 0.3, 0.1, 2.0], disc.size // 4)).cuda()
    best, ms = disc.autotune(u, torch.empty_like(u), reps=3)
    assert all(t > 0.0 for t in ms) and best in (0, 1, 2)
    if one_launch:
        assert best == 0 and len(set(ms)) == 1
