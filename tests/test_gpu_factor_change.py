"""A plan whose factors change kind after its applies were captured: built from
a trilinear mesh (recomputed), then the caller's or a curved mesh's (read), and
back.  Solvers that keep a captured iteration, and graphs of the caller's that
are replayed, use the factors the plan holds at the replay: bit for bit what an
eager plan with the same factors gives."""

import numpy as np
import pytest
import torch

from libceed_amd import batch, ops
from libceed_amd.mesh import hex_mesh, node_coordinates

pytestmark = pytest.mark.gpu


def recomputing(op):
    """The plan, in the line layout also where a tuner has found another faster for such plans before."""
    if not op.recomputes_factors():
        op.set_layout(ops.LAYOUT_LINES)
    assert op.recomputes_factors()
    return op


def curved(op, m):
    """Three mesh nodes per direction on the p = 2 numbering, off the straight edges."""
    xyz = node_coordinates(m, np.array([-1.0, 0.0, 1.0])) + np.random.default_rng(5).uniform(-0.01, 0.01, (3, m.num_nodes))
    op.build_qdata(m.offsets, torch.from_numpy(xyz.reshape(-1)).cuda(), m.num_nodes, mesh_P=3)


def trilinear(op, m):
    op.build_qdata(m.mesh_offsets, torch.from_numpy(m.coords).cuda(), m.num_vertices)


def weights(op, seed):
    """Other factors: the plan's own, scaled element by element."""
    qd = op.get_qdata()
    w = torch.from_numpy(np.random.default_rng(seed).uniform(0.5, 2.0, op.num_elem)).to(qd.dtype).cuda()
    return (qd.view(op.num_elem, -1) * w[:, None]).reshape(-1).contiguous()


@pytest.mark.parametrize("mixed", [False, True])
def test_cg_follows_the_factors(cuda, mixed):
    m, Q = hex_mesh(4, 2, seed=3, perturb=0.2), 4
    op64 = recomputing(ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q))
    plans = [op64] + ([recomputing(ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, dtype=torch.float32))] if mixed else [])
    cg = ops.CG(plans[1], op64) if mixed else ops.CG(op64)
    u = torch.from_numpy(np.random.default_rng(1).uniform(-1, 1, m.num_nodes)).cuda()
    b, x, x_ref = torch.empty_like(u), torch.empty_like(u), torch.empty_like(u)

    def check(what):
        op64.apply(u, b)
        for rep in range(2):
            x.zero_(), x_ref.zero_()
            print(what, "mixed", mixed, flush=True)
            cg.solve(b, x, max_iter=40, rtol=0.0, check_every=10)
            ref.solve(b, x_ref, max_iter=40, rtol=0.0, check_every=10, use_graph=False)
            assert torch.equal(x, x_ref), what

    ref = ops.CG(plans[1], op64) if mixed else ops.CG(op64)
    check("trilinear")
    for op in plans:
        op.set_qdata(weights(op, 7))
    check("set")
    for op in plans:
        trilinear(op, m)
    check("trilinear again")
    for op in plans:
        curved(op, m)
    check("curved")


def test_batch_cg_follows_the_factors(cuda):
    systems = batch.random_systems(count=6, seed=4, max_n=5, p_range=(2, 3))
    bcg, ref = batch.BatchCG(systems, autotune=False), batch.BatchCG(systems, autotune=False)
    b = torch.from_numpy(np.random.default_rng(2).uniform(-1, 1, bcg.n)).cuda()
    for i in range(len(systems)):
        b[bcg.range(i)] -= b[bcg.range(i)].mean()  # in the range of the Neumann operators
    x, x_ref = torch.empty_like(b), torch.empty_like(b)

    def check(what):
        for rep in range(2):
            x.zero_(), x_ref.zero_()
            print(what, flush=True)
            bcg.solve(b, x, max_iter=20, rtol=0.0, check_every=5)
            ref.solve(b, x_ref, max_iter=20, rtol=0.0, check_every=5, use_graph=False)
            assert torch.equal(x, x_ref), what

    check("trilinear")
    for k, (op, rop) in enumerate(zip(bcg.ops, ref.ops)):
        if op.qf == ops.QF_DIFFUSION:
            qd = weights(op, k)
            op.set_qdata(qd), rop.set_qdata(qd)
    check("set")


# n^3 elements, order, points: E^T in the launch, its gather, colours, split; one thread per element; three components
GRAPHS = [(3, 2, 4, 1, "tmap"), (9, 3, 5, 1, "tmap"), (5, 4, 6, 1, "color"), (4, 6, 8, 1, "split"), (33, 1, 2, 1, "tmap"), (3, 3, 5, 3, "tmap")]


@pytest.mark.parametrize("n,p,Q,nc,scatter", GRAPHS)
def test_captured_apply_follows_the_factors(cuda, n, p, Q, nc, scatter):
    m = hex_mesh(n, p, seed=n, perturb=0.2)
    op, ref = (ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, num_comp=nc, scatter=scatter) for _ in range(2))
    u, w = (torch.from_numpy(np.random.default_rng(s).uniform(-1, 1, nc * m.num_nodes)).cuda() for s in (0, 1))
    v, add, diag, v_ref, add_ref, diag_ref = (torch.empty_like(u) for _ in range(6))
    qd = torch.empty_like(op.get_qdata())
    recomputing(op), recomputing(ref)

    def calls(o, v, add, diag):
        o.apply(u, v)
        add.copy_(w)
        o.apply_add(u, add)
        o.assemble_diagonal(diag)

    calls(op, v, add, diag)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        calls(op, v, add, diag)

    def check(what):
        for rep in range(2):
            for t in (v, add, diag, v_ref, add_ref, diag_ref):
                t.fill_(7.0)
            print(what, n, p, Q, nc, scatter, flush=True)
            g.replay()
            torch.cuda.synchronize()
            calls(ref, v_ref, add_ref, diag_ref)
            assert torch.equal(v, v_ref) and torch.equal(add, add_ref) and torch.equal(diag, diag_ref), what
            calls(op, v, add, diag)  # eager between the replays
            assert torch.equal(v, v_ref) and torch.equal(add, add_ref) and torch.equal(diag, diag_ref), what

    check("trilinear")
    new = weights(op, 9)
    for o in (op, ref):
        o.set_qdata(new)
    check("set")
    for o in (op, ref):
        trilinear(o, m)
    check("trilinear again")
    # the caller's factors set from within a graph: in force from its replay on
    gs = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gs):
        op.set_qdata(qd)
    check("set_qdata captured")
    qd.copy_(new * 0.5)
    gs.replay()
    ref.set_qdata(qd)
    check("set_qdata replayed")
    for o in (op, ref):
        trilinear(o, m)
    check("trilinear a third time")
    qd.copy_(new * 0.25)
    gs.replay()
    ref.set_qdata(qd)
    check("set_qdata replayed again")


def test_captured_kappa_follows_the_factors(cuda):
    m, Q = hex_mesh(4, 2, seed=3, perturb=0.2), 4
    op, ref = (ops.HexOperator.from_mesh(ops.QF_DIFFUSION_KAPPA, m, Q=Q) for _ in range(2))
    rng = np.random.default_rng(0)
    u, lam = (torch.from_numpy(rng.uniform(-1, 1, m.num_nodes)).cuda() for _ in range(2))
    kappa = torch.from_numpy(np.exp(rng.uniform(-1, 1, m.num_elem * Q ** 3))).cuda()
    out, out_ref = ([torch.empty_like(u), torch.empty_like(u), torch.empty_like(kappa), torch.empty_like(u)] for _ in range(2))
    recomputing(op), recomputing(ref)

    def calls(o, v, gu, gk, kept):
        o.apply_kappa(kappa, u, v)
        o.apply_adjoint(u, lam, gu, gk, kappa=kappa)
        o.apply(u, kept)  # the plan's own kappa from then on

    calls(op, *out)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        calls(op, *out)

    def check(what):
        for rep in range(2):
            kappa.copy_(torch.from_numpy(np.exp(rng.uniform(-1, 1, kappa.numel()))))
            for t in out + out_ref:
                t.fill_(7.0)
            print(what, flush=True)
            g.replay()
            torch.cuda.synchronize()
            calls(ref, *out_ref)
            assert all(torch.equal(a, b) for a, b in zip(out, out_ref)), what
            calls(op, *out)
            assert all(torch.equal(a, b) for a, b in zip(out, out_ref)), what

    check("trilinear")
    for o in (op, ref):
        curved(o, m)
    check("curved")
    for o in (op, ref):
        trilinear(o, m)
    check("trilinear again")
