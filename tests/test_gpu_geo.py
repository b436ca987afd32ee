"""Plans on a trilinear geometry, whose line kernel recomputes the geometric
factors from the element's map instead of reading them: bitwise equal to the
same plan reading the factors it hands out, at every workgroup size and in
every kind of element map; factors and applies against the oracle at 1e-12.
A geometry that is not trilinear, or factors set by the caller, are read."""

import numpy as np
import pytest
import torch

import oracle
from libceed_amd import ops
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def host(t):
    return t.cpu().numpy()


# every Q of 2..10; one element, elements that do not fill a workgroup, more than one workgroup; both precisions; three
# components computing the factors once (Q <= 7) and per component (Q >= 8); mass and (FP32, Q = 8) keep reading
CASES = [(1, 1, 1, 1, 2, False), (1, 1, 5, 1, 3, False), (1, 1, 3, 2, 4, False), (1, 1, 2, 3, 5, False), (1, 1, 4, 4, 6, False),
         (1, 1, 3, 5, 7, False), (1, 1, 3, 6, 8, False), (1, 1, 2, 7, 9, False), (1, 1, 2, 8, 10, False), (1, 1, 3, 4, 5, False),
         (1, 3, 3, 1, 3, False), (1, 3, 2, 4, 6, False), (1, 3, 2, 6, 8, False), (1, 3, 1, 8, 9, False), (1, 1, 3, 4, 6, True),
         (1, 1, 2, 6, 8, True), (1, 3, 2, 5, 7, True), (1, 3, 2, 7, 8, True), (2, 1, 3, 3, 4, False), (2, 1, 2, 6, 7, False), (0, 1, 3, 3, 5, False)]


@pytest.mark.parametrize("kind,nc,n,p,Q,fp32", CASES)
def test_recomputed_factors_bitwise(cuda, kind, nc, n, p, Q, fp32):
    m = hex_mesh(n, p, seed=17 * p + n, perturb=0.3)
    dtype = torch.float32 if fp32 else torch.float64
    rng = np.random.default_rng(p + nc)
    u = torch.from_numpy(rng.uniform(-1, 1, nc * m.num_nodes)).to(dtype).cuda()
    w0 = torch.from_numpy(rng.uniform(-1, 1, nc * m.num_nodes)).to(dtype).cuda()
    kappa = torch.from_numpy(np.exp(rng.uniform(-1, 1, m.num_elem * Q ** 3))).cuda()
    qd_ref = oracle.hex_build_qdata(min(kind, 1), m, Q)
    for scatter in ("tmap", "color"):
        op = ops.HexOperator.from_mesh(kind, m, Q=Q, num_comp=nc, dtype=dtype, scatter=scatter)
        stored = ops.HexOperator.from_mesh(kind, m, Q=Q, num_comp=nc, dtype=dtype, scatter=scatter)
        if kind == 2:  # the column layout reads the factors
            op.set_kappa(kappa)
            stored.set_kappa(kappa)
            stored.set_layout(ops.LAYOUT_COLUMNS)
        else:
            stored.set_qdata(op.get_qdata())
            assert rel_l2(host(op.get_qdata()).astype(float), qd_ref) < (1e-6 if fp32 else 1e-12)
        ref, ref_add = torch.full_like(u, 3.0), w0.clone()
        stored.apply(u, ref)
        stored.apply_add(u, ref_add)
        if not fp32:
            kq = host(kappa) if kind == 2 else None
            want = (oracle.hex_apply_kappa(m.num_elem, p + 1, Q, m.offsets, qd_ref, kq, host(u)) if kind == 2 else
                    oracle.hex_apply(kind, nc, m.num_elem, p + 1, Q, m.offsets, m.num_nodes, qd_ref, host(u)))
            assert rel_l2(host(ref), want) < 1e-12
        epbs = [0] + sorted({1, 2, 256 // (Q * Q)})
        for epb in epbs:
            try:
                if epb:
                    op.set_layout(ops.LAYOUT_LINES, epb)
            except ops.CeedMi355Error:
                continue  # more than a CU's LDS
            print("kind", kind, "nc", nc, "p", p, "Q", Q, scatter, "launch", op.launch(), flush=True)
            v, w = torch.full_like(u, -2.0), w0.clone()
            op.apply(u, v)
            op.apply_add(u, w)
            assert torch.equal(v, ref), (scatter, epb)
            assert torch.equal(w, ref_add), (scatter, epb)


def test_recomputed_factors_follow_the_geometry(cuda):
    """A second geometry replaces the first; the caller's factors replace both; a quadratic mesh basis is read."""
    m, m2, Q = hex_mesh(3, 2, seed=1), hex_mesh(3, 2, seed=2), 4
    u = np.random.default_rng(0).uniform(-1, 1, m.num_nodes)
    ud, v = torch.from_numpy(u).cuda(), torch.empty(m.num_nodes, dtype=torch.float64, device="cuda")
    op = ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q)

    def check(qd):
        op.apply(ud, v)
        assert rel_l2(host(v), oracle.hex_apply(1, 1, m.num_elem, 3, Q, m.offsets, m.num_nodes, qd, u)) < 1e-12

    check(oracle.hex_build_qdata(1, m, Q))
    op.build_qdata(m2.mesh_offsets, torch.from_numpy(m2.coords).cuda(), m2.num_vertices)
    check(oracle.hex_build_qdata(1, m2, Q))
    qd = oracle.hex_build_qdata(1, m, Q) * 0.5
    op.set_qdata(torch.from_numpy(qd).cuda())
    check(qd)
    # three mesh nodes per direction on the solution's own numbering (p = 2), midpoints off the straight edges
    rng = np.random.default_rng(5)
    from libceed_amd.mesh import node_coordinates
    xyz = node_coordinates(m, np.array([-1.0, 0.0, 1.0])) + rng.uniform(-0.01, 0.01, (3, m.num_nodes))
    op.build_qdata(m.offsets, torch.from_numpy(xyz.reshape(-1)).cuda(), m.num_nodes, mesh_P=3)
    got = host(op.get_qdata())
    check(got)
    one = torch.ones_like(ud)
    op.apply(one, v)
    assert v.abs().max().item() < 1e-12
    op.build_qdata(m.mesh_offsets, torch.from_numpy(m.coords).cuda(), m.num_vertices)
    check(oracle.hex_build_qdata(1, m, Q))
