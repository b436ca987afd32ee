"""The fused adjoint and the kappa-weighted apply at every order pair: factors
recomputed (trilinear geometry) and read (the same geometry through a
quadratic map), kappa held by the plan and taken from the caller on the way,
against the oracle at 1e-12; taking kappa on the way changes no bit and leaves
it in the plan."""

import numpy as np
import pytest
import torch

import oracle
from libceed_amd import ops
from libceed_amd.mesh import hex_mesh, node_coordinates

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return np.linalg.norm(a.cpu().numpy() - b) / np.linalg.norm(b)


# (elements per side, p, Q): one element, workgroups that are not full, several workgroups; every order pair
CASES = [(1, 1, 2), (5, 1, 3), (3, 2, 3), (4, 2, 4), (2, 3, 4), (3, 3, 5), (3, 4, 5), (1, 4, 6), (3, 5, 6), (2, 5, 7), (3, 6, 7),
         (1, 6, 8), (2, 7, 8), (2, 7, 9), (1, 8, 9), (2, 8, 10)]


# (a quadratic geometry needs Q >= 3)
@pytest.mark.parametrize("n,p,Q,read", [(*c, r) for c in CASES for r in (False, True) if c[2] >= 3 or not r])
def test_adjoint_orders(cuda, n, p, Q, read):
    m, P = hex_mesh(n, p, seed=5 * p + n), p + 1
    rng = np.random.default_rng(31 * p + Q)
    u, lam = rng.uniform(-1, 1, (2, m.num_nodes))
    kappa = np.exp(rng.uniform(-1, 1, m.num_elem * Q ** 3))
    qd = oracle.hex_build_qdata(1, m, Q)
    want_u = oracle.hex_apply_kappa(m.num_elem, P, Q, m.offsets, qd, kappa, u)
    want_v = oracle.hex_apply_kappa(m.num_elem, P, Q, m.offsets, qd, kappa, lam)
    want_g = -oracle.hex_kappa_gradient(m.num_elem, P, Q, m.offsets, qd, u, lam)
    ud, ld, kd = (torch.from_numpy(a).cuda() for a in (u, lam, kappa))
    for scatter in ("tmap", "color", "split"):
        op = ops.HexOperator.from_mesh(ops.QF_DIFFUSION_KAPPA, m, Q=Q, scatter=scatter)
        if read:
            m2 = hex_mesh(n, 2, seed=5 * p + n)  # the same vertices
            xyz = node_coordinates(m2, np.array([-1.0, 0.0, 1.0]))
            op.build_qdata(m2.offsets, torch.from_numpy(np.ascontiguousarray(xyz).reshape(-1)).cuda(), m2.num_nodes, mesh_P=3)
        for layout in (ops.LAYOUT_LINES, ops.LAYOUT_COLUMNS):
            print("p", p, "Q", Q, scatter, "read", read, "layout", layout, flush=True)
            try:
                op.set_layout(layout)
            except ops.CeedMi355Error:
                continue
            op.set_kappa(torch.full_like(kd, 7.0))
            v0, v1, w0, w1 = (torch.full_like(ud, c) for c in (1.0, 2.0, 3.0, 4.0))
            g0, g1 = torch.zeros_like(kd), torch.ones_like(kd)
            op.apply_kappa(kd, ud, v0)
            op.apply(ud, v1)
            assert torch.equal(v0, v1) and rel_l2(v0, want_u) < 1e-12
            op.apply_adjoint(ud, ld, w0, g0)
            op.set_kappa(torch.full_like(kd, 7.0))
            op.apply_adjoint(ud, ld, w1, g1, kappa=kd)
            assert rel_l2(w0, want_v) < 1e-12 and rel_l2(g0, want_g) < 1e-12
            assert torch.equal(g0, g1) and torch.equal(w0, w1)
            op.apply(ud, v1)  # the plan kept kappa
            assert torch.equal(v0, v1)
