"""Diagonal assembly at every order, against the sum over quadrature points
written out in numpy (FP64 within 1e-12, FP32 within 2e-6), with the factors
recomputed, read, and (kappa) weighted; workgroups that are full, partly full
and of one element."""

import numpy as np
import pytest
import torch

import oracle
from libceed_amd import ops
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu


def numpy_diag(m, Q, kind, qd, kappa=None):
    B, G, _, _ = oracle.lagrange_1d(m.P, Q)
    B, G = B.reshape(Q, m.P), G.reshape(Q, m.P)
    grad = [np.kron(np.kron(*zy), x) for zy, x in (((B, B), G), ((B, G), B), ((G, B), B))]  # z slowest
    qd = qd.reshape(m.num_elem, -1, Q ** 3)
    if kind == ops.QF_MASS:
        elem = qd[:, 0] @ np.kron(np.kron(B, B), B) ** 2
    else:
        if kappa is not None:
            qd = qd * kappa.reshape(m.num_elem, 1, Q ** 3)
        voigt = {(0, 0): 0, (1, 1): 1, (2, 2): 2, (1, 2): 3, (0, 2): 4, (0, 1): 5}
        elem = sum((1 if a == b else 2) * qd[:, k] @ (grad[a] * grad[b]) for (a, b), k in voigt.items())
    d = np.zeros(m.num_nodes)
    np.add.at(d, m.offsets.reshape(-1), elem.reshape(-1))
    return d


@pytest.mark.parametrize("p,Q,n", [(1, 2, 5), (1, 3, 4), (2, 4, 3), (3, 5, 3), (4, 6, 2), (5, 6, 2), (5, 7, 2), (6, 8, 2), (7, 9, 2), (8, 9, 1), (8, 10, 2)])
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_diagonal_orders(cuda, p, Q, n, kind):
    m = hex_mesh(n, p, seed=p, perturb=0.25)
    qd = oracle.hex_build_qdata(min(kind, 1), m, Q)
    kappa = np.exp(np.random.default_rng(p).uniform(-1, 1, m.num_elem * Q ** 3)) if kind == 2 else None
    ref = numpy_diag(m, Q, kind, qd, kappa)
    for dtype, tol in ((torch.float64, 1e-12), (torch.float32, 2e-6)):
        for read in (False, True):
            if read and kind == 2:  # such a plan's factors come from its geometry
                continue
            op = ops.HexOperator.from_mesh(kind, m, Q=Q, dtype=dtype)
            if read:
                op.set_qdata(torch.from_numpy(qd).to(dtype).cuda())
            if kind == 2:
                op.set_kappa(torch.from_numpy(kappa).cuda())
            d = torch.full((m.num_nodes,), 7.0, dtype=dtype, device="cuda")
            op.assemble_diagonal(d)
            got = d.double().cpu().numpy()
            assert np.linalg.norm(got - ref) < tol * np.linalg.norm(ref), (dtype, read)
