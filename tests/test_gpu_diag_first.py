"""The diagonal of a gallery operator before any apply of it, and after its
q_data vector has changed since the last one: that of the vector's values."""

import numpy as np
import pytest

import oracle
from libceed_amd import ceed as libceed
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1])
def test_diagonal_before_apply(cuda, kind):
    ceed, m, Q = libceed.Ceed("/gpu/hip/mi355"), hex_mesh(2, 2, seed=1), 4
    E, N, nq, qc = m.num_elem, m.num_nodes, Q ** 3, 6 if kind else 1
    qd = oracle.hex_build_qdata(kind, m, Q).reshape(-1)
    rstr, basis = ceed.ElemRestriction(E, 27, 1, 1, N, m.offsets), ceed.BasisTensorH1Lagrange(3, 1, 3, Q, libceed.GAUSS)
    rq, q = ceed.StridedElemRestriction(E, nq, qc, E * nq * qc, libceed.STRIDES_BACKEND), ceed.Vector(E * nq * qc)
    q.set_array(qd)
    op = ceed.Operator(ceed.QFunctionByName("Poisson3DApply" if kind else "MassApply"))
    op.set_field("du" if kind else "u", rstr, basis, libceed.VECTOR_ACTIVE)
    op.set_field("qdata", rq, libceed.BASIS_NONE, q)
    op.set_field("dv" if kind else "v", rstr, basis, libceed.VECTOR_ACTIVE)
    eye = np.eye(N)
    want = np.array([oracle.hex_apply(kind, 1, E, 3, Q, m.offsets, N, qd, eye[j])[j] for j in range(N)])
    d = ceed.Vector(N)
    for scale in (1.0, 2.5):
        q.set_array(scale * qd)
        d.set_array(np.full(N, 7.0))
        op.linear_assemble_diagonal(d)
        assert np.linalg.norm(d.to_numpy() - scale * want) < 1e-12 * np.linalg.norm(scale * want)
        op.linear_assemble_add_diagonal(d)
        assert np.linalg.norm(d.to_numpy() - 2 * scale * want) < 1e-12 * np.linalg.norm(2 * scale * want)
