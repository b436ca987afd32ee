"""An output vector that is also an input of the operator (the active one, or a
passive field updated in place): the fused operators give what the staged path
gives, which reads all inputs first and whose Apply clears the output before."""

from pathlib import Path

import numpy as np
import pytest

from libceed_amd import ceed as libceed
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu
QF_FILE = Path(__file__).resolve().parent / "qfunctions" / "t-points.h"


def vector(ceed, a):
    v = ceed.Vector(a.size)
    v.set_array(a)
    return v


@pytest.mark.parametrize("n,p,Q", [(2, 1, 2), (3, 2, 4), (9, 3, 5)])
def test_output_is_a_passive_field(cuda, monkeypatch, n, p, Q):
    ceed, m = libceed.Ceed("/gpu/hip/mi355"), hex_mesh(n, p, seed=n)
    rng = np.random.default_rng(0)
    E, nq = m.num_elem, m.num_elem * Q ** 3
    u, f0, got = rng.uniform(-1, 1, m.num_nodes), rng.uniform(0.5, 1.5, nq), []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CEED_MI355_FUSE_QFUNCTIONS", fuse)
        rstr, rq = ceed.ElemRestriction(E, (p + 1) ** 3, 1, 1, m.num_nodes, m.offsets), ceed.StridedElemRestriction(E, Q ** 3, 1, nq, libceed.STRIDES_BACKEND)
        basis = ceed.BasisTensorH1Lagrange(3, 1, p + 1, Q, libceed.GAUSS)
        qf = ceed.QFunction(1, None, f"{QF_FILE}:values_at_points")
        qf.add_input("u", 1, libceed.EVAL_INTERP)
        qf.add_input("f", 1, libceed.EVAL_NONE)
        qf.add_output("out", 1, libceed.EVAL_NONE)
        op, uv, f, other = ceed.Operator(qf), vector(ceed, u), vector(ceed, f0), vector(ceed, np.zeros(nq))
        op.set_field("u", rstr, basis, libceed.VECTOR_ACTIVE)
        op.set_field("f", rq, libceed.BASIS_NONE, f)
        op.set_field("out", rq, libceed.BASIS_NONE, libceed.VECTOR_ACTIVE)
        out = []
        for call in (op.apply_add, op.apply):
            f.set_array(f0)
            call(uv, f)
            out.append(f.to_numpy())
            f.set_array(f0)
            op.apply(uv, other)  # and the fused kernel after it
            out.append(other.to_numpy())
        got.append(out)
    for a, b in zip(*got):
        assert np.linalg.norm(a - b) <= 1e-13 * np.linalg.norm(b)
    assert np.all(got[0][2] == 0)  # (u + 1) f of the cleared f


@pytest.mark.parametrize("n,p,Q", [(2, 2, 4), (9, 3, 5)])
@pytest.mark.parametrize("scatter", ["color", "tmap"])
def test_output_is_the_active_input(cuda, monkeypatch, n, p, Q, scatter):
    monkeypatch.setenv("CEED_MI355_SCATTER", scatter)
    ceed, m = libceed.Ceed("/gpu/hip/mi355"), hex_mesh(n, p, seed=n)
    rng = np.random.default_rng(0)
    E, nq = m.num_elem, m.num_elem * Q ** 3
    u, passive, got = rng.uniform(-1, 1, m.num_nodes), [rng.uniform(0.5, 1.5, k * nq) for k in (1, 2, 3)], []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CEED_MI355_FUSE_QFUNCTIONS", fuse)
        rstr = ceed.ElemRestriction(E, (p + 1) ** 3, 1, 1, m.num_nodes, m.offsets)
        rq = [ceed.StridedElemRestriction(E, Q ** 3, k, k * nq, libceed.STRIDES_BACKEND) for k in (1, 2, 3)]
        basis = ceed.BasisTensorH1Lagrange(3, 1, p + 1, Q, libceed.GAUSS)
        qf = ceed.QFunction(1, None, f"{QF_FILE}:three_passive")
        for name, size, mode in (("f", 1, libceed.EVAL_NONE), ("u", 1, libceed.EVAL_INTERP), ("g", 2, libceed.EVAL_NONE),
                                 ("du", 3, libceed.EVAL_GRAD), ("h", 3, libceed.EVAL_NONE)):
            qf.add_input(name, size, mode)
        qf.add_output("dv", 3, libceed.EVAL_GRAD)
        qf.add_output("v", 1, libceed.EVAL_INTERP)
        op, vecs = ceed.Operator(qf), [vector(ceed, a) for a in passive]
        for k, name in enumerate("fgh"):
            op.set_field(name, rq[k], libceed.BASIS_NONE, vecs[k])
        for name in ("u", "du", "dv", "v"):
            op.set_field(name, rstr, basis, libceed.VECTOR_ACTIVE)
        out = []
        for call in (op.apply_add, op.apply):
            v = vector(ceed, u)
            call(v, v)
            out.append(v.to_numpy())
        got.append(out)
    for a, b in zip(*got):
        assert np.linalg.norm(a - b) <= 1e-13 * np.linalg.norm(b)
