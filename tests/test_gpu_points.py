"""Operators that one run-time compiled kernel took over from the staged path
(output at the quadrature points; several passive fields), against the staged
path itself, which CEED_MI355_FUSE_QFUNCTIONS=0 keeps: every kind of input,
components, bases with Q = P, P + 1, more, and collocated, one element up to
several workgroups, nodes in any numbering, Apply and ApplyAdd.  The two run
the same contractions with other roundings: 1e-13 relative L2."""

from pathlib import Path

import numpy as np
import pytest

from libceed_amd import ceed as libceed
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu
QF_FILE = Path(__file__).resolve().parent / "qfunctions" / "t-points.h"


@pytest.fixture(scope="module")
def ceed(cuda):
    return libceed.Ceed("/gpu/hip/mi355")


def rel_l2(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def vector(ceed, a):
    v = ceed.Vector(a.size)
    v.set_array(a)
    return v


def field(ceed, rng, E, nq, nc, strides=libceed.STRIDES_BACKEND):
    """A passive field of nc values per point: its restriction and vector."""
    return ceed.StridedElemRestriction(E, nq, nc, E * nq * nc, strides), vector(ceed, rng.uniform(0.5, 1.5, E * nq * nc))


def both(ceed, monkeypatch, make, u, n_out, v0):
    """Apply and ApplyAdd of the operator make() builds, fused and staged."""
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CEED_MI355_FUSE_QFUNCTIONS", fuse)
        op = make()
        uv, vv = vector(ceed, u), vector(ceed, v0)
        op.apply(uv, vv)
        a = vv.to_numpy()
        vv.set_array(v0)
        op.apply_add(uv, vv)
        op.apply_add(uv, vv)
        out.append((a, vv.to_numpy(), op))
    (a1, b1, _), (a0, b0, _) = out
    assert np.linalg.norm(a0) > 0 and a0.size == n_out
    assert rel_l2(a1, a0) < 1e-13 and rel_l2(b1, b0) < 1e-13
    assert rel_l2(b1, v0 + 2 * a1) < 1e-13


@pytest.mark.parametrize("nc,n,p,Q,quad", [(1, 1, 1, 2, 0), (3, 3, 1, 6, 0), (3, 2, 1, 10, 0), (2, 2, 2, 3, 0), (3, 2, 2, 4, 0), (1, 3, 3, 4, 0),
                                           (1, 2, 4, 8, 0), (3, 2, 5, 7, 0), (2, 1, 8, 9, 0), (1, 2, 8, 10, 0), (3, 2, 3, 4, 1), (1, 4, 1, 3, 0)])
def test_values_at_points(ceed, monkeypatch, nc, n, p, Q, quad):
    m = hex_mesh(n, p, seed=n + p)
    rng = np.random.default_rng(10 * p + nc)
    E, P, N = m.num_elem, p + 1, m.num_nodes
    stride = N + 5                                              # components apart, nodes renumbered, entries unused
    offsets = rng.permutation(stride)[:N].astype(np.int32)[m.offsets]
    u = rng.uniform(-1, 1, nc * stride)
    rstr = ceed.ElemRestriction(E, P ** 3, nc, stride, nc * stride, offsets)
    basis = ceed.BasisTensorH1Lagrange(3, nc, P, Q, quad)
    (rf, f), (rg, g) = field(ceed, rng, E, Q ** 3, 2), field(ceed, rng, E, Q ** 3, 1)
    ctx = ceed.QFunctionContext()
    ctx.set_data(np.array([0.7, -0.3]))

    def make():
        qf = ceed.QFunction(1, None, f"{QF_FILE}:mixed_at_points_{nc}")
        qf.add_input("f", 2, libceed.EVAL_NONE)
        qf.add_input("du", 3 * nc, libceed.EVAL_GRAD)
        qf.add_input("w", 1, libceed.EVAL_WEIGHT)
        qf.add_input("u", nc, libceed.EVAL_INTERP)
        qf.add_input("g", 1, libceed.EVAL_NONE)
        qf.add_output("out", 2, libceed.EVAL_NONE)
        qf.set_context(ctx)
        op = ceed.Operator(qf)
        op.set_field("f", rf, libceed.BASIS_NONE, f)
        op.set_field("du", rstr, basis, libceed.VECTOR_ACTIVE)
        op.set_field("w", libceed.ELEMRESTRICTION_NONE, basis, libceed.VECTOR_NONE)
        op.set_field("u", rstr, basis, libceed.VECTOR_ACTIVE)
        op.set_field("g", rg, libceed.BASIS_NONE, g)
        op.set_field("out", ceed.StridedElemRestriction(E, Q ** 3, 2, 2 * E * Q ** 3, libceed.STRIDES_BACKEND), libceed.BASIS_NONE,
                     libceed.VECTOR_ACTIVE)
        return op

    both(ceed, monkeypatch, make, u, 2 * E * Q ** 3, rng.uniform(-1, 1, 2 * E * Q ** 3))


@pytest.mark.parametrize("passive_strides,out_strides,extra", [("backend", "backend", 0), ("own", "backend", 0), ("backend", "own", 0), ("backend", "backend", 7)])
def test_values_at_points_strides(ceed, monkeypatch, passive_strides, out_strides, extra):
    """Values without a gradient; a passive field or an output with strides of its own (staged on both sides), and an
    output vector longer than its values."""
    m = hex_mesh(3, 2, seed=4)
    rng = np.random.default_rng(2)
    E, P, Q, N = m.num_elem, 3, 4, m.num_nodes
    nq = Q ** 3
    strides = {"backend": libceed.STRIDES_BACKEND, "own": [E, E * nq, 1]}
    rstr, basis = ceed.ElemRestriction(E, P ** 3, 1, 1, N, m.offsets), ceed.BasisTensorH1Lagrange(3, 1, P, Q, libceed.GAUSS)
    rf, f = field(ceed, rng, E, nq, 1, strides[passive_strides])

    def make():
        qf = ceed.QFunction(1, None, f"{QF_FILE}:values_at_points")
        qf.add_input("u", 1, libceed.EVAL_INTERP)
        qf.add_input("f", 1, libceed.EVAL_NONE)
        qf.add_output("out", 1, libceed.EVAL_NONE)
        op = ceed.Operator(qf)
        op.set_field("u", rstr, basis, libceed.VECTOR_ACTIVE)
        op.set_field("f", rf, libceed.BASIS_NONE, f)
        op.set_field("out", ceed.StridedElemRestriction(E, nq, 1, E * nq + extra, strides[out_strides]), libceed.BASIS_NONE, libceed.VECTOR_ACTIVE)
        return op

    v0 = np.zeros(E * nq + extra)
    v0[:E * nq] = rng.uniform(-1, 1, E * nq)
    both(ceed, monkeypatch, make, rng.uniform(-1, 1, N), E * nq + extra, v0)


@pytest.mark.parametrize("n,p,Q", [(1, 1, 2), (3, 2, 4), (2, 4, 6), (2, 5, 7), (2, 6, 8), (1, 8, 10), (3, 3, 4), (2, 3, 6)])
@pytest.mark.parametrize("scatter", ["", "color"])
def test_three_passive_fields(ceed, monkeypatch, n, p, Q, scatter):
    """Passive fields of 1, 2 and 3 values, one with strides of its own; a new value of one is seen by the next apply."""
    if scatter:
        monkeypatch.setenv("CEED_MI355_SCATTER", scatter)
    m = hex_mesh(n, p, seed=n + p)
    rng = np.random.default_rng(p)
    E, P, N, nq = m.num_elem, p + 1, m.num_nodes, Q ** 3
    rstr, basis = ceed.ElemRestriction(E, P ** 3, 1, 1, N, m.offsets), ceed.BasisTensorH1Lagrange(3, 1, P, Q, libceed.GAUSS)
    (rf, f), (rg, g), (rh, h) = field(ceed, rng, E, nq, 1), field(ceed, rng, E, nq, 2, [E, E * nq, 1]), field(ceed, rng, E, nq, 3)

    def make():
        qf = ceed.QFunction(1, None, f"{QF_FILE}:three_passive")
        for name, size, mode in (("f", 1, libceed.EVAL_NONE), ("u", 1, libceed.EVAL_INTERP), ("g", 2, libceed.EVAL_NONE),
                                 ("du", 3, libceed.EVAL_GRAD), ("h", 3, libceed.EVAL_NONE)):
            qf.add_input(name, size, mode)
        qf.add_output("dv", 3, libceed.EVAL_GRAD)
        qf.add_output("v", 1, libceed.EVAL_INTERP)
        op = ceed.Operator(qf)
        for name, r, b, v in (("f", rf, libceed.BASIS_NONE, f), ("u", rstr, basis, libceed.VECTOR_ACTIVE), ("g", rg, libceed.BASIS_NONE, g),
                              ("du", rstr, basis, libceed.VECTOR_ACTIVE), ("h", rh, libceed.BASIS_NONE, h),
                              ("dv", rstr, basis, libceed.VECTOR_ACTIVE), ("v", rstr, basis, libceed.VECTOR_ACTIVE)):
            op.set_field(name, r, b, v)
        return op

    u, v0 = rng.uniform(-1, 1, N), rng.uniform(-1, 1, N)
    both(ceed, monkeypatch, make, u, N, v0)
    got = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CEED_MI355_FUSE_QFUNCTIONS", fuse)
        op, uv, vv = make(), vector(ceed, u), vector(ceed, v0)
        g.set_array(np.linspace(0.1, 0.9, E * nq * 2))
        op.apply(uv, vv)
        g.set_array(np.linspace(-0.9, 0.3, E * nq * 2))
        op.apply(uv, vv)
        got.append(vv.to_numpy())
    assert rel_l2(got[0], got[1]) < 1e-13
