"""Which kernel takes a call, on either side of each rule's line, so that the
tests that compare two kernels compare two: recomputed against stored factors,
one thread per element against the line kernel, E^T in the apply's own launch
against the gather's, and the paths of a CeedOperator.  A launch the caller
sets is the one that runs."""

from pathlib import Path

import numpy as np
import pytest
import torch

from libceed_amd import ceed as libceed
from libceed_amd import ops
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu
QF_FILE = Path(__file__).resolve().parent / "qfunctions" / "t-points.h"


@pytest.mark.parametrize("kind,nc,p,Q,fp32,recomputes", [
    (1, 1, 1, 2, False, True), (1, 1, 4, 6, False, True), (1, 1, 6, 8, False, True), (1, 1, 8, 10, False, True), (1, 1, 5, 7, True, True),
    (1, 1, 6, 8, True, False), (1, 3, 2, 3, False, True), (1, 3, 3, 4, False, False), (1, 3, 6, 8, False, True), (2, 1, 3, 4, False, True),
    (0, 1, 3, 5, False, False), (1, 3, 2, 3, True, True), (1, 3, 3, 4, True, False), (1, 3, 3, 5, True, False), (1, 3, 4, 5, True, True),
    (1, 3, 4, 6, True, False), (1, 3, 5, 6, True, True), (1, 3, 6, 7, True, False), (1, 3, 7, 8, True, False), (1, 3, 7, 9, True, True),
    (1, 3, 8, 10, True, True)])
def test_recomputed_or_stored(cuda, kind, nc, p, Q, fp32, recomputes):
    m = hex_mesh(2, p, seed=1)
    op = ops.HexOperator.from_mesh(kind, m, Q=Q, num_comp=nc, dtype=torch.float32 if fp32 else torch.float64, scatter="tmap")
    op.set_layout(ops.LAYOUT_LINES)  # the default launch, whatever a tuner has found for such plans before
    assert op.recomputes_factors() == recomputes
    op.set_layout(ops.LAYOUT_COLUMNS)
    assert not op.recomputes_factors()
    op.set_layout(ops.LAYOUT_LINES, 1)
    assert op.recomputes_factors() == recomputes
    if kind != 2:
        u = torch.from_numpy(np.random.default_rng(p).uniform(-1, 1, nc * m.num_nodes)).to(op.dtype).cuda()
        v, w = torch.empty_like(u), torch.empty_like(u)
        op.apply(u, v)
        op.set_qdata(op.get_qdata())
        assert not op.recomputes_factors()
        op.apply(u, w)
        assert torch.equal(v, w)
    for scatter in ("brick", "segment") if kind != 2 else ():
        assert not ops.HexOperator.from_mesh(kind, m, Q=Q, num_comp=nc, dtype=op.dtype, scatter=scatter).recomputes_factors()


# the last and the first side of a cube of elements: a launch (one of eight colours: the largest) of 32768 for FP64 Q = 2,
# 98304 otherwise
@pytest.mark.parametrize("n,Q,fp32,scatter,kernel", [
    (31, 2, False, "tmap", "lines"), (32, 2, False, "tmap", "elements"), (46, 3, False, "tmap", "lines"), (47, 3, False, "split", "elements"),
    (46, 2, True, "tmap", "lines"), (47, 2, True, "atomic", "elements"), (62, 2, False, "color", "lines"), (64, 2, False, "color", "elements")])
def test_one_thread_per_element(cuda, n, Q, fp32, scatter, kernel):
    m = hex_mesh(n, 1, seed=n)
    dtype = torch.float32 if fp32 else torch.float64
    op = ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, dtype=dtype, scatter=scatter)
    op.set_layout(ops.LAYOUT_LINES)
    assert op.kernel()[0] == kernel
    u = torch.from_numpy(np.random.default_rng(n).uniform(-1, 1, m.num_nodes)).to(dtype).cuda()
    v, w = torch.empty_like(u), torch.empty_like(u)
    op.apply(u, v)
    op.set_launch(3)  # the caller's launch: the line kernel with three elements
    assert op.kernel()[0] == "lines" and op.launch() == (ops.LAYOUT_LINES, 3)
    op.apply(u, w)
    assert scatter == "atomic" or torch.equal(v, w)
    op.set_layout(ops.LAYOUT_LINES)  # the default again
    assert op.kernel()[0] == kernel
    _, ms = op.autotune(2)
    assert ms > 0
    op.apply(u, w)
    assert scatter == "atomic" or torch.equal(v, w)
    other = ops.HexOperator.from_mesh(ops.QF_DIFFUSION, hex_mesh(n, 1, seed=n + 1), Q=Q, dtype=dtype, scatter=scatter)
    assert (other.launch(), other.kernel()) == (op.launch(), op.kernel())  # what the tuner chose, for the next plan too
    op.set_qdata(op.get_qdata())
    assert op.kernel()[0] != "elements"


@pytest.mark.parametrize("n,p,Q,nc,gather", [(1, 1, 2, 1, False), (12, 1, 3, 1, False), (13, 1, 3, 1, True), (10, 2, 4, 1, False), (11, 2, 4, 1, True),
                                             (6, 3, 5, 1, False), (3, 4, 6, 1, True), (3, 2, 4, 3, True)])
def test_transpose_in_the_launch(cuda, n, p, Q, nc, gather):
    m = hex_mesh(n, p, seed=1)
    op = ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, num_comp=nc, scatter="tmap")
    op.set_layout(ops.LAYOUT_LINES)
    assert op.kernel() == ("lines", gather)
    op.set_layout(ops.LAYOUT_COLUMNS)
    assert op.kernel() == ("columns", True)
    hole = ops.HexOperator(ops.QF_DIFFUSION, m.offsets, m.num_elem, p + 1, Q, nc * m.num_nodes + 1, num_comp=nc, comp_stride=m.num_nodes, scatter="tmap")
    hole.set_layout(ops.LAYOUT_LINES)
    assert hole.kernel() == ("lines", True)  # an entry no element reaches
    assert not ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, num_comp=nc, scatter="color").kernel()[1]
    assert ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, num_comp=nc, scatter="split").kernel()[1]


@pytest.mark.parametrize("name,passive_strides,path", [("values_at_points", "backend", "points"), ("values_at_points", "own", "staged"),
                                                       ("three_passive", "backend", "fused-qfunction"), ("three_passive", "own", "fused-qfunction"),
                                                       ("MassApply", "backend", "fused")])
def test_operator_paths(cuda, monkeypatch, name, passive_strides, path):
    ceed, m, Q = libceed.Ceed("/gpu/hip/mi355"), hex_mesh(2, 2, seed=1), 4
    E, nq = m.num_elem, Q ** 3
    strides = libceed.STRIDES_BACKEND if passive_strides == "backend" else [E, E * nq, 1]
    rstr, basis = ceed.ElemRestriction(E, 27, 1, 1, m.num_nodes, m.offsets), ceed.BasisTensorH1Lagrange(3, 1, 3, Q, libceed.GAUSS)

    def make():
        if name == "MassApply":
            qf = ceed.QFunctionByName("MassApply")
            fields, outs = [("u", 1, libceed.EVAL_INTERP), ("qdata", 1, libceed.EVAL_NONE)], [("v", 1, libceed.EVAL_INTERP)]
        else:
            qf = ceed.QFunction(1, None, f"{QF_FILE}:{name}")
            fields, outs = {"values_at_points": ([("u", 1, libceed.EVAL_INTERP), ("f", 1, libceed.EVAL_NONE)], [("out", 1, libceed.EVAL_NONE)]),
                            "three_passive": ([("f", 1, libceed.EVAL_NONE), ("u", 1, libceed.EVAL_INTERP), ("g", 2, libceed.EVAL_NONE),
                                               ("du", 3, libceed.EVAL_GRAD), ("h", 3, libceed.EVAL_NONE)],
                                              [("dv", 3, libceed.EVAL_GRAD), ("v", 1, libceed.EVAL_INTERP)])}[name]
            for f in fields:
                qf.add_input(*f)
            for f in outs:
                qf.add_output(*f)
        op = ceed.Operator(qf)
        for field, size, mode in fields:
            if mode == libceed.EVAL_NONE:
                v = ceed.Vector(E * nq * size)
                v.set_array(np.ones(E * nq * size))
                op.set_field(field, ceed.StridedElemRestriction(E, nq, size, E * nq * size, strides), libceed.BASIS_NONE, v)
            else:
                op.set_field(field, rstr, basis, libceed.VECTOR_ACTIVE)
        for field, size, mode in outs:
            at_points = mode == libceed.EVAL_NONE
            op.set_field(field, ceed.StridedElemRestriction(E, nq, size, E * nq * size, libceed.STRIDES_BACKEND) if at_points else rstr,
                         libceed.BASIS_NONE if at_points else basis, libceed.VECTOR_ACTIVE)
        return op

    assert make().path() == path
    monkeypatch.setenv("CEED_MI355_FUSE_QFUNCTIONS", "0")
    assert make().path() == ("fused" if path == "fused" else "staged")


@pytest.mark.parametrize("n,p,Q,epb", [(25, 3, 5, 2), (26, 3, 5, 5), (4, 5, 7, 1)])
def test_three_component_workgroups(cuda, n, p, Q, epb):
    """Stored factors, three components, transpose map: full wavefronts at Q = 5 from 16384 elements, not at Q = 7."""
    m = hex_mesh(n, p, seed=1)
    op = ops.HexOperator(ops.QF_DIFFUSION, m.offsets, m.num_elem, p + 1, Q, 3 * m.num_nodes, num_comp=3, comp_stride=m.num_nodes, scatter="tmap")
    op.set_layout(ops.LAYOUT_LINES)
    assert op.launch() == (ops.LAYOUT_LINES, epb)
