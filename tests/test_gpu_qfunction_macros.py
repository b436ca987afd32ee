"""User QFunctions whose source defines macros with names the fused run-time
compiled kernels use themselves: the operators run, by the staged path, and
give what it gives."""

from pathlib import Path

import numpy as np
import pytest

from libceed_amd import ceed as libceed
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu
QF_FILE = Path(__file__).resolve().parent / "qfunctions" / "t-macros.h"
CASES = {  # inputs (name, values per point of one component, mode), outputs, components of the active field
    "macros_at_points": ([("u", 3, libceed.EVAL_INTERP), ("w", 1, libceed.EVAL_WEIGHT), ("f", 1, libceed.EVAL_NONE)], [("out", 1, libceed.EVAL_NONE)], 3),
    "macros_two_passive": ([("du", 3, libceed.EVAL_GRAD), ("u", 1, libceed.EVAL_INTERP), ("f", 1, libceed.EVAL_NONE), ("g", 1, libceed.EVAL_NONE)],
                           [("dv", 3, libceed.EVAL_GRAD), ("v", 1, libceed.EVAL_INTERP)], 1),
    "macros_mass": ([("u", 1, libceed.EVAL_INTERP), ("q", 1, libceed.EVAL_NONE)], [("v", 1, libceed.EVAL_INTERP)], 1),
}


@pytest.mark.parametrize("name", CASES)
def test_macros_of_the_users_source(cuda, monkeypatch, name):
    ceed = libceed.Ceed("/gpu/hip/mi355")
    ins, outs, nc = CASES[name]
    m, Q = hex_mesh(2, 2, seed=3), 4
    rng = np.random.default_rng(1)
    n, npts = m.num_nodes, m.num_elem * Q ** 3
    u = rng.uniform(-1, 1, nc * n)
    passive = {k: rng.uniform(0.5, 1.5, npts) for k in "fgq"}
    got = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CEED_MI355_FUSE_QFUNCTIONS", fuse)
        rstr, rq = ceed.ElemRestriction(m.num_elem, 27, nc, n, nc * n, m.offsets), ceed.StridedElemRestriction(m.num_elem, Q ** 3, 1, npts, libceed.STRIDES_BACKEND)
        basis = ceed.BasisTensorH1Lagrange(3, nc, 3, Q, libceed.GAUSS)
        qf = ceed.QFunction(1, None, f"{QF_FILE}:{name}")
        for field, size, mode in ins:
            qf.add_input(field, size, mode)
        for field, size, mode in outs:
            qf.add_output(field, size, mode)
        op, keep = ceed.Operator(qf), []
        for field, size, mode in ins + outs:
            if mode == libceed.EVAL_WEIGHT:
                op.set_field(field, libceed.ELEMRESTRICTION_NONE, basis, libceed.VECTOR_NONE)
            elif mode == libceed.EVAL_NONE and field in passive:
                v = ceed.Vector(npts)
                v.set_array(passive[field])
                keep.append(v)
                op.set_field(field, rq, libceed.BASIS_NONE, v)
            else:
                op.set_field(field, rq if mode == libceed.EVAL_NONE else rstr, libceed.BASIS_NONE if mode == libceed.EVAL_NONE else basis,
                             libceed.VECTOR_ACTIVE)
        uv, vv = ceed.Vector(nc * n), ceed.Vector(npts if outs[0][2] == libceed.EVAL_NONE else n)
        uv.set_array(u)
        print(name, "fuse", fuse, flush=True)
        op.apply(uv, vv)
        got.append(vv.to_numpy())
    assert np.linalg.norm(got[0]) > 0
    assert np.array_equal(got[0], got[1])
