"""Geometric factors of elements without volume, inverted or not finite: the
trilinear map's factors are what the division w / det J makes of them, in the
stored factors and in the recomputing apply alike."""

import numpy as np
import pytest
import torch

import oracle
from libceed_amd import ops
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,Q,fp32", [(1, 2, False), (2, 4, False), (3, 5, True), (6, 8, False)])
def test_degenerate_elements(cuda, p, Q, fp32):
    m = hex_mesh(2, p, seed=1, perturb=0.2)
    flat, mirrored, broken = 0, 3, 6
    nv = m.num_vertices
    # each of the three elements gets eight vertices of its own
    coords = m.coords.reshape(3, nv)
    off = m.mesh_offsets.reshape(m.num_elem, 8).copy()
    extra = []
    for k, e in enumerate((flat, mirrored, broken)):
        x = coords[:, off[e]].copy()
        if e == flat:
            x = np.stack([x[0], x[1], np.full(8, 0.25)])
            x[:, 4:] = x[:, :4]  # top on bottom: d/dzeta is exactly 0
        elif e == mirrored:
            x = x[:, [1, 0, 3, 2, 5, 4, 7, 6]]
        else:
            x[0, 5] = np.inf
        extra.append(x)
        off[e] = nv + 8 * k + np.arange(8)
    coords = np.concatenate([coords] + extra, axis=1)
    dtype = torch.float32 if fp32 else torch.float64
    op = ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, dtype=dtype)
    op.build_qdata(off.reshape(-1), torch.from_numpy(coords.reshape(-1).copy()).cuda(), coords.shape[1])
    qd = op.get_qdata().cpu().numpy().reshape(m.num_elem, 6, Q ** 3)
    # flat: det J = 0, the cofactors of d/dxi and d/deta are 0 too and that of d/dzeta is not
    assert np.all(np.isposinf(qd[flat, 2]))
    assert np.all(np.isnan(qd[flat][[0, 1, 3, 4, 5]]))
    assert np.all(np.isnan(qd[broken]))
    want = oracle.hex_build_qdata(1, m, Q).reshape(m.num_elem, 6, Q ** 3)
    tol = 1e-5 if fp32 else 1e-12
    for e in range(m.num_elem):
        if e in (flat, broken):
            continue
        if e == mirrored:  # det J < 0
            assert np.all(qd[e, :3] < 0)
            continue
        assert np.linalg.norm(qd[e] - want[e]) < tol * np.linalg.norm(want[e])
    # the apply meets the same factors as one that reads them
    stored = ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, dtype=dtype)
    stored.set_qdata(op.get_qdata())
    u = torch.from_numpy(np.random.default_rng(0).uniform(-1, 1, m.num_nodes)).to(dtype).cuda()
    v, v_ref = torch.empty_like(u), torch.empty_like(u)
    op.apply(u, v)
    stored.apply(u, v_ref)
    assert torch.equal(torch.isnan(v), torch.isnan(v_ref))
    assert torch.equal(torch.nan_to_num(v, nan=0.0), torch.nan_to_num(v_ref, nan=0.0))
