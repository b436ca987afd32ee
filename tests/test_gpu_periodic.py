"""Periodic meshes, down to one element per direction, whose elements reach a
node several times: the kernels that sum E^T in another way (in the apply's own
launch, one thread per element) give the bits of the column layout's gather."""

import numpy as np
import pytest
import torch

from libceed_amd import ops
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu


def periodic_offsets(m):
    """The mesh's nodes with the last layer of each direction folded onto the first: (offsets, number of nodes)."""
    nd = m.n * m.p + 1
    i = np.arange(nd ** 3)
    x, y, z = i % nd % (nd - 1), i // nd % nd % (nd - 1), i // nd ** 2 % (nd - 1)
    return ((z * (nd - 1) + y) * (nd - 1) + x).astype(np.int32)[m.offsets.reshape(-1)], (nd - 1) ** 3


@pytest.mark.parametrize("n,p,Q,in_launch", [(1, 1, 2, True), (1, 1, 3, True), (2, 1, 3, True), (1, 2, 4, True), (2, 2, 3, True), (1, 3, 5, True),
                                             (3, 3, 4, True), (2, 4, 6, False), (32, 1, 2, False), (47, 1, 3, False)])
def test_periodic(cuda, n, p, Q, in_launch):
    m = hex_mesh(n, p, seed=n)
    offsets, N = periodic_offsets(m)
    op, ref = (ops.HexOperator(ops.QF_DIFFUSION, offsets, m.num_elem, p + 1, Q, N, scatter="tmap") for _ in range(2))
    coords = torch.from_numpy(m.coords).cuda()
    for o in (op, ref):
        o.build_qdata(m.mesh_offsets, coords, m.num_vertices)
    op.set_layout(ops.LAYOUT_LINES)
    ref.set_layout(ops.LAYOUT_COLUMNS)
    assert op.kernel() == ("elements" if n >= 32 else "lines", not in_launch)
    rng = np.random.default_rng(p)
    for rep in range(3):
        u, w = (torch.from_numpy(rng.uniform(-1, 1, N)).cuda() for _ in range(2))
        v, v_ref, add, add_ref = torch.full_like(u, 3.0), torch.full_like(u, 4.0), w.clone(), w.clone()
        print(n, p, Q, rep, flush=True)
        op.apply(u, v)
        op.apply_add(u, add)
        ref.apply(u, v_ref)
        ref.apply_add(u, add_ref)
        assert torch.equal(v, v_ref) and torch.equal(add, add_ref)
