"""Small plans sum E^T in the apply's own launch (the last contribution to
arrive at an entry adds them up): the same bits as the launch that gathers
(the column layout's), call after call, overwriting and adding, on a structured
and on a shuffled numbering, and in a replayed graph."""

import numpy as np
import pytest
import torch

from libceed_amd import ops
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu


# one element; the last mesh within 256 workgroups and the first beyond at p = 1 (7 elements in one) and p = 2 (4 in one)
@pytest.mark.parametrize("n,p,Q,kind,fp32", [(1, 1, 2, 1, False), (12, 1, 3, 1, False), (13, 1, 3, 1, False), (10, 2, 4, 1, False), (11, 2, 4, 1, False),
                                             (6, 2, 4, 1, True), (6, 2, 3, 0, False), (9, 3, 5, 1, False), (10, 3, 4, 0, True)])
@pytest.mark.parametrize("shuffled", [False, True])
def test_last_contribution_sums(cuda, n, p, Q, kind, fp32, shuffled):
    m = hex_mesh(n, p, seed=n)
    rng = np.random.default_rng(n + 10 * p)
    dtype = torch.float32 if fp32 else torch.float64
    offsets = m.offsets
    if shuffled:
        offsets = rng.permutation(m.num_nodes).astype(np.int32)[m.offsets.reshape(m.num_elem, -1)[rng.permutation(m.num_elem)]].reshape(-1)
    op = ops.HexOperator(kind, offsets, m.num_elem, p + 1, Q, m.num_nodes, dtype=dtype, scatter="tmap")
    ref = ops.HexOperator(kind, offsets, m.num_elem, p + 1, Q, m.num_nodes, dtype=dtype, scatter="tmap")
    qd = torch.from_numpy(rng.uniform(0.5, 1.5, m.num_elem * op.q_comp * Q ** 3)).to(dtype).cuda()
    op.set_qdata(qd)
    ref.set_qdata(qd)
    ref.set_layout(ops.LAYOUT_COLUMNS)
    print("n", n, "p", p, "Q", Q, "kind", kind, dtype, "launch", op.launch(), flush=True)
    for rep in range(4):
        u, w = (torch.from_numpy(rng.uniform(-1, 1, m.num_nodes)).to(dtype).cuda() for _ in range(2))
        v, v_ref, add, add_ref = torch.full_like(u, 3.0), torch.full_like(u, 4.0), w.clone(), w.clone()
        op.apply(u, v)
        op.apply_add(u, add)
        ref.apply(u, v_ref)
        ref.apply_add(u, add_ref)
        assert torch.equal(v, v_ref) and torch.equal(add, add_ref)
    u_ref = u.clone()  # v in u's place, as where a gather follows
    op.apply(u, u)
    ref.apply(u_ref, u_ref)
    assert torch.equal(u, u_ref)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        op.apply(u, v)
        op.apply_add(v, add)
    for rep in range(3):
        u.copy_(torch.from_numpy(rng.uniform(-1, 1, m.num_nodes)).to(dtype))
        add.copy_(w)
        add_ref.copy_(w)
        g.replay()
        torch.cuda.synchronize()
        ref.apply(u, v_ref)
        ref.apply_add(v_ref, add_ref)
        assert torch.equal(v, v_ref) and torch.equal(add, add_ref)
        op.apply(u, v)  # eager between the replays
        assert torch.equal(v, v_ref)
