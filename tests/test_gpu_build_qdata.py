"""What building the factors leaves behind: the elements' maps stay in device
memory only where the plan's applies recompute factors from them, and a refused
build leaves the plan as it was."""

import gc

import numpy as np
import pytest
import torch

from libceed_amd import ops
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,keeps", [(ops.QF_MASS, False), (ops.QF_DIFFUSION, True)])
def test_memory_after_the_build(cuda, kind, keeps):
    m = hex_mesh(64, 1, seed=1)
    op = ops.HexOperator.from_mesh(kind, m, Q=2, build=False)
    coords = torch.from_numpy(m.coords).cuda()
    maps = 192 * m.num_elem
    gc.collect()  # plans of tests before this one
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    op.build_qdata(m.mesh_offsets, coords, m.num_vertices)
    torch.cuda.synchronize()
    taken = free - torch.cuda.mem_get_info()[0]
    assert (taken >= maps) if keeps else (taken < maps // 2), (taken, maps)


def test_refused_build(cuda):
    m, Q = hex_mesh(3, 2, seed=1), 4
    op = ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q)
    op.set_layout(ops.LAYOUT_LINES)  # whatever a tuner has found for such plans before
    u = torch.from_numpy(np.random.default_rng(0).uniform(-1, 1, m.num_nodes)).cuda()
    v, w = torch.empty_like(u), torch.empty_like(u)
    op.apply(u, v)
    with pytest.raises(ops.CeedMi355Error):
        op.build_qdata(m.mesh_offsets, torch.from_numpy(2 * m.coords).cuda(), m.num_vertices, mesh_P=Q + 1)
    assert op.recomputes_factors()
    op.apply(u, w)
    assert torch.equal(v, w)
