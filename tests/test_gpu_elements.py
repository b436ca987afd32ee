"""Order 1 on many elements runs one thread per element: the same bits as the
line kernel reading the factors the plan hands out, in every kind of E^T, with
a last wavefront that is not full, overwriting and adding."""

import numpy as np
import pytest
import torch

from libceed_amd import ops
from libceed_amd.mesh import hex_mesh

pytestmark = pytest.mark.gpu


# (elements per side, Q, FP32, E^T mode): just below and above the number of elements of a launch from which the kernel
# runs (32768 for FP64 Q = 2, 98304 otherwise); in colours a launch has an eighth of the elements
@pytest.mark.parametrize("n,Q,fp32,scatter", [
    (31, 2, False, "tmap"), (33, 2, False, "tmap"), (33, 2, False, "split"), (65, 2, False, "color"), (33, 2, False, "atomic"),
    (46, 3, False, "tmap"), (47, 3, False, "tmap"), (47, 3, False, "split"), (93, 3, False, "color"), (47, 3, False, "atomic"),
    (47, 2, True, "tmap"), (47, 3, True, "tmap"), (47, 3, True, "split"), (93, 2, True, "color")])
def test_one_thread_per_element(cuda, n, Q, fp32, scatter):
    m = hex_mesh(n, 1, seed=n, perturb=0.3)
    dtype = torch.float32 if fp32 else torch.float64
    rng = np.random.default_rng(n + Q)
    u, w = (torch.from_numpy(rng.uniform(-1, 1, m.num_nodes)).to(dtype).cuda() for _ in range(2))
    op = ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, dtype=dtype, scatter=scatter)
    read = ops.HexOperator.from_mesh(ops.QF_DIFFUSION, m, Q=Q, dtype=dtype, scatter=scatter)
    read.set_qdata(op.get_qdata())
    print("elements", m.num_elem, "Q", Q, dtype, scatter, flush=True)
    v, ref, add, ref_add = torch.full_like(u, 3.0), torch.full_like(u, 4.0), w.clone(), w.clone()
    op.apply(u, v)
    op.apply_add(u, add)
    read.apply(u, ref)
    read.apply_add(u, ref_add)
    if scatter == "atomic":  # a node's eight terms in any order: seven roundings of partial sums below 8 max|term|
        tol = 64 * torch.finfo(dtype).eps * max(ref.abs().max().item(), 1.0)
        assert (v - ref).abs().max().item() <= tol and (add - ref_add).abs().max().item() <= tol
    else:
        assert torch.equal(v, ref) and torch.equal(add, ref_add)
