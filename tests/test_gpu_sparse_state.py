"""The state an SpGrid is left in: after a step that fails, and where the mesh has more blocks than the numbering adds
up without a prefix launch."""
import numpy as np
import pytest
import torch

import tesserae_hip as th
from gpu_util import grid_np, particles_np, rel_err, to_gpu
from tesserae_hip.scenes import random_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
def test_failed_step_leaves_the_length_of_its_numbering(dim):
    """A step renumbers the blocks and then refuses a particle length: the grid knows the storage its new numbering
    needs, so that a P2G on the storage at hand is refused, and a step with the length put right runs as on a dense
    grid."""
    basis = th.uGIMP()
    sc = random_box(dim, 2000, 3, basis, h=0.02 if dim == 2 else 0.05, lo=0.2, hi=0.3, with_l=True)
    sc.mesh.block_size_log2 = 1
    mesh, P, _ = to_gpu(sc)
    G = th.generate_grid(th.SpArray, mesh, device="cuda")
    ctx = th.Context()
    th.update_sparsity(G, P.x, ctx=ctx)
    capacity = G.capacity
    assert G.spinds.storage_len == capacity
    x = 0.2 + 6.0 * (sc.x - 0.2)  # spread over far more blocks
    bad = sc.l.copy()
    bad[7] = 2.0 * mesh.h
    P.set("x", x)
    P.set("l", bad)
    with pytest.raises(th.ArgumentError, match="uGIMP requires"):
        th.step(G, P, basis, sc.params, nsteps=2, ctx=ctx)
    blocks = int(G.spinds.blocknumbering.max())
    assert G.spinds.storage_len == blocks << dim and G.spinds.storage_len > capacity
    P.set("l", sc.l)
    with pytest.raises(th.DimensionMismatch):
        th.P2G(G, P, basis, sc.params, ctx=ctx)
    th.step(G, P, basis, sc.params, nsteps=2, ctx=ctx)
    ctx.sync()
    _, Pd, Gd = to_gpu(sc)
    Pd.set("x", x)
    th.step(Gd, Pd, basis, sc.params, nsteps=2, ctx=th.Context())
    torch.cuda.synchronize()
    a, b, dense = particles_np(P), particles_np(Pd), grid_np(Gd)
    for name in b:
        np.testing.assert_array_equal(a[name], b[name], err_msg=name)
    for name in dense:
        np.testing.assert_array_equal(G.to_dense(name), dense[name], err_msg=name)
    ctx.close()
