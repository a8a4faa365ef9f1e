"""The tile kernels of stored and of general corrected weights, several waves to a tile: particles spread thin, classes
with fewer particles than a tile has waves, a tile past the ids that LDS holds (1024), windows cut by the wall (rows not
whole), contiguous fields and weights and strided ones, against the oracle."""
import pytest
import torch

import tesserae_hip as th
from gpu_util import grid_np, particles_np, rel_err, to_gpu
from oracle_bind import HostState, Oracle
from tesserae_hip.scenes import random_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis", [th.BSpline(th.Linear()), th.BSpline(th.Quadratic()), th.BSpline(th.Cubic()),
                                   th.WLS(th.BSpline(th.Quadratic()))], ids=repr)
@pytest.mark.parametrize("dim,n,lo,span", [(2, 1, 0.4, 0.2), (2, 67, 0.0, 0.9), (2, 3000, 0.21, 0.06),
                                           (3, 65, 0.0, 0.9), (3, 2500, 0.21, 0.06)])
@pytest.mark.parametrize("layout", ["julia", "soa"])
def test_stored_tiles(basis, dim, n, lo, span, layout):
    sc = random_box(dim, n, 29 + n, basis, dtype=torch.float64, h=0.1, vscale=0.3, lo=lo, hi=lo + span, stress=1.0)
    ref = HostState(sc)
    o = Oracle()
    Wo = o.update_weights(ref, sc.basis)
    o.p2g(ref, sc.basis, sc.params, Wo)
    o.g2p(ref, sc.basis, sc.params, Wo)
    for deferred in (False, True):
        mesh, P, G = to_gpu(sc, layout=layout)
        W = th.generate_basis_weights(sc.basis, mesh, sc.n, deferred=deferred)
        th.update(W, P, mesh)
        th.P2G(G, P, W, sc.params)
        th.G2P(G, P, W, sc.params)
        torch.cuda.synchronize()
        g, p = grid_np(G), particles_np(P)
        wls = "WLS" in repr(basis)  # a 3 x 3 or 4 x 4 moment solve per particle, its condition below 1e3
        for k, r in (("m", ref.m), ("mv", ref.mv), ("f", ref.f), ("v", ref.gv)):
            assert rel_err(g[k], r) <= (1e-10 if wls else 1e-12), (k, deferred)
        for k in ("x", "v", "V", "grad_v", "F", "sigma"):
            assert rel_err(p[k], getattr(ref, k)) <= (1e-9 if wls else 1e-10), (k, deferred)
