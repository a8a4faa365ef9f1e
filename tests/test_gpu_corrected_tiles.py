"""General corrected bases in Float64 on both sides of the line (512 active tiles) where P2G gives a tile fewer waves:
the same particles in few tiles of one mesh, and among far more tiles."""
import numpy as np
import pytest
import torch

import tesserae_hip as th
from gpu_util import grid_np, rel_err, to_gpu
from oracle_bind import HostState
from tesserae_hip.scenes import random_box

pytestmark = pytest.mark.gpu

BASES = {"linear": th.WLS(th.BSpline(th.Linear())), "quadratic": th.WLS(th.BSpline(th.Quadratic())),
         "cubic": th.WLS(th.BSpline(th.Cubic())), "ugimp": th.WLS(th.uGIMP())}


@pytest.mark.parametrize("name", list(BASES))
@pytest.mark.parametrize("dim,h,lo,hi", [(2, 0.004, 0.3, 0.5), (2, 0.004, 0.02, 0.98), (3, 0.025, 0.3, 0.6),
                                         (3, 0.025, 0.03, 0.97)])
def test_wls_p2g_equals_the_oracle(oracle, name, dim, h, lo, hi):
    sc = random_box(dim, 3000, 11, BASES[name], dtype=torch.float64, h=h, lo=lo, hi=hi, stress=1.0,
                    with_l=name == "ugimp")
    _, P, G = to_gpu(sc)
    ctx = th.Context()
    th.P2G(G, P, sc.basis, sc.params, ctx=ctx)
    ctx.sync()
    assert (ctx.stats()["active_tiles"] >= 512) == (hi > 0.9)
    ctx.close()
    st = HostState(sc)
    oracle.p2g(st, sc.basis, sc.params)
    got = grid_np(G)
    for f, ref in (("m", st.m), ("mv", st.mv), ("f", st.f), ("vn", st.vn), ("v", st.gv)):
        assert rel_err(got[f], ref) <= 1e-10, f
