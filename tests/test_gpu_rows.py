"""G2P's ways of storing a particle (Float64 Julia-layout rows through LDS, strided stores, plain and non-temporal) and
of walking a tile (ids staged in LDS up to 2048 sorted slots in 3D, read from memory past them), P2G's Float64 kernel
with one register set: every layout and size against the oracle, and the two layouts against each other."""
import pytest
import torch

import tesserae_hip as th
from gpu_util import grid_np, particles_np, rel_err, to_gpu
from oracle_bind import HostState, Oracle
from tesserae_hip.scenes import random_box

pytestmark = pytest.mark.gpu

FIELDS = ("x", "v", "V", "grad_v", "F", "sigma")


def _scene(dim, n, basis, dtype, span):
    """n particles over `span` of the unit box, strained, in random order (no two neighbours in storage share a cell)."""
    return random_box(dim, n, 17 + n, basis, dtype=dtype, h=0.1, vscale=0.3, lo=0.41, hi=0.41 + span, stress=1.0)


@pytest.mark.parametrize("basis", [th.BSpline(th.Linear()), th.BSpline(th.Quadratic()), th.BSpline(th.Cubic())], ids=repr)
@pytest.mark.parametrize("n,span", [(1, 0.3), (63, 0.3), (65, 0.3), (2047, 0.35), (2500, 0.05), (9000, 0.3)])
def test_g2p_stores_and_walks_3d(basis, n, span):
    sc = _scene(3, n, basis, torch.float64, span)
    ref = HostState(sc)
    Oracle().step(ref, sc.basis, sc.params, 2)
    out = []
    for layout in ("julia", "soa"):
        mesh, P, G = to_gpu(sc, layout=layout)
        ctx = th.Context()
        th.step(G, P, sc.basis, sc.params, nsteps=2, ctx=ctx)
        ctx.sync()
        out.append((particles_np(P), grid_np(G)))
        ctx.close()
    (a, ga), (b, gb) = out
    for k in FIELDS:
        assert rel_err(a[k], getattr(ref, k)) <= 1e-10, k
        assert rel_err(a[k], b[k]) <= 1e-12, k
    for k in ("m", "mv"):
        assert rel_err(ga[k], gb[k]) <= 1e-12, k


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [65, 3000])
def test_streamed_and_plain_stores_agree(dim, n):
    """Float32: a loop that reorders at every step (streamed stores, the particles being put in the layered order) ends
    with the particles that a loop without reorders has (plain stores), told apart by their log E, bit for bit: the
    order of every sum is the same when no particle changes its key."""
    from tesserae_hip.scenes import uniform01
    sc = random_box(dim, n, 23, th.BSpline(th.Quadratic()), dtype=torch.float32, h=0.1, vscale=1e-4, lo=0.2, hi=0.8)
    sc.logE = uniform01(99, n)
    out = []
    for thr in (0.0, 1.0):
        mesh, P, G = to_gpu(sc)
        ctx = th.Context()
        th.step(G, P, sc.basis, sc.params, nsteps=3, reorder_threshold=thr, ctx=ctx)
        ctx.sync()
        assert ctx.stats()["movers"] in (0, -1)
        out.append(particles_np(P))
        ctx.close()
    a, b = out
    ia, ib = a["logE"].argsort(), b["logE"].argsort()
    for k in FIELDS:
        assert (a[k][ia] == b[k][ib]).all(), k
