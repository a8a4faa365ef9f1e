"""What a P2G leaves on a grid is its own: the node blocks that an earlier P2G on the same grid wrote and this one does
not touch are zero again, whatever the context did in between.

Each case moves the particles to another part of the mesh and compares every grid field with that of a fresh context
and a fresh grid (Float64; the particles may be summed in another order: 1e-12)."""
import numpy as np
import pytest
import torch

import tesserae_hip as th
from gpu_util import grid_np, rel_err, to_gpu
from tesserae_hip.scenes import random_box, uniform01

pytestmark = pytest.mark.gpu

QUADRATIC = th.BSpline(th.Quadratic())


def _p2g_alone(sc, x):
    """The grid of one P2G at x on a context and a grid of its own."""
    _, P, G = to_gpu(sc)
    P.set("x", x)
    ctx = th.Context()
    th.P2G(G, P, sc.basis, sc.params, ctx=ctx)
    ctx.sync()
    out = grid_np(G)
    ctx.close()
    return out


def _equal_grids(got, ref, what):
    for name in ref:
        assert rel_err(got[name], ref[name]) <= 1e-12, (what, name)
        assert not np.any(got[name][ref[name] == 0.0]), (what, name)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("fine", [1, 4], ids=["same-tiles", "more-tiles"])
@pytest.mark.parametrize("between", [1, 2, 3])
def test_g2p_on_another_mesh_between_two_p2g(dim, fine, between):
    """P2G(A), G2P(B) some times, P2G(A): no P2G on B tells the context that the grid changed, and B's tables (of as
    many tiles as A's, or of more than A's buffers hold) are built in the sets that held the node blocks of A."""
    h = 0.02 if dim == 2 else 0.05
    a = random_box(dim, 700, 3, QUADRATIC, h=h, lo=0.1, hi=0.3)
    b = random_box(dim, 900, 5, QUADRATIC, h=h / fine, lo=0.1, hi=0.9, vscale=30.0)
    _, Pa, Ga = to_gpu(a)
    _, Pb, Gb = to_gpu(b)
    ctx = th.Context()
    th.P2G(Ga, Pa, a.basis, a.params, ctx=ctx)
    for k in range(between):
        Pb.set("x", 0.1 + 0.8 * uniform01(40 + k, b.n * dim).reshape(b.n, dim))
        th.G2P(Gb, Pb, b.basis, b.params, ctx=ctx)
    x = a.x + 0.5
    Pa.set("x", x)
    th.P2G(Ga, Pa, a.basis, a.params, ctx=ctx)
    ctx.sync()
    _equal_grids(grid_np(Ga), _p2g_alone(a, x), between)
    ctx.close()


@pytest.mark.parametrize("nsteps,every,repeats", [(2, 10, 1), (3, 10, 1), (2, 1, 2), (21, 10, 2), (11, 10, 3)])
def test_p2g_after_a_pullback(nsteps, every, repeats):
    """A rollout whose steps re-bin, its pullback, then a P2G elsewhere on the same grid: the pullback works from kept
    binnings of other steps, which say nothing about what the rollout's last P2G wrote."""
    sc = random_box(2, 600, 7, QUADRATIC, h=0.02, lo=0.1, hi=0.3)
    sc.v[:] = (5.0, 3.0)  # a quarter of a cell per step: some particles change their cell in every step
    _, P, G = to_gpu(sc)
    ctx = th.Context()
    adj = th.Adjoint(sc.n, 2)
    for r in range(repeats):
        P.set("x", sc.x)
        P.set("v", sc.v)
        P.set("F", sc.F)
        th.rollout(G, P, sc.basis, sc.params, nsteps, checkpoint_every=every, ctx=ctx)
        adj.x.fill_(1.0)
        th.rollout_adjoint(G, sc.basis, sc.params, adj, ctx=ctx)
        _, P0, _ = to_gpu(sc)
        x = sc.x + 0.5 - 0.1 * r
        P0.set("x", x)
        th.P2G(G, P0, sc.basis, sc.params, ctx=ctx)
        ctx.sync()
        _equal_grids(grid_np(G), _p2g_alone(sc, x), r)
    ctx.close()


def _on_mesh(sc, mesh):
    out = sc.copy()
    out.mesh = mesh
    return out


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("shared", [False, True], ids=["own-grid", "shared-grid"])
def test_meshes_of_equal_counts(dim, shared):
    """Two meshes with as many nodes and tiles, their axes exchanged: the particles' keys are the same numbers on both
    (they lie in the first tile), but not the node blocks around them.  With `shared` the second mesh takes over the
    arrays of the first one's grid."""
    h = 1.0 / 32
    ends = (1.0, 2.0) if dim == 2 else (0.5, 1.0, 0.75)
    mesh_a = th.CartesianMesh(h, *[(0.0, e) for e in ends], dtype=torch.float64)
    mesh_b = th.CartesianMesh(h, *[(0.0, e) for e in ends[::-1]], dtype=torch.float64)
    assert mesh_a.nnodes() == mesh_b.nnodes() and tuple(mesh_a.size()) != tuple(mesh_b.size())
    sc = random_box(dim, 500, 3, QUADRATIC, h=h, lo=0.01, hi=0.09 if dim == 3 else 0.23)
    a, b = _on_mesh(sc, mesh_a), _on_mesh(sc, mesh_b)
    _, P, Ga = to_gpu(a)
    _, _, Gb = to_gpu(b)
    if shared:
        Gb.tensors = Ga.tensors
    ctx = th.Context()
    for s, G in ((a, Ga), (b, Gb), (a, Ga)):
        th.P2G(G, P, s.basis, s.params, ctx=ctx)
        ctx.sync()
        _equal_grids(grid_np(G), _p2g_alone(s, sc.x), "a" if s is a else "b")
    ctx.close()
