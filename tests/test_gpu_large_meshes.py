"""Meshes past the sizes whose per-workgroup sums the table kernels add up by themselves (1,048,576 tiles; 262,144 SpGrid
blocks): a launch of its own makes the prefix there."""
import os

import numpy as np
import pytest
import torch

import tesserae_hip as th
from gpu_util import grid_np, particles_np, rel_err, to_gpu
from tesserae_hip import _abi
from tesserae_hip.scenes import random_box, uniform01

pytestmark = pytest.mark.gpu

QUADRATIC = th.BSpline(th.Quadratic())
NODES, SMALL, PER = 8200, 65, 400  # 1025 x 1025 tiles; a cluster's own mesh; particles per cluster
ORIGINS = [(0, 0), (4096, 2048), (8192 - 56, 8192 - 56), (8, 8192 - 56)]  # multiples of the tile's 8 cells


def _cluster(k, origin):
    """Particles around the middle of a mesh of SMALL nodes at `origin`, spacing 1."""
    sc = random_box(2, PER, 20 + k, QUADRATIC, h=1.0, extent=float(SMALL - 1), lo=20.0, hi=36.0, vscale=400.0)
    sc.mesh = th.CartesianMesh(1.0, *[(float(o), float(o + SMALL - 1)) for o in origin], dtype=torch.float64)
    sc.x = sc.x + np.array(origin, dtype=np.float64)
    sc.params = th.MPMParams(dt=1e-3, E=1e3, nu=0.3, rho0=1e3, V0=1.0)
    return sc


@pytest.mark.skipif(not os.path.exists(_abi.DEBUG_LIB_PATH), reason="debug build not made")
def test_tables_of_a_million_tiles():
    """Far apart clusters on one mesh equal each cluster on a mesh of its own: a full binning, one that keeps its tables,
    one of replaced positions, and a loop whose keys the G2P writes.  (Spacing 1 and origins at whole tiles: the same
    weights, to the bit.)"""
    parts = [_cluster(k, o) for k, o in enumerate(ORIGINS)]
    big = parts[0].copy()
    big.mesh = th.CartesianMesh(1.0, (0.0, NODES - 1.0), (0.0, NODES - 1.0), dtype=torch.float64)
    for name in ("x", "v", "V", "F", "sigma", "grad_v"):
        setattr(big, name, np.concatenate([getattr(p, name) for p in parts]))
    _, P, G = to_gpu(big)
    small = [to_gpu(p) for p in parts]
    ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
    ctxs = [th.Context() for _ in parts]
    replaced = [8.0 + 48.0 * uniform01(60 + k, 2 * PER).reshape(PER, 2) + np.array(o) for k, o in enumerate(ORIGINS)]
    for what in ("full", "kept", "replaced", "steps"):
        if what == "replaced":
            P.set("x", np.concatenate(replaced))
            for (_, p, _), x in zip(small, replaced):
                p.set("x", x)
        if what == "steps":
            th.step(G, P, QUADRATIC, big.params, nsteps=4, ctx=ctx)
        else:
            th.P2G(G, P, QUADRATIC, big.params, ctx=ctx)
        ctx.sync()
        got = particles_np(P)
        for k, ((_, p, g), c, o) in enumerate(zip(small, ctxs, ORIGINS)):
            if what == "steps":
                th.step(g, p, QUADRATIC, big.params, nsteps=4, ctx=c)
            else:
                th.P2G(g, p, QUADRATIC, big.params, ctx=c)
            c.sync()
            ref, rp = grid_np(g), particles_np(p)
            for name in ref:
                t = G.get(name).reshape(NODES, NODES, -1)[o[1]:o[1] + SMALL, o[0]:o[0] + SMALL]
                t = torch.nn.functional.pad(t, (0, 0, 0, SMALL - t.shape[1], 0, SMALL - t.shape[0]))
                assert rel_err(t.reshape(SMALL * SMALL, -1).cpu().numpy(), ref[name].reshape(SMALL * SMALL, -1)) <= 1e-12, (
                    what, k, name)
            for name in rp:
                assert rel_err(got[name][k * PER:(k + 1) * PER], rp[name]) <= 1e-9, (what, k, name)
        # nothing elsewhere
        nonzero = sum(int((g.get("m") != 0).sum()) for _, _, g in small)
        assert int((G.get("m") != 0).sum()) == nonzero, what
    assert ctx.stats()["kept_binnings"] >= 1 and ctx.stats()["movers"] > 0
    for c in [ctx] + ctxs:
        c.close()


def test_numbering_of_many_blocks(oracle):
    """275,625 blocks: numbering and length equal the oracle's, an unchanged set is reported as such."""
    mesh = th.CartesianMesh(1.0, (0.0, 2099.0), (0.0, 2099.0), dtype=torch.float64, block_size_log2=2)
    G = th.generate_grid(th.SpArray, mesh, device="cuda")
    for seed, n in ((1, 5000), (2, 300), (3, 40000)):
        x = 2110.0 * uniform01(seed, 2 * n).reshape(n, 2) - 5.0
        xt = torch.from_numpy(x).cuda()
        got = th.update_sparsity(G, xt)
        num, length, _ = oracle.sparsity(mesh, x, dtype=np.float64)
        np.testing.assert_array_equal(G.spinds.blocknumbering.cpu().numpy(), num)
        assert got == length == G.spinds.storage_len
        assert th.update_sparsity(G, xt) is None
