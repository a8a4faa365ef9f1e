"""Re-binnings that sort every key in place of merging the changed ones: too many arrivals in one tile, tiles too full for
one workgroup, particles put elsewhere altogether, particles that come back into the mesh.

Run through the debug build, which checks every binning on the host.  The sizes lie on both sides of the lines (2048 +
n/256 arrivals of a tile, 4096 + n/128 particles in a tile, an eighth of the waves with three quarters of
their first 64 particles gone to other tiles) and of the merge's LDS list (512 arrivals)."""
import os

import numpy as np
import pytest
import torch

import tesserae_hip as th
from gpu_util import grid_np, particles_np, rel_err, to_gpu
from tesserae_hip import _abi
from tesserae_hip.scenes import random_box, uniform01

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not os.path.exists(_abi.DEBUG_LIB_PATH), reason="debug build not made")]

QUADRATIC = th.BSpline(th.Quadratic())


def _positions(dim, n, h):
    """Position sets by name; one tile lies around 0.3."""
    u = [uniform01(70 + k, n * dim).reshape(n, dim) for k in range(4)]
    spread = 0.05 + 0.9 * u[0]
    tile = 0.3 + 0.5 * h * u[1]

    def part(k, where):
        x = spread.copy()
        x[::k] = where[::k]
        return x

    return {"spread": spread, "again": spread.copy(), "tile": tile, "tile again": tile.copy(), "outside": 1.5 + u[2],
            "a tenth into one tile": part(10, tile), "a tenth outside": part(10, 1.5 + u[2]), "anew": 0.05 + 0.9 * u[3]}


ORDER = ["spread", "again", "tile", "tile again", "spread", "a tenth into one tile", "spread", "anew", "a tenth outside",
         "outside", "outside", "tile", "outside", "spread", "tile", "anew"]


@pytest.mark.parametrize("dim,h", [(2, 0.05), (2, 0.02), (3, 0.1)])
@pytest.mark.parametrize("n", [1800, 6000, 30000])
def test_replaced_positions(dim, h, n):
    """P2G after every such change equals a fresh context's to Float64 rounding (the particles of a class are summed in
    another order)."""
    sc = random_box(dim, n, 7, QUADRATIC, h=h)
    sets = _positions(dim, n, h)
    _, P, G = to_gpu(sc)
    ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
    ref = {}
    for k, name in enumerate(ORDER):
        P.set("x", sets[name])
        th.P2G(G, P, sc.basis, sc.params, ctx=ctx)
        ctx.sync()
        got, stats = grid_np(G), ctx.stats()
        if name not in ref:
            _, P2, G2 = to_gpu(sc)
            P2.set("x", sets[name])
            c2 = th.Context()
            th.P2G(G2, P2, sc.basis, sc.params, ctx=c2)
            c2.sync()
            ref[name] = grid_np(G2), c2.stats()
            c2.close()
        grid, st = ref[name]
        for f in grid:
            assert rel_err(got[f], grid[f]) <= 1e-12, (k, name, f)
        for s in ("n_inside", "active_tiles", "node_blocks"):
            assert stats[s] == st[s], (k, name, s)
        if name in ("again", "tile again"):
            assert stats["movers"] == 0, (k, name)
    ctx.close()


@pytest.mark.parametrize("dim,h", [(2, 0.125), (3, 0.25)])
@pytest.mark.parametrize("n", [3000, 20000])
def test_step_loops_in_few_tiles(dim, h, n):
    """One call of steps (keys of the previous G2P) equals calls of one step (keys from the positions) bit for bit where
    a handful of tiles holds every particle; fast particles change their tile, leave the mesh and stay out."""
    sc = random_box(dim, n, 3, QUADRATIC, h=h, vscale=25.0, lo=0.05, hi=0.95)
    out = []
    for calls, per in ((1, 5), (5, 1)):
        _, P, G = to_gpu(sc)
        ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
        for _ in range(calls):
            th.step(G, P, sc.basis, sc.params, nsteps=per, ctx=ctx)
        ctx.sync()
        assert ctx.stats()["movers"] > 0
        out.append((particles_np(P), grid_np(G)))
        ctx.close()
    for a, b in zip(out[0], out[1]):
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=True), k


@pytest.mark.parametrize("dim,h", [(2, 0.125), (3, 0.25)])
def test_batches_in_few_tiles(dim, h):
    """Eager steps of a batch (which sort) equal its captured steps (which always merge) bit for bit."""
    out = []
    for variant in (0, 8):
        scenes = [random_box(dim, n, 5 + n, QUADRATIC, h=h, vscale=25.0, lo=0.05, hi=0.95) for n in (20000, 3000)]
        members = []
        for sc in scenes:
            _, P, G = to_gpu(sc)
            members.append((G, P, sc.params))
        ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
        b = th.Batch(members, QUADRATIC, ctx=ctx)
        b.set_variant(variant)
        b.step(5)
        ctx.sync()
        out.append([(particles_np(P), grid_np(G)) for G, P, _ in members])
        b.close()
        ctx.close()
    for eager, captured in zip(*out):
        for a, c in zip(eager, captured):
            for k in a:
                assert np.array_equal(a[k], c[k], equal_nan=True), k
