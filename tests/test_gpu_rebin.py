"""Re-binning between steps: the merge of the particles whose key changed (from the keys the previous G2P wrote, or
from the positions) against a full sort.

Run through the debug build, which checks every binning on the host (permutation, sorted keys, tile runs, lists).
Sizes sit at the edges the kernels have: a wave (64), a workgroup (256), one tile holding more arrivals than the
merge's LDS list (512), particles that leave the mesh and come back."""
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


@pytest.mark.parametrize("dim,n,vscale", [(2, 64, 40.0), (2, 1000, 25.0), (3, 257, 40.0), (3, 5000, 25.0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_step_loop_equals_single_step_calls(dim, n, vscale, dtype):
    """One call of 6 steps (keys from the previous G2P) equals 6 calls of one step on a context (keys from the
    positions) bit for bit: both merges give the stable order, which fixes the order of every sum.  Fast particles
    cross several cells per step and leave the mesh."""
    sc = random_box(dim, n, 3 + n, th.BSpline(th.Quadratic()), dtype=dtype, h=0.1, vscale=vscale, lo=0.05, hi=0.95)
    out = []
    for calls, per in ((1, 6), (6, 1)):
        mesh, P, G = to_gpu(sc)
        ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
        for _ in range(calls):
            th.step(G, P, sc.basis, sc.params, nsteps=per, ctx=ctx)
        ctx.sync()
        moved = ctx.stats()["movers"]
        out.append((particles_np(P), grid_np(G)))
        ctx.close()
    assert moved > 0
    for a, b in zip(out[0], out[1]):
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=True), k


def _positions(dim, n, seed):
    """A sequence of position sets: spread, into one tile, all outside, back inside, half outside, spread."""
    u = [uniform01(seed + 10 * k, n * dim).reshape(n, dim) for k in range(6)]
    half = 0.1 + 0.8 * u[4]
    half[::2] += 2.0
    return [0.1 + 0.8 * u[0], 0.41 + 0.08 * u[1], 1.5 + u[2], 0.1 + 0.8 * u[3], half, 0.1 + 0.8 * u[5]]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 63, 65, 513, 3000])
def test_rebinning_of_replaced_positions(dim, n):
    """P2G on a context whose previous binning belongs to other positions equals a fresh context's: the merge orders
    particles of one class differently from a fresh sort, so the sums agree to Float64 rounding."""
    sc = random_box(dim, n, 7, th.BSpline(th.Quadratic()), dtype=torch.float64, h=0.02 if dim == 2 else 0.05)
    mesh, P, G = to_gpu(sc)
    ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
    for k, x in enumerate(_positions(dim, n, 11)):
        P.set("x", x)
        th.P2G(G, P, sc.basis, sc.params, ctx=ctx)
        ctx.sync()
        got = grid_np(G)
        mesh2, P2, G2 = to_gpu(sc)
        P2.set("x", x)
        ref_ctx = th.Context()
        th.P2G(G2, P2, sc.basis, sc.params, ctx=ref_ctx)
        ref_ctx.sync()
        ref = grid_np(G2)
        for f in ref:
            assert rel_err(got[f], ref[f]) <= 1e-12, (k, f)
        assert ctx.stats()["n_inside"] == ref_ctx.stats()["n_inside"]
        assert ctx.stats()["node_blocks"] == ref_ctx.stats()["node_blocks"]
        ref_ctx.close()
    ctx.close()


@pytest.mark.parametrize("dim,basis,n", [(2, th.BSpline(th.Quadratic()), 1), (2, th.uGIMP(), 900),
                                         (3, th.BSpline(th.Cubic()), 65), (3, th.BSpline(th.Quadratic()), 4000)])
@pytest.mark.parametrize("layout", ["julia", "soa"])
@pytest.mark.parametrize("threshold,steps", [(1.0, 5), (1.0, 4), (0.85, 6)])
def test_reorders_of_a_loop(dim, basis, n, layout, threshold, steps):
    """Reorders in a loop (the G2P of the step writes the particles at their new places): one call equals calls of one
    step bit for bit where every step reorders, and either gives each particle (told apart by its log E) the state it
    has without reorders.  Some particles leave the mesh; odd and even numbers of reorders end a call."""
    sc = random_box(dim, n, 5 + n, basis, dtype=torch.float64, h=0.1, vscale=20.0, lo=0.03, hi=0.97,
                    with_l=basis.kernel == 16)
    sc.logE = 0.1 * uniform01(99, n)
    if sc.l is not None:
        sc.l = sc.l * (0.5 + uniform01(98, n))

    def run(calls, per, thr):
        mesh, P, G = to_gpu(sc, layout=layout)
        ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
        for _ in range(calls):
            th.step(G, P, sc.basis, sc.params, nsteps=per, reorder_threshold=thr, ctx=ctx)
        ctx.sync()
        st = ctx.stats()
        ctx.close()
        return particles_np(P), grid_np(G), st

    got, ggrid, st = run(1, steps, threshold)
    plain, pgrid, _ = run(1, steps, 0.0)
    if threshold == 1.0:
        assert st["reorders"] == steps
        one, ogrid, _ = run(steps, 1, threshold)
        for k in got:
            assert np.array_equal(got[k], one[k]), k
        for k in ggrid:
            assert np.array_equal(ggrid[k], ogrid[k]), k
    ia, ib = np.argsort(got["logE"]), np.argsort(plain["logE"])
    for k in got:
        assert rel_err(got[k][ia], plain[k][ib]) <= 1e-9, k
    assert rel_err(ggrid["m"], pgrid["m"]) <= 1e-12


@pytest.mark.parametrize("layout", ["julia", "soa"])
@pytest.mark.parametrize("passes", [3, 4])
def test_reorders_of_a_g2p2g_loop(layout, passes):
    """The same for @G2P2G passes, whose P2G half follows the G2P that moves the particles."""
    sc = random_box(3, 2000, 8, th.BSpline(th.Quadratic()), dtype=torch.float64, h=0.1, vscale=10.0, lo=0.1, hi=0.9)
    sc.logE = 0.1 * uniform01(99, sc.n)
    out = []
    for thr in (0.0, 1.0):
        mesh, P, G = to_gpu(sc, layout=layout)
        ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
        th.P2G(G, P, sc.basis, sc.params, ctx=ctx)
        th.g2p2g_steps(G, P, sc.basis, sc.params, nsteps=passes, reorder_threshold=thr, ctx=ctx)
        ctx.sync()
        assert ctx.stats()["reorders"] == (passes if thr else 0)
        out.append((particles_np(P), grid_np(G)))
        ctx.close()
    (a, ga), (b, gb) = out
    ia, ib = np.argsort(a["logE"]), np.argsort(b["logE"])
    for k in a:
        assert rel_err(b[k][ib], a[k][ia]) <= 1e-9, k
    assert rel_err(gb["m"], ga["m"]) <= 1e-12


@pytest.mark.parametrize("n", [700, 3000])
def test_rebinning_spreads_over_many_tiles(n):
    """Particles of one tile spread over some 900 at once and gather again: far more active tiles than the merge launched
    behind the tables allows for, then far fewer; P2G equals a fresh context's to Float64 rounding."""
    sc = random_box(2, n, 7, th.BSpline(th.Quadratic()), dtype=torch.float64, h=0.004)
    mesh, P, G = to_gpu(sc)
    ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
    spread = 0.01 + 0.98 * (sc.x - sc.x.min(0)) / (sc.x.max(0) - sc.x.min(0))
    for k, x in enumerate((0.5 + 0.02 * spread, spread, 0.3 + 0.02 * spread, spread[::-1].copy())):
        P.set("x", x)
        th.P2G(G, P, sc.basis, sc.params, ctx=ctx)
        ctx.sync()
        got, stats = grid_np(G), ctx.stats()
        mesh2, P2, G2 = to_gpu(sc)
        P2.set("x", x)
        ref_ctx = th.Context()
        th.P2G(G2, P2, sc.basis, sc.params, ctx=ref_ctx)
        ref_ctx.sync()
        ref = grid_np(G2)
        for f in ref:
            assert rel_err(got[f], ref[f]) <= 1e-12, (k, f)
        assert stats["active_tiles"] == ref_ctx.stats()["active_tiles"]
        assert (stats["active_tiles"] > 400) == (k % 2 == 1)
        ref_ctx.close()
    ctx.close()
