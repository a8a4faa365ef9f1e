"""Many particles leave the mesh in one step of a loop: what follows, and that it takes no longer than steps that keep
them (both in one process on one device; each leaver once cost an atomic on one word, 6 times a plain call's time)."""
import os
import time

import numpy as np
import pytest
import torch

import tesserae_hip as th
from gpu_util import grid_np, particles_np, to_gpu
from tesserae_hip import _abi
from tesserae_hip.scenes import random_box

pytestmark = pytest.mark.gpu

QUADRATIC = th.BSpline(th.Quadratic())


def _scene(dim, n, dtype, h, shift):
    """Particles in the middle of the mesh that all move by `shift` along x in a step."""
    sc = random_box(dim, n, 3, QUADRATIC, dtype=dtype, h=h, lo=0.2, hi=0.8, vscale=0.0)
    sc.v[:, 0] = shift / 1e-3
    sc.params = th.MPMParams(dt=1e-3, E=1e-9, nu=0.3, rho0=1e3, V0=0.6 ** dim / n)
    return sc


def _time(call, reset, sync):
    best = np.inf
    for _ in range(5):
        reset()
        torch.cuda.synchronize()
        t = time.perf_counter()
        call()
        sync()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.skipif(not os.path.exists(_abi.DEBUG_LIB_PATH), reason="debug build not made")
@pytest.mark.parametrize("dim,h", [(2, 0.02), (3, 0.1)])
@pytest.mark.parametrize("n", [63, 5000, 20000])
@pytest.mark.parametrize("shift", [0.25, 0.5, 1.0])
def test_steps_that_lose_particles(dim, h, n, shift):
    """One call of steps (keys of the previous G2P) equals calls of one step (keys from the positions) bit for bit."""
    out = []
    for calls, per in ((1, 4), (4, 1)):
        sc = _scene(dim, n, torch.float64, h, shift)
        _, P, G = to_gpu(sc)
        ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
        for _ in range(calls):
            th.step(G, P, QUADRATIC, sc.params, nsteps=per, ctx=ctx)
        ctx.sync()
        assert ctx.stats()["n_inside"] < n
        out.append((particles_np(P), grid_np(G)))
        ctx.close()
    for a, b in zip(out[0], out[1]):
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=True), k


@pytest.mark.parametrize("dim,n,h", [(2, 800000, 1 / 256), (3, 1000000, 1 / 64)])
def test_steps_that_lose_particles_take_no_longer(dim, n, h):
    t = {}
    for shift in (0.3 * h, 1.0):
        sc = _scene(dim, n, torch.float32, h, shift)
        _, P, G = to_gpu(sc)
        x = P.x.clone()
        ctx = th.Context()

        def reset():
            P.x.copy_(x)
            P.set("v", sc.v)

        t[shift] = _time(lambda: th.step(G, P, QUADRATIC, sc.params, nsteps=5, ctx=ctx), reset, ctx.sync)
        ctx.close()
    assert t[1.0] <= 2.5 * t[0.3 * h], t


@pytest.mark.skipif(not os.path.exists(_abi.DEBUG_LIB_PATH), reason="debug build not made")
@pytest.mark.parametrize("dim,h", [(2, 0.02), (3, 0.1)])
@pytest.mark.parametrize("n", [2000, 2200, 9000, 40001])
def test_batches_that_lose_particles(dim, h, n):
    """Eager steps of a batch equal its captured steps bit for bit, on both sides of 2048 + n/256 arrivals outside."""
    out = []
    for variant in (0, 8):
        members = []
        for k, shift in ((n, 0.5), (n // 3, 0.1), (n // 2, 0.02)):
            sc = _scene(dim, k, torch.float64, h, shift)
            _, P, G = to_gpu(sc)
            members.append((G, P, sc.params))
        ctx = th.Context(library=_abi.DEBUG_LIB_PATH)
        b = th.Batch(members, QUADRATIC, ctx=ctx)
        b.set_variant(variant)
        b.step(6)
        ctx.sync()
        out.append([(particles_np(P), grid_np(G)) for G, P, _ in members])
        b.close()
        ctx.close()
    for (pa, ga), (pb, gb) in zip(*out):
        for a, b in ((pa, pb), (ga, gb)):
            for k in a:
                assert np.array_equal(a[k], b[k], equal_nan=True), k


@pytest.mark.parametrize("dim,n,h", [(2, 800000, 1 / 256), (3, 800000, 1 / 64)])
def test_captured_steps_that_lose_particles_take_no_longer(dim, n, h):
    t = {}
    for shift in (0.3 * h, 1.0):
        sc = _scene(dim, n, torch.float32, h, shift)
        _, P, G = to_gpu(sc)
        x = P.x.clone()
        ctx = th.Context()
        b = th.Batch([(G, P, sc.params)], QUADRATIC, ctx=ctx)
        b.set_variant(8)

        def reset():
            P.x.copy_(x)
            P.set("v", sc.v)

        t[shift] = _time(lambda: b.step(6), reset, ctx.sync)
        b.close()
        ctx.close()
    assert t[1.0] <= 2.5 * t[0.3 * h], t
