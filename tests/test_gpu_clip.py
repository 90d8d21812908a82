"""The batched per-patch kernels against the oracle, bit for bit, at the sizes
where a wave's sharing and remainders can go wrong: tolerances whose square
decides convergence, pairs that share a wave with none, one or many others,
hits tied between regions, and waves of patches with a remainder."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rng, say
from test_gpu_parity import assert_bits_equal, random_patch_pairs

pytestmark = pytest.mark.gpu


def clip_equal(ctx, oracle, rays, P, tol=2.0 ** -12):
    out = ctx.bezier_clip(rays, P, tol)
    o, w = oracle.clip_batch(rays, P, tol)
    assert w["overflows"] == 0
    assert np.array_equal(out.view(np.uint32)[:, 3] == 1, o[:, 3] == 1)
    assert_bits_equal(out[:, :3], o[:, :3], "t,u,v")
    return w


@pytest.mark.parametrize("tol", [2.0 ** -12, 2.0 ** -4, 1e-3, 0.3, 1e20])
def test_tolerances(ctx, oracle, tol):
    say("bezier_clip: tolerance", tol)
    clip_equal(ctx, oracle, *random_patch_pairs(5000, 33), tol=tol)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000])
def test_wave_remainders(ctx, oracle, n):
    """Idle lanes take regions of the few busy ones (n below a wave)."""
    say("bezier_clip, subdivision: pairs", n)
    rays, P = random_patch_pairs(n, 40 + n)
    clip_equal(ctx, oracle, rays, P)
    subdivide_equal(ctx, oracle, rays, P, 2.0 ** -4)


def subdivide_equal(ctx, oracle, rays, P, threshold):
    g = ctx.subdivision(rays, P, threshold)
    o, w = oracle.clip_batch(rays, P, method=1, threshold=threshold)
    assert np.array_equal(g.view(np.uint32)[:, 3] == 1, o[:, 3] == 1)
    assert_bits_equal(g[:, :3], o[:, :3], "t,u,v")


@pytest.mark.parametrize("n", [40_003, 70_003, 100_003, 131_137])
def test_pairs_of_full_waves(ctx, oracle, n):
    """16 to 64 pairs a wave, with a remainder: waves whose lanes share only when
    some have ended, and waves that hold more than one load of pairs."""
    say("bezier_clip, subdivision: pairs", n)
    rays, P = random_patch_pairs(4099, 34)
    at = np.arange(n) % 4099
    for method in (0, 1):
        g = ctx.subdivision(rays[at], P[at], 0.25) if method else ctx.bezier_clip(rays[at], P[at])
        o, _ = oracle.clip_batch(rays, P, method=method, **(dict(threshold=0.25) if method else {}))
        assert np.array_equal(g.view(np.uint32)[:, 3] == 1, o[at, 3] == 1)
        assert_bits_equal(g[:, :3], o[at, :3], "t,u,v")


def grazing_pairs(n, seed):
    """Rays nearly in the plane of nearly flat patches: hundreds of passes over
    as many regions, shared by the whole wave."""
    r = rng(seed)
    size = 8.0
    g = np.linspace(0, size, 4)
    P = np.zeros((n, 16, 4), np.float32)
    P[:, :, 0], P[:, :, 1] = np.tile(g, 4), np.repeat(g, 4)
    P[:, :, 2] = r.uniform(-1e-4, 1e-4, (n, 16))
    P[:, :, 3] = 1.0
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0], rays[:, 1] = -0.2 * size, r.uniform(0.1, 0.9, n) * size
    rays[:, 2] = r.uniform(-5e-5, 5e-5, n)
    rays[:, 3] = np.inf
    rays[:, 4:7] = np.stack([np.ones(n), r.uniform(-0.3, 0.3, n), r.uniform(-1e-6, 1e-6, n)], 1)
    return rays, P


@pytest.mark.parametrize("n", [5, 64, 200])
def test_grazing_pairs(ctx, oracle, n):
    say("bezier_clip, subdivision: grazing pairs", n)
    rays, P = grazing_pairs(n, 50)
    w = clip_equal(ctx, oracle, rays, P)
    assert w["subdivs"] > 40 * n
    subdivide_equal(ctx, oracle, rays, P, 2.0 ** -5)


@pytest.mark.parametrize("threshold", [0.6, 2.0 ** -1, 2.0 ** -8])
def test_tied_hits(ctx, oracle, threshold):
    """Flat patches folded onto themselves (u and 1 - u at the same point):
    every hit is found at the same distance in two regions, and the first in
    the reference's order is reported."""
    say("bezier_clip, subdivision: ties, threshold", threshold)
    n = 130
    r = rng(60)
    P = np.zeros((n, 16, 4), np.float32)
    P[:, :, 0] = np.tile([0.0, 1.0, 1.0, 0.0], 4)
    P[:, :, 1] = np.repeat(np.linspace(0, 1, 4), 4)
    P[:, :, 3] = 1.0
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0], rays[:, 1] = r.uniform(0.05, 0.7, n), r.uniform(0.1, 0.9, n)
    rays[:, 2], rays[:, 3], rays[:, 6] = 2.0, np.inf, -1.0
    clip_equal(ctx, oracle, rays, P)
    subdivide_equal(ctx, oracle, rays, P, threshold)


@pytest.mark.parametrize("n", [1, 7, 64, 300])
def test_many_hits_of_one_pair(ctx, oracle, n):
    """Tangled nets that a ray crosses several times: lanes at work on one pair
    find candidates in the same turn, and the nearest one's (u, v) is kept."""
    say("bezier_clip, subdivision: tangled nets", n)
    r = rng(90 + n)
    P = np.ones((n, 16, 4), np.float32)
    P[:, :, :3] = r.uniform(0.0, 1.0, (n, 16, 3))
    o, to = r.uniform(-1.0, 2.0, (n, 3)), r.uniform(0.35, 0.65, (n, 3))
    o[:, 2] = 3.0
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3], rays[:, 3], rays[:, 4:7] = o, np.inf, (to - o) / np.linalg.norm(to - o, axis=1, keepdims=True)
    clip_equal(ctx, oracle, rays, P)
    subdivide_equal(ctx, oracle, rays, P, 2.0 ** -5)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 129])
def test_subpatch_remainders(ctx, oracle, n):
    say("subpatch", n)
    _, P = random_patch_pairs(n, 70)
    a = rng(71).uniform(0.0, 0.5, (n, 2)).astype(np.float32)
    R = np.stack([a[:, 0], a[:, 0] + 0.4, a[:, 1], a[:, 1] + 0.5], 1).astype(np.float32)
    g = ctx.subpatch(P, R)
    o = np.stack([oracle.subpatch(P[k], *R[k]) for k in range(n)])
    assert_bits_equal(g.reshape(n, -1), o.reshape(n, -1), "points")


@pytest.mark.parametrize("n", [100, 32767, 32768, 32769, 33001])
def test_subpatch_at_the_kernel_switch(ctx, oracle, n):
    """Per lane up to 32,768 patches, through LDS above."""
    say("subpatch", n)
    test_subpatch_remainders(ctx, oracle, n)
