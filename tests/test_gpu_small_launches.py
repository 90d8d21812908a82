"""Launches of few rays or pixels, whose waves take fewer than 64 work items
each (powers of two down to 8), against the oracle, bit for bit: at 8 items a
wave, where a launch has fewer waves than items in one, and around the sizes at
which a wave's items double."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu

SIZES = [1, 7, 8, 9, 63, 64, 65, 1025]


@pytest.mark.parametrize("n", SIZES)
def test_few_rays(ctx, oracle, c3_small, n):
    from cgspline_amd import scenes
    ds = ctx.scene(c3_small.scene)
    osc = oracle.OracleScene(c3_small.scene)
    rays = scenes.camera_rays(c3_small.camera)
    rays = np.ascontiguousarray(rays[:: max(1, rays.shape[0] // n)][:n])
    say("closest, any, shade: rays", n)
    tuv, patch, obj = ds.trace_closest(rays)
    oh, op, oo, _ = osc.trace(rays)
    assert np.array_equal(obj, oo) and np.array_equal(patch, op)
    assert np.array_equal(tuv.view(np.uint32), oh.view(np.uint32))
    assert np.array_equal(ds.trace_any(rays) == 1, osc.trace(rays, any_hit=True)[0])
    color, _, _, _, sobj, _ = ds.shade(rays, depth=1)
    ocolor = osc.shade(rays, depth=1)[0]
    assert np.array_equal(sobj, oo)
    assert np.array_equal(color.view(np.uint32), np.asarray(ocolor, np.float32).view(np.uint32))


@pytest.mark.parametrize("size", [(1, 1), (9, 7), (64, 8), (130, 33), (300, 200)])
@pytest.mark.parametrize("samples", [None, 3])
def test_small_frames(ctx, oracle, size, samples):
    from cgspline_amd import scenes
    wl = scenes.heightfield_c1(width=size[0], height=size[1])
    say("render: size, samples", size, samples)
    ds = ctx.scene(wl.scene)
    osc = oracle.OracleScene(wl.scene)
    if samples is None:
        want = osc.render(wl.camera, eps=wl.eps, depth=1)
    else:
        want = osc.render_sampled(wl.camera, samples=samples, seed=42, eps=wl.eps, depth=1)
    for again in range(3):     # the first render takes the tiles in row order, later ones longest first
        color, _, n = ds.render(wl.camera, eps=wl.eps, depth=1, samples=samples)
        assert n["overflow"] == 0 and n["primary"] == size[0] * size[1] * (samples or 1)
        assert np.array_equal(color.view(np.uint32), np.asarray(want[0], np.float32).reshape(color.shape).view(np.uint32))


# Around the sizes at which a wave's items double, for kernels of two and of three
# waves per SIMD on 256 CUs (8 items a wave up to 8 x 4 x 512 or 768, and so on).
STEPS = [s + d for s in (16_384, 24_576, 32_768, 49_152, 65_536, 98_304) for d in (0, 1)] + [70_001, 131_137]


@pytest.fixture(scope="module")
def step_rays(c3_small, oracle):
    """3,001 camera rays and what the oracle gives for them; a launch repeats them."""
    from cgspline_amd import scenes
    rays = np.ascontiguousarray(scenes.camera_rays(c3_small.camera)[::21][:3001])
    osc = oracle.OracleScene(c3_small.scene)
    return rays, osc.trace(rays)[:3], osc.trace(rays, any_hit=True)[0], osc.shade(rays, depth=1)[0]


@pytest.mark.parametrize("n", STEPS)
def test_steps_of_a_launch(ctx, c3_small, step_rays, n):
    rays, (oh, op, oo), occ, ocolor = step_rays
    at = np.arange(n) % rays.shape[0]
    many = np.ascontiguousarray(rays[at])
    ds = ctx.scene(c3_small.scene)
    say("closest, any, shade: rays", n)
    tuv, patch, obj = ds.trace_closest(many)
    assert np.array_equal(obj, oo[at]) and np.array_equal(patch, op[at])
    assert np.array_equal(tuv.view(np.uint32), oh[at].view(np.uint32))
    assert np.array_equal(ds.trace_any(many) == 1, occ[at])
    color = ds.shade(many, depth=1)[0]
    assert np.array_equal(color.view(np.uint32), np.asarray(ocolor, np.float32).reshape(-1, 3)[at].view(np.uint32))
    ds.destroy()


@pytest.mark.parametrize("n", STEPS)
def test_steps_of_a_pick(ctx, oracle, n):
    from cgspline_amd import scenes
    r = np.random.default_rng(9)
    v, i = scenes.heightfield_grid(r, n=16)
    o = r.uniform([0, 0, 0.8], [1, 1, 1.5], (3001, 3))
    d = r.uniform([-0.3, -0.3, -0.2], [1.3, 1.3, 0.2], (3001, 3)) - o
    rays = np.zeros((3001, 8), np.float32)
    rays[:, 0:3], rays[:, 3], rays[:, 4:7] = o, np.inf, d / np.linalg.norm(d, axis=1, keepdims=True)
    at = np.arange(n) % 3001
    pick = ctx.patch_bvh(v, i)
    say("pick: rays", n)
    few, many = pick.intersect(rays), pick.intersect(np.ascontiguousarray(rays[at]))
    for a, b in zip(few, many):
        assert np.array_equal(np.asarray(a)[at].view(np.uint32), np.asarray(b).view(np.uint32))
    assert np.array_equal(pick.intersect_any(rays)[at], pick.intersect_any(np.ascontiguousarray(rays[at])))
    pick.destroy()
