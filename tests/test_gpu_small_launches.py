"""Launches of few rays or pixels, whose waves take fewer than 64 work items
each (powers of two down to 8), against the oracle, bit for bit, at sizes
around those steps."""
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
