"""Rays with a zero direction component in scenes with a cull tree: they take
the reference's top-level traversal, beside lanes that take the tree's, and a
wave's lanes wait for each other between its objects.  Results equal the
oracle's bit for bit, alone and mixed, and the rays of an orthographic view are
not much slower than ones turned a little off the plane."""
from __future__ import annotations

import time

import numpy as np
import pytest

from conftest import rng, say
from test_gpu_cull import cull_off
from test_gpu_lights import with_lights
from test_gpu_parity import assert_bits_equal

pytestmark = pytest.mark.gpu


def parallel_rays(box, n, direction, shift=0.0):
    """n x n rays of one direction over a square above the scene."""
    g = (np.arange(n) + 0.5) / n * box
    rays = np.zeros((n * n, 8), np.float32)
    rays[:, 0], rays[:, 1], rays[:, 2] = np.repeat(g, n), np.tile(g, n) + shift, 2 * box
    rays[:, 3], rays[:, 4:7] = np.inf, direction
    return rays


def mixed_rays(scene_rays, seed):
    """Every other ray with one or two components of its direction zero."""
    rays = np.array(scene_rays)
    r = rng(seed)
    for k in range(0, rays.shape[0], 2):
        axes = r.permutation(3)[:r.integers(1, 3)]
        d = rays[k, 4:7].copy()
        d[axes] = 0.0
        if np.any(d):
            rays[k, 4:7] = d / np.linalg.norm(d)
    return rays


def compare(ctx, oracle, wl, rays, what):
    ds = ctx.scene(wl.scene)
    assert ds.culled
    osc = oracle.OracleScene(wl.scene)
    say("rays with zero components:", what, rays.shape[0])
    tuv, patch, obj = ds.trace_closest(rays)
    oh, op, oo, _ = osc.trace(rays)
    assert np.array_equal(obj, oo) and np.array_equal(patch, op)
    assert_bits_equal(tuv, oh, what)
    assert np.array_equal(ds.trace_any(rays) == 1, osc.trace(rays, any_hit=True)[0])
    color = ds.shade(rays, depth=1)[0]
    assert_bits_equal(color, np.asarray(osc.shade(rays, depth=1)[0], np.float32).reshape(color.shape), what)
    ds.destroy()
    return obj


@pytest.mark.parametrize("name, direction, shift", [("z", (0, 0, -1), 0.0), ("yz", (0, -0.6, -0.8), 1.5),
                                                    ("-x z", (-0.0, 0.6, -0.8), -1.5)])
def test_parallel_rays(ctx, oracle, c3_small, name, direction, shift):
    rays = parallel_rays(6.0, 90, direction, 6.0 * shift)
    obj = compare(ctx, oracle, c3_small, rays, name)
    assert (obj >= 0).sum() > 200


def test_mixed_with_other_rays(ctx, oracle, c2_small, c3_small):
    from cgspline_amd import scenes
    for k, wl in enumerate((c2_small, c3_small)):
        obj = compare(ctx, oracle, wl, mixed_rays(scenes.camera_rays(wl.camera)[::7], 30 + k), wl.scene.name)
        assert (obj >= 0).sum() > 200


@pytest.mark.parametrize("lights", [1, 9])
def test_frames_without_a_cull_tree(ctx, oracle, lights):
    """Every ray, shadow rays from a list too, on the reference's traversal."""
    from cgspline_amd import scenes
    wl = with_lights(scenes.displaced_grids(grids=40, width=61, height=47, box=4.0), lights, 4.0)
    say("frame without a cull tree: lights", lights)
    with cull_off():
        ds = ctx.scene(wl.scene)
    assert not ds.culled
    color, _, n = ds.render(wl.camera, eps=wl.eps, depth=2)
    ocolor, _, _, rc = oracle.OracleScene(wl.scene).render(wl.camera, eps=wl.eps, depth=2)
    assert (n["primary"], n["shadow"], n["secondary"]) == (rc["primary"], rc["shadow"], rc["secondary"])
    assert np.array_equal(color.view(np.uint32), ocolor.view(np.uint32))
    ds.destroy()


def test_parallel_rays_keep_pace(ctx):
    """A million parallel any-hit rays through 2,048 grids, in an axis plane
    against turned off it by 1e-5 (the cull tree's traversal): 1.7 times as
    long; 3.1 times when a wave's lanes did not wait for each other."""
    import cgspline_amd as cgs
    from cgspline_amd import scenes
    box = 25.0 * 0.5 ** (1.0 / 3.0)
    wl = scenes.displaced_grids(grids=2048, width=64, height=64, box=box)
    ds = ctx.scene(wl.scene, hash_retries=3)
    out = cgs.DeviceArray(ctx, 4 * 1_000_000)
    best = []
    for dx in (0.0, 1e-5):
        rays = cgs.DeviceArray.from_host(ctx, parallel_rays(box, 1000, (dx, -0.6, -0.8), 1.5 * box))
        times = []
        for _ in range(6):
            ctx.sync()
            t = time.perf_counter()
            ds.trace_any_dev(rays, 1_000_000, out)
            ctx.sync()
            times.append(1e3 * (time.perf_counter() - t))
        best.append(min(times))
    say("parallel rays: ms in the plane, off it", best)
    ds.destroy()
    assert best[0] < 2.4 * best[1]
