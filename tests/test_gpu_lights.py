"""Renders of scenes with one, two and many lights against the oracle, bit for
bit: from two lights on a wave's shadow rays go through one list, eight lights
of a full wave at a time."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from conftest import rng, say

pytestmark = pytest.mark.gpu


def with_lights(wl, n, box):
    """The workload with n lights around it: points, every third one with a
    range, every fifth one a spot, every seventh one directional."""
    r = rng(80)
    L = np.zeros((n, 12), np.float32)
    L[:, 0:3] = r.uniform(2.0, 40.0, (n, 3))
    L[:, 3] = 1.0
    L[:, 4:7] = r.uniform(-box, 2 * box, (n, 3))
    d = box / 2 - L[:, 4:7]
    L[:, 8:11] = d / np.linalg.norm(d, axis=1, keepdims=True)
    L[:, 11] = 3.1415
    k = np.arange(n)
    L[k % 3 == 1, 7] = 1.5 * box
    L[k % 5 == 2, 11] = 0.8
    L[k % 7 == 3, 11] = 0.0
    return dataclasses.replace(wl, scene=dataclasses.replace(wl.scene, lights=L))


@pytest.mark.parametrize("lights", [0, 1, 2, 3, 8, 9, 70])
@pytest.mark.parametrize("name", ["closed", "displaced"])
def test_light_counts(ctx, oracle, name, lights):
    from cgspline_amd import scenes
    if name == "closed":
        wl, box = scenes.closed_surfaces(count=12, width=45, height=37), 10.0
        wl.depth = 2
    else:
        wl, box = scenes.displaced_grids(grids=40, width=45, height=37, box=4.0), 4.0
    wl = with_lights(wl, lights, box)
    say("render: scene, lights", name, lights)
    ds = ctx.scene(wl.scene, hash_retries=3)
    color, frame, n = ds.render(wl.camera, eps=wl.eps, depth=wl.depth)
    ocolor, oframe, _, rc = oracle.OracleScene(ds.scene).render(wl.camera, eps=wl.eps, depth=wl.depth)
    assert n["overflow"] == 0
    assert (n["primary"], n["shadow"], n["secondary"]) == (rc["primary"], rc["shadow"], rc["secondary"])
    assert lights == 0 or n["shadow"] > 0
    assert np.array_equal(color.view(np.uint32), ocolor.view(np.uint32))
    ds.destroy()


@pytest.mark.parametrize("lights", [1, 3, 12])
def test_surface_with_a_cull_tree(ctx, oracle, grazing, lights):
    """Several lights on a surface of 16,384 patches: the shadow-ray list with
    the paths for large surfaces."""
    wl = with_lights(dataclasses.replace(grazing, camera=dataclasses.replace(grazing.camera, width=53, height=41)), lights, 1.0)
    say("render: surface with a cull tree, lights", lights)
    ds = ctx.scene(wl.scene)
    assert ds.bvh_culled(0)
    color, _, n = ds.render(wl.camera, eps=wl.eps, depth=1)
    ocolor, _, _, rc = oracle.OracleScene(wl.scene).render(wl.camera, eps=wl.eps, depth=1)
    assert n["overflow"] == 0
    assert (n["primary"], n["shadow"], n["secondary"]) == (rc["primary"], rc["shadow"], rc["secondary"])
    assert lights == 1 or n["shadow"] > 0
    assert np.array_equal(color.view(np.uint32), ocolor.view(np.uint32))
    ds.destroy()


@pytest.mark.parametrize("lights", [1, 2, 9])
def test_overflow_of_listed_shadow_rays(ctx, lights):
    """A vertical planar patch above the camera and directional lights in its
    plane: the shadow rays of the frame's middle column lie in that plane and
    overflow the patch's clip.  Shaded queries, which take no list, give the same
    colours and the same count."""
    from cgspline_amd import scenes
    from test_gpu_errors import planar_patch
    floor = planar_patch(16.0)
    floor[:, :2] -= 8.0
    wall = np.ones((16, 4), np.float32)
    wall[:, 0], wall[:, 1], wall[:, 2] = 0.0, 2.5 * floor[:, 0] - 10.0, 12.0 + planar_patch(16.0)[:, 1]
    idx = np.arange(16, dtype=np.uint32)[None]
    material = np.array([0.5] * 6 + [0.0, 0.5], np.float32)
    L = np.zeros((lights, 12), np.float32)
    L[:, 0:4], L[:, 9], L[:, 10] = 1.0, 0.6, -0.8
    floor[:, 2] = np.float32(0.05) * np.linspace(0, 1, 16, dtype=np.float32)   # (a box of some thickness)
    sc = scenes.assemble([(floor, idx), (wall, idx)], [(k, scenes.IDENTITY16, scenes.IDENTITY16, material) for k in (0, 1)],
                         list(L), name="floor and wall")
    cam = scenes.make_camera((0.0, 0.0, 6.0), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 60.0, 65, 33)
    ds = ctx.scene(sc)
    say("render: shadow rays in a patch's plane, lights", lights)
    color, _, n = ds.render(cam, eps=1e-3, depth=0)
    say("shade: the same")
    scolor, _, _, _, _, sn = ds.shade(scenes.camera_rays(cam), eps=1e-3, depth=0)
    assert n["shadow"] == sn["shadow"] > 0 and n["overflow"] == sn["overflow"]
    assert np.array_equal(color.reshape(-1, 3).view(np.uint32), scolor.view(np.uint32))
    assert 0 < n["overflow"] <= 33
    ds.destroy()
