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
