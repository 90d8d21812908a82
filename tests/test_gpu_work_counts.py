"""The counting build counts every render's events on the kernel that the render
uses: one light, several (the shadow-ray list's kernels), sampled."""
from __future__ import annotations

import json
import os
import subprocess
import sys

import pytest

import conftest
from conftest import say

pytestmark = pytest.mark.gpu

CHILD = r"""
import ctypes as C, json, sys
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
import cgspline_amd as cgs
from cgspline_amd import scenes, workmodel
from test_gpu_lights import with_lights
ctx, out = cgs.Context(0), []
n = len(workmodel.GPU_EVENTS)
c = (C.c_uint64 * n)()
for lights, samples in ((1, None), (5, None), (1, 2)):
    wl = with_lights(scenes.displaced_grids(grids=40, width=64, height=64, box=4.0), lights, 4.0)
    ds = ctx.scene(wl.scene, hash_retries=3)
    cgs.check(cgs.lib().cgs_work_counts(ctx.h, c, n, 1))
    _, _, rays = ds.render(wl.camera, eps=wl.eps, depth=1, samples=samples)
    cgs.check(cgs.lib().cgs_work_counts(ctx.h, c, n, 1))
    out.append([dict(zip(workmodel.GPU_EVENTS, [int(x) for x in c])), rays])
print("COUNTS " + json.dumps(out))
"""


def test_every_render_is_counted():
    from cgspline_amd import _build
    if not os.path.exists(_build.COUNTING_LIB):
        pytest.skip("no counting build")
    say("work counts of three renders in the counting build")
    env = dict(os.environ, CGS_LIBRARY=_build.COUNTING_LIB)
    r = subprocess.run([sys.executable, "-c", CHILD, conftest.ROOT], env=env, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:]
    for events, rays in json.loads([x for x in r.stdout.splitlines() if x.startswith("COUNTS ")][0][7:]):
        say(rays, events)
        # every ray that starts inside the cull tree reads its root at least, and each hit was a patch test
        assert events["cullNodes"] >= rays["primary"] and events["patchTests"] > 0 and events["onHits"] > 0, events


def test_no_render_is_counted_on_another_kernel():
    """launchRender chooses the same kernels in a counting build."""
    with open(os.path.join(conftest.ROOT, "cgspline_amd", "csrc", "cgs_trace.hip")) as f:
        src = f.read()
    body = src[src.index("hipError_t launchRender(const SceneDev&"):]
    assert "CGS_WORK_COUNTS" not in body[:body.index("\n}\n")]
