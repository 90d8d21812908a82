"""The batched clipper against the oracle, bit for bit: tolerances whose square
decides convergence."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import say
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
