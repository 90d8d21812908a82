"""Words of a wave's LDS that lanes change by atomics in the same turn are read
back by atomics too (the kernels' source, checked as text): a plain load after a
lane's own ldsMin could be given that lane's result instead of the word."""
from __future__ import annotations

import os
import re

import pytest

import conftest


@pytest.mark.parametrize("name, words", [("cgs_clip_wave.hpp", "kClipKey"), ("cgs_trace.hip", "kSubKey")])
def test_key_is_read_back_by_an_atomic(name, words):
    with open(os.path.join(conftest.ROOT, "cgspline_amd", "csrc", name)) as f:
        src = f.read()
    mins = [m.end() for m in re.finditer(r"ldsMin\(w \+ " + words, src)]
    assert len(mins) == 1
    after = src[mins[0]:mins[0] + 400]
    first = re.search(r"(ldsLoad\(w \+ |w\[)" + words, after)
    assert first and first.group(1).startswith("ldsLoad"), after
