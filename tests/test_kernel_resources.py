"""Registers of the kernels in the built library, from its code objects' own
metadata: the query kernels whose speed rests on three waves per SIMD (512
vector registers each SIMD) get them, without spilling their clip loop."""
from __future__ import annotations

import os
import re
import struct
import subprocess

import pytest

import conftest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: {vgpr, spill}} over the library's gfx950 code objects."""
    import cgspline_amd
    cgspline_amd.lib()
    with open(os.path.join(conftest.ROOT, "cgspline_amd", "libcgs.so"), "rb") as f:
        data = f.read()
    out, at = {}, data.find(MAGIC)
    while at >= 0:
        count, p = struct.unpack_from("<Q", data, at + len(MAGIC))[0], at + len(MAGIC) + 8
        for _ in range(count):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + idlen]:
                co = tmp_path_factory.mktemp("co") / "kernels.co"
                co.write_bytes(data[at + off:at + off + size])
                notes = subprocess.run([READELF, "--notes", str(co)], stdout=subprocess.PIPE, text=True, check=True).stdout
                for k in re.split(r"- \.agpr_count", notes)[1:]:
                    field = lambda n: re.search(r"\." + n + r":\s+(\S+)", k).group(1)   # noqa: E731
                    agpr = int(re.match(r":\s+(\d+)", k).group(1))
                    out[field("name")] = dict(vgpr=int(field("vgpr_count")) + agpr, spill=int(field("vgpr_spill_count")))
            p += 24 + idlen
        at = data.find(MAGIC, at + 1)
    return out


# Registers that a kernel holds around its clips go to scratch memory once per
# clip; more than about a hundred are spilled in the loop over a clip's passes.
@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
@pytest.mark.parametrize("name, spills", [("5kPickILb0E", 8), ("5kPickILb1E", 8), ("9kTraceAnyILi0E", 40),
                                          ("11kTraceBatchILi0ELb0ELb0ELi3E", 80),
                                          ("11kTraceBatchILi0ELb0ELb1ELi3E", 100)])
def test_three_waves_per_simd(kernels, name, spills):
    k = [v for n, v in kernels.items() if n.startswith("_ZN3cgs" + name)]
    assert len(k) == 1
    assert k[0]["vgpr"] <= 512 // 3 // 8 * 8 and k[0]["spill"] <= spills, k


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
@pytest.mark.parametrize("name", ["11kTraceBatchILi0ELb0ELb0ELi2E", "11kTraceBatchILi0ELb0ELb1ELi2E", "13kTraceClosestILi0ELb0E",
                                  "7kRenderILb0ELb0ELb0E", "7kRenderILb1ELb0ELb0E"])
def test_two_waves_per_simd_without_spills(kernels, name):
    k = [v for n, v in kernels.items() if n.startswith("_ZN3cgs" + name)]
    assert len(k) == 1
    assert k[0]["vgpr"] <= 256 and k[0]["spill"] == 0, k
