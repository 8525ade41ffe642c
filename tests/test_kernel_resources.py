"""What the compiler gave each kernel of the built library, read from the metadata of its
gfx950 code objects: no register spills and no scratch memory.  The attribute queries of the
C-ABI describe one kernel per tile; this sees every instantiation that a launch may pick."""
from __future__ import annotations

import os
import re
import shutil
import struct
import subprocess

import pytest

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
READELF = next((p for p in (shutil.which("llvm-readelf"), "/opt/rocm/llvm/bin/llvm-readelf")
                if p and os.path.exists(p)), None)
# The bounds-checked register-staged kernel at 256 x 256: shapes narrower than a tile, or
# with K too short for the direct-to-LDS kernels.
MAY_SPILL = re.compile(r"^_ZN8mcke_amd\d+(gemm_mfma_kernelILi256ELi256E|gemm_lp_kernelI\w+Li256ELi256E)")


def _code_objects(path):
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + length].decode()
            pos += 24 + length
            if triple.endswith("gfx950") and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


@pytest.fixture(scope="module")
def kernels(mcke, tmp_path_factory):
    if READELF is None:
        pytest.skip("llvm-readelf is not installed")
    mcke.lib()
    found, where = {}, tmp_path_factory.mktemp("co")
    for i, obj in enumerate(_code_objects(mcke.library_path())):
        f = where / f"{i}.co"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], check=True, capture_output=True,
                               text=True).stdout
        for entry in re.split(r"\n  - ", notes):
            name = re.search(r"^\s+\.name:\s+(\S+)$", entry, re.M)
            if name:
                found[name.group(1)] = {k: int(v) for k, v in re.findall(
                    r"^\s*\.(\w+(?:_count|_size)):\s+(\d+)$", entry, re.M)}
    return found


def test_every_kernel_family_is_there(kernels):
    for family in ("gemm_rows_kernel", "gemm_mfma_dma_kernel", "gemm_lp_split_kernel",
                   "gemm_lp_dma16_kernel", "gemm_lp_dma_kernel", "row_reduce_short_kernel",
                   "softmax_regs_kernel", "bias_act_flat_kernel"):
        assert any(family in k for k in kernels), family


def test_no_spills(kernels):
    bad = {k: v for k, v in kernels.items() if not MAY_SPILL.match(k) and
           (v.get("vgpr_spill_count", 0) or v.get("sgpr_spill_count", 0) or
            v.get("private_segment_fixed_size", 0))}
    assert not bad, bad
