"""Registers of the built histogram kernels, from the code objects' own metadata (no GPU)."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from padenti_amd import _lib as L

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(path):
    """The gfx950 code objects of a library (one bundle per translation unit)."""
    data = open(path, "rb").read()
    for m in re.finditer(MAGIC, data):
        at = m.start() + len(MAGIC)
        n, = struct.unpack_from("<Q", data, at)
        at += 8
        if n > 16:
            continue   # the text in some other place
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, at)
            triple = data[at + 24:at + 24 + length]
            at += 24 + length
            if size and b"gfx950" in triple:
                yield data[m.start() + off:m.start() + off + size]


@pytest.mark.skipif(shutil.which(READELF) is None, reason="needs llvm-readelf")
def test_histogram_kernels_fit_eight_waves(tmp_path):
    """At most 80 scalar and 64 vector registers and none of the latter spilled:
    eight waves of the histogram kernel fit a SIMD in every instantiation."""
    seen = 0
    for i, co in enumerate(_code_objects(L.LIB_PATH)):
        f = tmp_path / ("%d.co" % i)
        f.write_bytes(co)
        notes = subprocess.run([READELF, "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for k in re.split(r"\n  - \.", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", k)
            if not name or "k_histI" not in name.group(1):
                continue
            reg = {r: int(re.search(r"\.%s:\s+(\d+)" % r, k).group(1))
                   for r in ("sgpr_count", "vgpr_count", "vgpr_spill_count", "sgpr_spill_count")}
            assert reg["sgpr_count"] <= 80 and reg["vgpr_count"] <= 64 and reg["vgpr_spill_count"] == 0, (name.group(1), reg)
            seen += 1
    assert seen >= 4
