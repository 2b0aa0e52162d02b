"""How a level is cut into histogram work items (include/padenti/pd_placement.hpp),
compiled for the host by g++ (no GPU)."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs a C++ compiler")

SRC = r"""
#include "padenti/pd_placement.hpp"
extern "C" {
uint32_t item_chunk(uint64_t level_samples, uint32_t nF, uint32_t ftiles, uint32_t nT, uint32_t nC, uint32_t cus,
                    uint32_t blocks_per_cu, uint32_t launches)
{
  return pd::engine::item_chunk(level_samples, nF, ftiles, nT, nC, cus, blocks_per_cu, launches);
}
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("placement")
    src, lib = d / "placement.cpp", d / "libplacement.so"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-I", os.path.join(ROOT, "include"), str(src), "-o",
                    str(lib)], check=True)
    return C.CDLL(str(lib))


def _chunk(host, samples, nF, nT, nC, cus=256, blocks=16, launches=1):
    return host.item_chunk(C.c_uint64(samples), nF, (nF + 63) // 64, nT, nC, cus, blocks, launches)


def test_chunks_of_small_levels_weigh_the_flush(host):
    """Items shorter than 1024 samples where a level would leave CUs idle, but
    not where their histogram flushes cost more than the CUs gain."""
    assert _chunk(host, 8192, 100, 10, 4) < 128             # 40 counts a candidate: many short items
    assert _chunk(host, 64, 100, 10, 4) == 64
    assert _chunk(host, 4000, 4000, 32, 16) == 1024         # 512 counts a candidate: 65 Mi atomics a level in short ones
    assert _chunk(host, 16000, 1000, 32, 21) == 1024
    for samples, nF, nT, nC in [(2000, 2000, 20, 8), (4000, 500, 20, 8), (1000, 64, 5, 2)]:
        c = _chunk(host, samples, nF, nT, nC)
        assert 64 <= c <= 1024 and c >= int((samples * nF * nT * nC) ** 0.5 / 64)
    # node by node: as for one node of the mean size (or two items a CU)
    assert _chunk(host, 8000, 500, 10, 8) == int((8000 * 500 * 80) ** 0.5 / 64)
    assert _chunk(host, 8000, 500, 10, 8, launches=64) == 8000 * 8 // 512
    assert _chunk(host, 10_000_000, 4000, 32, 16) == 32768   # large levels: blocks_per_cu items a CU
    assert _chunk(host, 1_000_000, 2000, 20, 8) == -(-1_000_000 * 32 // (256 * 16))
