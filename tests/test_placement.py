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
uint32_t chunk_begin(uint32_t begin, uint32_t n, uint32_t chunks, uint32_t k)
{
  return pd::engine::chunk_begin(begin, n, chunks, k);
}
size_t deal(size_t n, const uint32_t *samples, uint32_t n_xcc, uint32_t *order, uint32_t *xcd)
{
  const pd::engine::GroupOrder r = pd::engine::deal_groups(std::vector<uint32_t>(samples, samples + n), n_xcc);
  std::copy(r.order.begin(), r.order.end(), order);
  std::copy(r.xcd.begin(), r.xcd.end(), xcd);
  return r.rows;
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
    so = C.CDLL(str(lib))
    so.chunk_begin.restype, so.chunk_begin.argtypes = C.c_uint32, [C.c_uint32] * 4
    so.deal.restype, so.deal.argtypes = C.c_size_t, [C.c_size_t, C.c_void_p, C.c_uint32, C.c_void_p, C.c_void_p]
    return so


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


def _deal(host, samples, X):
    n = len(samples)
    a, order, xcd = (C.c_uint32 * n)(*samples), (C.c_uint32 * n)(), (C.c_uint32 * n)()
    rows = host.deal(n, a, X, order, xcd)
    return list(order), list(xcd), rows


@pytest.mark.parametrize("X", [2, 4, 8])
@pytest.mark.parametrize("samples", [
    [1000], [5, 0, 7], [0] * 50, [11] * 64, [11] * 65,
    [50000] * 16 + [20] * 6000,                       # a few large groups among many tiny ones
    [400000] + [1] * 3000,
    [32768] * 3 + [0] * 4000,
    [30000] * 7 + [20] * 350,                         # the tiny ones would all go to the eighth XCD
    [(i * 2654435761 >> 7) % 5500 + 500 for i in range(968)],
])
def test_groups_are_dealt_once_and_evenly(host, samples, X):
    """Every group is launched once; the padding of the interleaved lists stays
    within a quarter of the groups (one row more), and where that does not bind
    the XCDs' shares differ by at most one group."""
    order, xcd, rows = _deal(host, samples, X)
    assert sorted(order) == list(range(len(samples)))
    per = [xcd.count(x) for x in range(X)]
    assert sum(per) == len(samples) and max(per) == rows
    share = -(-len(samples) // X)
    assert rows <= share + share // 4 + 1
    load = [sum(samples[g] + 64 for g in range(len(samples)) if xcd[g] == x) for x in range(X)]
    if rows < share + share // 4 + 1:
        assert max(load) - min(load) <= max(samples) + 64
    if len(set(samples)) > 1:   # the smallest ones come last
        assert samples[order[-1]] == min(samples)


@pytest.mark.parametrize("begin", [0, 1, 2, 3, 4, 1001, 4_294_000_000])
@pytest.mark.parametrize("n,chunk", [(0, 64), (1, 64), (64, 64), (65, 64), (128, 64), (200, 64), (1000, 333),
                                     (65536, 32768), (65537, 32768), (294_967, 32768)])
def test_chunks_of_a_node_begin_on_record_lines(host, begin, n, chunk):
    """The chunks of a node cover its records once and in order, differ by a few
    records, and every one but the first begins on a 64-byte line of them."""
    chunks = max(1, -(-n // chunk))
    cut = [host.chunk_begin(begin, n, chunks, k) & 0xffffffff for k in range(chunks + 1)]
    assert cut[0] == begin and cut[-1] == begin + n
    assert all(c % 4 == 0 for c in cut[1:-1])
    sizes = [b - a for a, b in zip(cut, cut[1:])]
    assert all(0 <= s <= min(chunk, -(-n // chunks)) + 3 and (n == 0 or s > 0) for s in sizes)
    assert max(sizes) - min(sizes) <= 7
