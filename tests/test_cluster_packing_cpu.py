"""Packing of clusters into workgroups (pack_clusters).

Every particle has one slot and a cluster lies within a block, on a multiple of the
sharing lanes, with its helpers after it; blocks hold the largest clusters first, every
second run of them reversed while there are at most as many runs as asked for (three for
the implicit kernel, five for Heun on two lanes, none on one), and in order beyond.
"""
import ctypes as C

import numpy as np
import pytest

from test_cluster_layout_cpu import compile_driver, ptr

DRIVER = r'''
#include "cluster_layout.hpp"
extern "C" int64_t pack(const int64_t *offsets, int64_t n, int block, int align, int64_t run,
                        int64_t most_runs, int64_t *slot, int *base, int *size)
{
    std::vector<std::pair<int64_t, int64_t>> m;
    for (int64_t i = 0; i < n; ++i) m.emplace_back(offsets[i], offsets[i + 1]);
    std::vector<int64_t> s;
    std::vector<int> b, c;
    mp_host::pack_clusters(m, block, align, (size_t)run, (size_t)most_runs, s, b, c);
    std::copy(s.begin(), s.end(), slot);
    std::copy(b.begin(), b.end(), base);
    std::copy(c.begin(), c.end(), size);
    return (int64_t)s.size();
}
extern "C" int reversed(int implicit, int lanes) { return (int)mp_host::reversed_runs(implicit != 0, lanes); }
'''


@pytest.fixture(scope="module")
def pack(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("packing")
    compile_driver(tmp, DRIVER, "-fPIC", "-shared", "-o", str(tmp / "d.so"))
    lib = C.CDLL(str(tmp / "d.so"))
    f = lib.pack
    f.restype = C.c_int64
    assert [lib.reversed(1, 1), lib.reversed(0, 2), lib.reversed(0, 1)] == [3, 5, 0]

    def of(sizes, block, align, run, most_runs=5):
        off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
        room = len(sizes) * block
        slot, base, size = np.empty(room, np.int64), np.empty(room, np.int32), np.empty(room, np.int32)
        n = f(ptr(off), C.c_int64(len(sizes)), block, align, C.c_int64(run), C.c_int64(most_runs),
              ptr(slot), ptr(base), ptr(size))
        shape = (n // block, block)
        return off, slot[:n].reshape(shape), base[:n].reshape(shape), size[:n].reshape(shape)
    return of


@pytest.mark.parametrize("block,align,largest,members,run", [
    (64, 1, 64, 900, 100), (64, 2, 8, 500, 8), (64, 4, 64, 700, 90), (256, 4, 256, 90, 40),
    (128, 1, 64, 60, 4), (64, 1, 64, 12, 1)])
def test_packing(pack, block, align, largest, members, run):
    rng = np.random.default_rng(block + align)
    sizes = rng.integers(1, largest + 1, size=members)
    off, slot, base, size = pack(sizes, block, align, run)
    assert sorted(slot[slot >= 0]) == list(range(off[-1]))
    member = np.repeat(np.arange(members), sizes)
    for b in range(slot.shape[0]):
        for i in np.flatnonzero(slot[b] >= 0):
            m = member[slot[b, i]]
            assert base[b, i] % align == 0 and size[b, i] == sizes[m]
            assert slot[b, i] == off[m] + i - base[b, i]
            taken = -(-sizes[m] // align) * align
            assert base[b, i] + taken <= block
            assert np.all(size[b, base[b, i]:base[b, i] + taken] == sizes[m])


@pytest.mark.parametrize("blocks,run,most,in_order", [
    (3, 4, 5, True), (8, 4, 5, False), (17, 4, 5, False), (20, 4, 5, False), (21, 4, 5, True),
    (36, 4, 5, True), (5, 2, 5, False), (11, 2, 5, True), (12, 4, 3, False), (13, 4, 3, True),
    (8, 4, 0, True)])
def test_order_of_blocks(pack, blocks, run, most, in_order):
    sizes = 65 + np.random.default_rng(blocks).permutation(blocks)   # one to a block of 128
    order = [int(s.max()) for s in pack(sizes, 128, 1, run, most)[3]]
    want = sorted(order, reverse=True)
    if not in_order:
        want = sum((want[i:i + run][::-1] if i // run % 2 else want[i:i + run]
                    for i in range(0, blocks, run)), [])
    assert order == want
