"""How many lanes share the pair sums of an implicit launch (field_targets).

Two without a cluster above 8 particles; four where every slot has room on one wave
per SIMD (65,536 slots of 256 CUs); else four only while the slots that small members'
helper lanes add are at most a sixth of the large clusters' particles: a cluster of 9
among many dimers must not take them to four lanes, nor a few dimers many clusters of
64 to two.
"""
import ctypes as C

import numpy as np
import pytest

from test_cluster_layout_cpu import compile_driver, ptr

DRIVER = r'''
#include "cluster_layout.hpp"
extern "C" int targets(const int64_t *offsets, int64_t n, int64_t one_wave)
{
    std::vector<std::pair<int64_t, int64_t>> m;
    for (int64_t i = 0; i < n; ++i) m.emplace_back(offsets[i], offsets[i + 1]);
    return mp_host::field_targets(m, one_wave);
}
'''


@pytest.fixture(scope="module")
def targets(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("targets")
    compile_driver(tmp, DRIVER, "-fPIC", "-shared", "-o", str(tmp / "d.so"))
    f = C.CDLL(str(tmp / "d.so")).targets

    def of(*sizes):
        sizes = np.concatenate([np.full(k, n) for n, k in sizes])
        offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
        return f(ptr(offsets), C.c_int64(sizes.size), C.c_int64(65536))
    return of


@pytest.mark.parametrize("sizes,lanes", [
    ([(2, 65536)], 2), ([(8, 20000)], 2), ([(1, 1)], 2),
    ([(9, 1)], 4), ([(9, 20000)], 4), ([(2, 64), (9, 1)], 4), ([(2, 512), (32, 64)], 4),
    ([(2, 65536), (9, 1)], 2), ([(2, 20000), (64, 2000)], 2), ([(2, 8000), (64, 2000)], 4),
    # four lanes: dimers take four slots, three or four particles no more than they had
    ([(2, 16381), (12, 1)], 4), ([(2, 16382), (12, 1)], 2), ([(3, 30000), (9, 1)], 4),
    ([(2, 5333), (64, 1000)], 4), ([(2, 5334), (64, 1000)], 2)])
def test_lanes_by_the_work_of_the_members(targets, sizes, lanes):
    assert targets(*sizes) == lanes
