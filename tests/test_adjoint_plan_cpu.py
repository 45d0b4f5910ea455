"""Batches of the adjoint maps (magpy_amd/csrc/adjoint_plan.hpp).

A batch takes up to 2^20 lanes and 8 GiB for the states and the pieces' maps together,
except that 2^18 lanes, or a single segment, are always one.  Over random schedules, few
samples to one at every step: these bounds hold, no coarser even split would also have
held them, and the pieces given are the most that any batch has.
"""
import ctypes as C

import numpy as np
import pytest

from test_cluster_layout_cpu import compile_driver, ptr

GIB = 1 << 30
DRIVER = r'''
#include "adjoint_plan.hpp"
extern "C" void batch(const int32_t *first, int64_t n_seg, int64_t n_pieces, int64_t block, int64_t P,
                      int64_t lanes, int64_t seg_bytes, int64_t piece_bytes, int64_t *out)
{
    const mp_host::MapBatch b = mp_host::map_batch(std::vector<int32_t>(first, first + n_seg),
                                                   n_pieces, block, P, lanes, seg_bytes, piece_bytes);
    out[0] = b.segments;
    out[1] = b.pieces;
}
'''


@pytest.fixture(scope="module")
def batch(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("plan")
    compile_driver(tmp, DRIVER, "-fPIC", "-shared", "-o", str(tmp / "d.so"))
    f = C.CDLL(str(tmp / "d.so")).batch

    def of(first, n_pieces, block, P, lanes, seg_bytes, piece_bytes):
        out = np.zeros(2, np.int64)
        f(ptr(first), C.c_int64(first.size), *(C.c_int64(int(v)) for v in (
            n_pieces, block, P, lanes, seg_bytes, piece_bytes)), ptr(out))
        return int(out[0]), int(out[1])
    return of


def most_pieces(first, n_pieces, block, segments):
    ends = np.append(first, n_pieces)
    return max(int(ends[min(j + segments, b + block, first.size)] - ends[j])
               for b in range(0, first.size, block)
               for j in range(b, min(b + block, first.size), segments))


@pytest.mark.parametrize("P,C_,block,per_segment", [
    (16384, 1000, 65, 0), (16384, 1000, 65, 60), (16384, 1000, 65, 999), (1024, 100, 655, 99),
    (65536, 200, 327, 20), (300000, 1000, 65, 999), (64, 4, 3072, 3), (1, 1000, 65, 999),
    (262144, 8, 40, 7)])
def test_batches_hold_their_bounds(batch, P, C_, block, per_segment):
    rng = np.random.default_rng(P + per_segment)
    n_seg = 2 * block + block // 3 + 1
    count = 1 + rng.integers(per_segment // 2, per_segment + 1, size=n_seg)
    first = np.concatenate([[0], np.cumsum(count)[:-1]]).astype(np.int32)
    n_pieces, lanes = int(count.sum()), 1 << 20
    for size in (4, 8):
        seg_bytes, piece_bytes = (C_ + 3) // 4 * 3 * P * size, 168 * P
        segments, pieces = batch(first, n_pieces, block, P, lanes, seg_bytes, piece_bytes)
        fits = lambda s: (s * seg_bytes + most_pieces(first, n_pieces, block, s) * piece_bytes  # noqa: E731
                          <= 8 * GIB or s * P <= 1 << 18 or s == 1)
        assert 1 <= segments <= block and (segments * P <= lanes or segments == 1)
        assert segments * seg_bytes <= 8 * GIB or segments == 1
        assert pieces == most_pieces(first, n_pieces, block, segments)
        assert fits(segments)
        n = -(-block // segments)
        if n > 1:     # the next coarser even split breaks a bound
            s = -(-block // (n - 1))
            assert s * P > lanes or s * seg_bytes > 8 * GIB or not fits(s)


def test_dense_samples_do_not_take_the_lanes_memory_for_maps(batch):
    # 1,024 particles, 100-step segments, a sample at every step: 655 segments a launch
    # would be 11.3 GB of maps
    first = (100 * np.arange(655)).astype(np.int32)
    segments, pieces = batch(first, 65500, 655, 1024, 1 << 20, 25 * 3 * 1024 * 4, 168 * 1024)
    assert segments * 1024 > 1 << 18 and pieces * 168 * 1024 < 8 * GIB
