"""The squared norm of a cluster in the implicit kernel (magpy_amd/csrc/cluster_norm.h).

Two or four lanes add their squares first (by lane swaps, so pairs, then pairs of
pairs); which of them a launch does depends on its largest cluster.  The norm of a
member, which decides its Newton count, must be the same bits either way: every size up
to the largest workgroup, from every start that two lanes allow, and within the
rounding of a sum of n terms of the exact one.
"""
import ctypes as C
from fractions import Fraction

import numpy as np
import pytest

from test_cluster_layout_cpu import compile_driver, ptr

DRIVER = r'''
#include "cluster_norm.h"
extern "C" double norm(int kt, const double *red, int cb, int ce)
{
    return kt == 2 ? mp::cluster_square<2>(red, cb, ce) : mp::cluster_square<4>(red, cb, ce);
}
'''


@pytest.fixture(scope="module")
def norm(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("norm")
    compile_driver(tmp, DRIVER, "-ffp-contract=off", "-fPIC", "-shared", "-o", str(tmp / "d.so"))
    f = C.CDLL(str(tmp / "d.so")).norm
    f.restype = C.c_double

    def of(kt, squares, start):
        lanes = np.zeros((start + len(squares) + 7) // 4 * 4)
        lanes[start:start + len(squares)] = squares      # helper lanes add nothing
        pairs = lanes[0::2] + lanes[1::2]
        red = pairs if kt == 2 else pairs[0::2] + pairs[1::2]
        return f(kt, ptr(np.ascontiguousarray(red)), start, start + len(squares))
    return of


@pytest.mark.parametrize("sizes", [range(1, 9), range(9, 66), [95, 96, 97, 127, 128, 255, 256]])
def test_two_and_four_lanes_give_the_same_bits(norm, sizes):
    rng = np.random.default_rng(1)
    for n in sizes:
        for _ in range(20):
            sq = rng.normal(size=n) ** 2 * 10.0 ** rng.uniform(-18, 0)
            four = norm(4, sq, 0)
            assert all(norm(2, sq, s) == four for s in (0, 2, 4, 6))
            assert norm(4, sq, 4) == four
            exact = sum(Fraction(x) for x in sq)
            assert abs(Fraction(four) - exact) <= n * Fraction(2) ** -53 * exact
