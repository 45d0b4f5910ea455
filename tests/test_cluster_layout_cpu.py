"""The host rules of the cluster kernels' layout (magpy_amd/csrc/cluster_layout.hpp).

The autotuner times the launch set with the most particles, wherever it stands among
the sets, and a layout is remembered for the device, the largest cluster, the particles
of that set, the precision and the forced lanes: a change of any one is another entry.
"""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "magpy_amd", "csrc")
DRIVER = r'''
#include "cluster_layout.hpp"
using namespace mp_host;
static LayoutCache cache;
extern "C" {
// sets as their sizes and, one after the other, their groups
int64_t largest(const int *sizes, int n_sets, const int *groups, const int64_t *begin, int n_groups,
                int64_t *particles)
{
    std::vector<std::vector<int>> sets;
    for (int i = 0; i < n_sets; groups += sizes[i++]) sets.emplace_back(groups, groups + sizes[i]);
    return (int64_t)largest_set(sets, std::vector<int64_t>(begin, begin + n_groups + 1), particles);
}
int known(int device, int64_t nmax, int64_t particles, int precision, int forced, int *block, int *lanes)
{
    ClusterLayout l;
    if (!cache.find(LayoutKey{device, nmax, particles, precision, forced}, l)) return 0;
    *block = l.block;
    *lanes = l.lanes;
    return 1;
}
void keep(int device, int64_t nmax, int64_t particles, int precision, int forced, int block, int lanes)
{
    ClusterLayout l;
    l.block = block;
    l.lanes = lanes;
    cache.keep(LayoutKey{device, nmax, particles, precision, forced}, l);
}
}
'''


def compile_driver(tmp, text, *flags):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    (tmp / "d.cpp").write_text(text)
    subprocess.run([gxx, "-std=c++17", "-O2", "-I", CSRC, *flags, str(tmp / "d.cpp")], check=True)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("layout")
    compile_driver(tmp, DRIVER, "-fPIC", "-shared", "-o", str(tmp / "d.so"))
    return C.CDLL(str(tmp / "d.so"))


def ptr(a):
    return a.ctypes.data_as(C.c_void_p)


@pytest.mark.parametrize("sets,sizes,best", [
    ([[0]], [5], 0), ([[0], [1, 2, 3]], [2, 900, 1, 40], 1), ([[0, 2], [1]], [3, 7, 5], 0),
    ([[0], [1]], [6, 6], 0), ([[0], [1, 3], [2]], [1, 1, 64, 1], 2)])
def test_the_largest_set_is_timed(lib, sets, sizes, best):
    n = np.array([len(s) for s in sets], np.int32)
    groups = np.array([g for s in sets for g in s], np.int32)
    begin = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    particles = C.c_int64()
    lib.largest.restype = C.c_int64
    assert lib.largest(ptr(n), len(sets), ptr(groups), ptr(begin), len(sizes),
                       C.byref(particles)) == best
    assert particles.value == sum(sizes[g] for g in sets[best])


def test_layouts_are_remembered_per_device_and_set(lib):
    key = [1, 64, 135000, 0, 0]
    args = lambda k: [C.c_int(k[0]), C.c_int64(k[1]), C.c_int64(k[2]), C.c_int(k[3]),  # noqa: E731
                      C.c_int(k[4])]
    block, lanes = C.c_int(), C.c_int()
    lib.keep(*args(key), 512, 2)
    assert lib.known(*args(key), C.byref(block), C.byref(lanes)) == 1
    assert (block.value, lanes.value) == (512, 2)
    for i in range(5):
        other = list(key)
        other[i] += 1
        assert lib.known(*args(other), C.byref(block), C.byref(lanes)) == 0
