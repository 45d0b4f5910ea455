"""Pathwise gradients whatever the forward blocks' lengths.

A last block shorter than a third of the others is dealt out to them, or a single
block and its rest are cut in two.  Runs on both sides of these lines (a block of 64
particles takes 2,048 segments in FP32 and 3,072 in FP64), in the default blocks and in
forced ones of a few segments: the forward results are the same bits, and the
gradient is the same sum of double-precision maps per segment, folded in the same
order (1e-12 of it, for the sums' roundings).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MS, T, DT, F, P, C = 4e5, 300.0, 1e-14, 3e5, 64, 4
THETA = np.array([23e3, 0.1, 0.02 / 1.25663706e-6, 10e-9])


@pytest.mark.parametrize("precision,segments", [
    ("fp32", 2047), ("fp32", 2049), ("fp32", 2730), ("fp32", 2731), ("fp32", 4097),
    ("fp32", 6143), ("fp64", 3072), ("fp64", 3073), ("fp64", 6200)])
def test_gradient_does_not_depend_on_blocks(precision, segments, monkeypatch):
    N = C * segments - 1
    rng = np.random.default_rng(segments)
    shape, ax = np.exp(0.1 * rng.normal(size=P)), G.uniform_random_axes(P, rng)
    seeds = rng.integers(1, 2 ** 31 - 1, size=P)
    ks = [0, 5, N // 2, C * 2048, N]
    ks = sorted(k for k in ks if k <= N)
    w = rng.normal(size=len(ks))
    out = []
    for forced in (None, "4096"):
        if forced:
            monkeypatch.setenv("MAGPY_AMD_ADJOINT_STEPS_PER_LAUNCH", forced)
        r = core.Adjoint(shape, ax, ax, seeds, MS, T, F, DT, N, ks, C, precision)
        ens, fin = r.forward(THETA)[:2]
        out.append((np.array(ens), fin, np.array(r.reverse(w, 0.7))))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
    np.testing.assert_allclose(out[0][2], out[1][2], rtol=1e-12)
