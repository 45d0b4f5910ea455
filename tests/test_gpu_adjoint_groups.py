"""Pathwise gradients where the 4-step groups and segments of the maps end.

Runs whose last group holds 1 to 4 steps, segments of one group, one segment
longer than the run, particle counts around a wave (so that a wave of the map
kernel spans two segments), samples inside groups and on their edges, runs of
several forward blocks: the FP64 gradient equals the oracle's forward-mode
tangent (1e-9, as in the other adjoint tests), and FP32 the FP64 one to 1e-3.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MS, T, DT, F = 4e5, 300.0, 1e-14, 1e10
THETA = np.array([23e3, 0.1, 0.02 / 1.25663706e-6, 10e-9])


@pytest.mark.parametrize("P,N,C,ks", [
    (1, 1, 4, [0, 1]), (63, 2, 4, [1]), (64, 3, 8, [0, 2, 3]), (65, 5, 4, [4, 5]),
    (65, 8, 4, [1, 4, 7]), (33, 9, 1000, [2, 3, 8]), (130, 402, 8, [0, 5, 8, 16, 17, 400]),
    (129, 1003, 100, [1, 99, 100, 101, 999, 1003]), (20, 96, 24, [])])
def test_gradient_at_group_ends(P, N, C, ks):
    print("CASE adjoint_groups", P, N, C, flush=True)
    rng = np.random.default_rng(P + N)
    shape, ax = np.exp(0.1 * rng.normal(size=P)), G.uniform_random_axes(P, rng)
    seeds = rng.integers(1, 2 ** 31 - 1, size=P)
    w = rng.normal(size=len(ks))
    grads = {}
    for precision in ("fp64", "fp32"):
        r = core.Adjoint(shape, ax, ax, seeds, MS, T, F, DT, N, ks, C, precision)
        r.forward(THETA)
        grads[precision] = r.reverse(w, 0.7)
    q, dq = core.adjoint_reduced(THETA, shape, MS, T, DT)
    pr = O.path_problem(ax, ax, q[:, 0], q[:, 1], q[:, 2], q[:, 3], F * DT, seeds, N, ks)
    tan, tan_f = O.path_tangent(pr, np.ascontiguousarray(np.transpose(dq, (0, 2, 1))))
    ref = 0.7 / P * tan_f + (MS / P * (w @ tan) if len(ks) else 0.0)
    scale = np.maximum(np.abs(ref), 1e-3 * np.max(np.abs(ref * THETA)) / THETA)
    assert np.max(np.abs(grads["fp64"] - ref) / scale) < 1e-9
    assert np.max(np.abs(grads["fp32"] - ref) / scale) < 1e-3
