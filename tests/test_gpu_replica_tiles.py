"""The replica product's tiles: block shapes, paddings, fused and separate stages.

A product runs in blocks of four wave pairs (from 1,024 pairs of 64 replicas x 32
particles on 256 CUs), of one pair of 64 replicas, or of one pair of 32; particles are
padded to 64 and replicas to 128.  Checked at the edges of each: the field of
replicas in every part of the first and last tiles against the FP64 product (the
tolerances of the modes: 2e-6 and 5e-5 of the field's norm), the stages in the
epilogue against the separate ones bit for bit, and replicas of a large ensemble
against the same replicas in a small one bit for bit (the sums have the same order
in every block shape).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MU0, MS, DT = 1.25663706e-6, 4e5, 1e-14
TOL = {"gemm_f32": 2e-6, "gemm_bf16x3": 5e-5}
# (particles, replicas): one pair of 32, the same with every padding, one pair of 64,
# four pairs
SHAPES = [(2, 1), (32, 64), (33, 65), (64, 128), (65, 31), (129, 200), (512, 2112), (512, 4096)]


def cluster(n):
    return G.random_cluster(n, 10e-9, 0.10, 2.2, np.random.default_rng(n))


def states(n, reps, seed=1):
    m = np.random.default_rng(seed).normal(size=(reps, n, 3))
    return m / np.linalg.norm(m, axis=2, keepdims=True)


@pytest.mark.parametrize("mode", list(TOL))
@pytest.mark.parametrize("n,reps", SHAPES)
def test_field(n, reps, mode):
    loc, radius, K = cluster(n), np.full(n, 10e-9), np.full(n, 23e3)
    m = states(n, reps)
    h = core.dipolar_field(loc, radius, K, MS, m, mode=mode)
    some = sorted({0, 31, 32, 63, 64, 127, reps // 2, reps - 33, reps - 1} & set(range(reps)))
    ref = core.dipolar_field(loc, radius, K, MS, m[some], mode="pairs")
    err = np.linalg.norm(h[some] - ref, axis=(1, 2)) / np.linalg.norm(ref, axis=(1, 2))
    assert err.max() < TOL[mode]


def run(n, reps, mode, steps=12, first=0, renorm=False):
    rng = np.random.default_rng(7)
    axes = G.uniform_random_axes(n, rng)
    K = 23e3 * np.exp(0.1 * rng.normal(size=n))
    e = dict(member_offsets=np.arange(reps + 1) * n, radius=np.full(n * reps, 10e-9),
             anisotropy=np.tile(K, reps), anisotropy_axis=np.tile(axes, (reps, 1)),
             magnetisation_direction=states(n, 4200 if n > 200 else 300, 3)[
                 first:first + reps].reshape(-1, 3),
             location=np.tile(cluster(n), (reps, 1)), magnetisation=MS, damping=0.1,
             temperature=300.0, field_shape=["sine"] * reps, field_amplitude=0.02 / MU0,
             field_frequency=3e5, seeds=np.arange(first, first + reps) + 11)
    ses = core.Session(time_step=DT, end_time=(steps + 0.5) * DT, max_samples=4, precision="fp32",
                       dipolar=mode, renorm=renorm, trajectories=n < 200, **e)
    assert ses.info()["dipolar"] == mode
    return ses.finish()


@pytest.mark.parametrize("mode", list(TOL))
@pytest.mark.parametrize("n,reps", [s for s in SHAPES if s[1] > 1])
def test_stages_in_the_epilogue(n, reps, mode, monkeypatch):
    res = {}
    for fused in ("1", "0"):
        monkeypatch.setenv("MAGPY_AMD_REPLICA_FUSED", fused)
        res[fused] = run(n, reps, mode, renorm=n == 33)
    for k in ("final_state", "status") + (("x", "y", "z") if n < 200 else ()):
        np.testing.assert_array_equal(res["1"][k], res["0"][k])
    scale = MS * n * reps
    np.testing.assert_allclose(res["1"]["ensemble_m"], res["0"]["ensemble_m"], rtol=0,
                               atol=1e-13 * scale)
    assert np.all(res["1"]["status"] == 0)


@pytest.mark.parametrize("mode", list(TOL))
@pytest.mark.parametrize("n,reps", [(129, 200), (512, 2112), (512, 4096)])
def test_replicas_do_not_depend_on_their_number(n, reps, mode):
    full = run(n, reps, mode)["final_state"].reshape(reps, n, 3)
    for first, count in ((0, 1), (reps - 33, 33)):
        part = run(n, count, mode, first=first)["final_state"].reshape(count, n, 3)
        np.testing.assert_array_equal(part, full[first:first + count])
