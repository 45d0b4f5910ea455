"""Uploads that share one copy, and states and samples on their way out.

Arrays of up to 1 MiB are placed in shared pieces of device memory and sent
together, larger ones alone; samples are repacked from [record][component][slot]
to the caller's [particle][sample] in tiles of 16, and a replica ensemble's state
is packed on the device.  Each must give what a run of its own gives, bit for bit:
a member alone (tile edges in both directions), a slice of an ensemble whose
arrays cross the 1 MiB line, and the replica states against the samples.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MU0, MS = 1.25663706e-6, 4e5


def spheres(P, seed=5):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=(2, P, 3))
    v /= np.linalg.norm(v, axis=2, keepdims=True)
    return dict(member_offsets=np.arange(P + 1), radius=np.full(P, 7e-9),
                anisotropy=np.full(P, 3e4), anisotropy_axis=v[0], magnetisation_direction=v[1],
                location=np.zeros((P, 3)), magnetisation=MS, damping=0.1, temperature=300.0,
                field_shape=["sine"] * P, field_amplitude=0.02 / MU0,
                field_frequency=np.full(P, 3e5), seeds=np.arange(P) + 100)


def cut(e, a, b):
    c = {k: (v[a:b] if np.ndim(v) and k not in ("member_offsets", "field_shape") else v)
         for k, v in e.items()}
    c.update(member_offsets=np.arange(b - a + 1), field_shape=e["field_shape"][a:b])
    return c


def run(e, steps, S, precision, traj=True):
    dt = 1e-13
    return core.simulate_ensemble(**e, time_step=dt, end_time=(steps + 0.5) * dt, max_samples=S,
                                  interactions=False, precision=precision, trajectories=traj)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("P", [1, 15, 16, 17, 33])
@pytest.mark.parametrize("S", [2, 15, 16, 17, 33])
def test_samples_of_members_alone(P, S, precision):
    e = spheres(P)
    r = run(e, 40, S, precision)
    for m in sorted({0, P // 2, P - 1}):
        one = run(cut(e, m, m + 1), 40, S, precision)
        for k in "xyz":
            np.testing.assert_array_equal(one[k][0], r[k][m])
        np.testing.assert_array_equal(one["final_state"][0], r["final_state"][m])


@pytest.mark.parametrize("P", [131072, 131073, 300001])
def test_arrays_around_the_limit_of_shared_uploads(P):
    e = spheres(P)
    r = run(e, 2, 2, "fp64", traj=False)
    for a, b in ((0, 65), (P // 2, P // 2 + 64), (P - 63, P)):
        c = run(cut(e, a, b), 2, 2, "fp64", traj=False)
        np.testing.assert_array_equal(c["final_state"], r["final_state"][a:b])


@pytest.mark.parametrize("mode", ["gemm_bf16x3", "gemm_f32"])
@pytest.mark.parametrize("n,reps", [(33, 5), (128, 129)])
def test_replica_states_are_the_samples(n, reps, mode):
    rng = np.random.default_rng(2)
    one = G.cluster_ensemble(np.array([n]), 10e-9, 0.10, 2.2, rng)
    e = {k: np.concatenate([one[k]] * reps) for k in
         ("radius", "anisotropy", "anisotropy_axis", "location")}
    m0 = rng.normal(size=(n * reps, 3))
    e["magnetisation_direction"] = m0 / np.linalg.norm(m0, axis=1, keepdims=True)
    ses = core.Session(member_offsets=np.arange(reps + 1) * n, magnetisation=MS, damping=0.1,
                       temperature=300.0, field_shape=["sine"] * reps,
                       field_amplitude=0.02 / MU0, field_frequency=3e5,
                       seeds=np.arange(reps) + 9, time_step=1e-14, end_time=8.5e-14,
                       max_samples=9, precision="fp32", dipolar=mode, trajectories=True, **e)
    half, step = ses.state()
    np.testing.assert_array_equal(half, e["magnetisation_direction"].astype(np.float32))
    states = [ses.state()[0] for _ in range(ses.info()["n_steps"]) if ses.advance(1)]
    r = ses.finish()
    np.testing.assert_array_equal(states[-1], r["final_state"])
    for s in range(1, 9):
        sample = np.stack([r[c][:, s] for c in "xyz"], axis=1)
        assert any(np.array_equal(sample, st * MS) for st in states)
