"""Runs long enough to tune the cluster layout whose members have several schedules.

The layout is timed on the largest launch set; results do not depend on it, so each
member equals its own run bit for bit, also after a resume too close to the end to
time anything.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MU0, DT, STEPS = 1.25663706e-6, 1e-14, 20000
PER = ("radius", "anisotropy", "anisotropy_axis", "magnetisation_direction", "location")


@pytest.mark.parametrize("precision,shape", [("fp64", "sine"), ("fp32", "constant")])
def test_members_of_a_tuned_run_equal_each_alone(precision, shape):
    print("CASE cluster_tuned_sets", precision, flush=True)
    sizes = np.array([3, 2, 2, 4, 3, 2])
    rng = np.random.default_rng(17)
    e = G.cluster_ensemble(sizes, 10e-9, 0.10, 2.2, rng)
    spread = np.array([1.3, 1.0, 1.0, 1.0, 1.1, 0.9])
    e["anisotropy"] = e["anisotropy"] * np.repeat(spread, sizes)
    e.update(magnetisation=4e5, damping=0.1, temperature=300.0, field_shape=shape,
             field_amplitude=0.02 / MU0, field_frequency=3e8,
             seeds=rng.integers(0, 2 ** 31 - 1, size=sizes.size))
    kw = dict(time_step=DT, end_time=STEPS * DT, max_samples=101, interactions=True,
              precision=precision)
    whole = core.simulate_ensemble(**kw, **e)
    assert np.all(whole["status"] == 0)
    late = core.simulate_ensemble(start_step=STEPS - 9, start_state=whole["final_state"],
                                  **kw, **e)
    for m, n in enumerate(sizes):
        b = int(e["member_offsets"][m])
        one = dict(e, member_offsets=np.array([0, n]), seeds=e["seeds"][m:m + 1],
                   **{k: e[k][b:b + n] for k in PER})
        a = core.simulate_ensemble(**kw, **one)
        for k in ("x", "y", "z", "final_state"):
            np.testing.assert_array_equal(a[k], whole[k][b:b + n])
        a = core.simulate_ensemble(start_step=STEPS - 9,
                                   start_state=whole["final_state"][b:b + n], **kw, **one)
        np.testing.assert_array_equal(a["final_state"], late["final_state"][b:b + n])
