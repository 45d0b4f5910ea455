"""Large implicit clusters among many dimers, where two lanes share the pair sums.

Alone or in small company clusters of 9 and more share them over four lanes; among many
dimers the launch takes two.  Every order of summation is the same for both, so each
equals its run alone bit for bit: one-wave workgroups (clusters up to 64) and workgroups
of four waves, with and without interactions.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MU0, DT, STEPS = 1.25663706e-6, 5e-13, 5
PER = ("radius", "anisotropy", "anisotropy_axis", "magnetisation_direction", "location")


@pytest.mark.parametrize("large,interactions", [
    ([9], True), ([10, 11, 12, 13, 14, 15, 16, 17], True), ([63, 33, 64], True),
    ([64, 9], False), ([65, 200, 131, 256, 9], True)])
def test_large_members_among_dimers_equal_each_alone(large, interactions):
    print("CASE cluster_targets", large, flush=True)
    sizes = np.array([2] * 9000 + large + [2] * 9000)
    rng = np.random.default_rng(sum(large))
    e = G.cluster_ensemble(sizes, 10e-9, 0.10, 2.2, rng)
    e.update(magnetisation=4e5, damping=0.1, temperature=300.0, field_shape="sine",
             field_amplitude=0.02 / MU0, field_frequency=3e8,
             seeds=rng.integers(0, 2 ** 31 - 1, size=sizes.size))
    kw = dict(time_step=DT, end_time=STEPS * DT, max_samples=3, interactions=interactions,
              use_implicit=True, precision="fp64")
    g = core.simulate_ensemble(**kw, **e)
    assert np.all(g["status"] == 0)
    for m in [0, 17, 8999] + list(range(9000, 9000 + len(large))) + [sizes.size - 1]:
        b, x = int(e["member_offsets"][m]), int(e["member_offsets"][m + 1])
        one = dict(e, member_offsets=np.array([0, x - b]), seeds=e["seeds"][m:m + 1],
                   **{k: e[k][b:x] for k in PER})
        a = core.simulate_ensemble(**kw, **one)
        for k in ("x", "y", "z", "final_state"):
            np.testing.assert_array_equal(a[k], g[k][b:x])
