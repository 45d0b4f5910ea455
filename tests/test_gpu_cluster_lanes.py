"""Implicit midpoint clusters at the sizes where the lane layout changes.

Clusters of up to 8 particles share their pair sums over two lanes, larger ones
over four, with helper lanes up to a multiple; up to 64 particles a workgroup is
one wave.  Sizes at, below and above each of these lines, alone and packed with
others, against the oracle's 3N x 3N Newton run (1e-10 of Ms, the tolerance of
the other implicit cluster tests, equal Newton counts), and bit for bit against
the same member alone, whatever the largest cluster beside it is.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MU0, DT = 1.25663706e-6, 5e-13
PER = ("radius", "anisotropy", "anisotropy_axis", "magnetisation_direction", "location")


def clusters(sizes, seed):
    rng = np.random.default_rng(seed)
    e = G.cluster_ensemble(sizes, 10e-9, 0.10, 2.2, rng)
    e.update(magnetisation=4e5, damping=0.1, temperature=300.0, field_shape="sine",
             field_amplitude=0.02 / MU0, field_frequency=3e8,
             seeds=rng.integers(0, 2 ** 31 - 1, size=len(sizes)))
    return e


def run(e, steps):
    return core.simulate_ensemble(time_step=DT, end_time=steps * DT, max_samples=5,
                                  interactions=True, use_implicit=True, precision="fp64", **e)


@pytest.mark.parametrize("sizes,steps", [([1], 40), ([2], 40), ([3, 1, 2], 40), ([8, 7], 40),
                                         ([9, 2, 8, 5], 20), ([13, 11, 10], 20), ([63, 64], 6),
                                         ([65, 3, 1], 4), ([128, 2], 2)])
def test_cluster_sizes_match_oracle(sizes, steps):
    print("CASE cluster_lanes", sizes, flush=True)
    e = clusters(sizes, 100 + sum(sizes))
    g = run(e, steps)
    assert np.all(g["status"] == 0)
    newton = 0
    for m, n in enumerate(sizes):
        b = int(e["member_offsets"][m])
        o = O.full_dynamics(*(e[k][b:b + n] for k in PER), 4e5, 0.1, 300.0, False, True, True,
                            1e-9, DT, steps * DT, 5, int(e["seeds"][m]), field_shape="sine",
                            field_amplitude=0.02 / MU0, field_frequency=3e8, rng="philox")
        for c in "xyz":
            assert np.allclose(g[c][b:b + n], o[c], rtol=0, atol=4e5 * 1e-10), (m, c)
        newton += o["stats"].newton_iters
        one = dict(e, member_offsets=np.array([0, n]), seeds=e["seeds"][m:m + 1],
                   **{k: e[k][b:b + n] for k in PER})
        alone = run(one, steps)
        for c in "xyz":
            np.testing.assert_array_equal(alone[c], g[c][b:b + n])
    assert g["newton_iters"] == newton


def test_largest_workgroup():
    """Clusters of up to 256 particles (four waves): the packed run equals each alone."""
    print("CASE cluster_lanes_256", flush=True)
    sizes = [255, 256, 129]
    e = clusters(sizes, 9)
    g = run(e, 3)
    assert np.all(g["status"] == 0) and np.all(np.isfinite(g["final_state"]))
    for m, n in enumerate(sizes):
        b = int(e["member_offsets"][m])
        one = dict(e, member_offsets=np.array([0, n]), seeds=e["seeds"][m:m + 1],
                   **{k: e[k][b:b + n] for k in PER})
        np.testing.assert_array_equal(run(one, 3)["final_state"], g["final_state"][b:b + n])
