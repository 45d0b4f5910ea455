"""FP64 Heun clusters on two lanes per particle: cached pair geometry and shared draws.

Each lane keeps the geometry of its first eight partners (clusters of up to 16) and
draws six of the twelve normals of four steps.  Sizes below, at and above that line
and at the largest workgroup of the cached kernel (128 particles), alone and packed,
with and without renormalisation, over step counts that end inside a group of four:
bit for bit against the kernel without the cache and against one lane per particle,
and one ensemble against the oracle (1e-10 of Ms, the tolerance of the other FP64
cluster tests).
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MU0, DT = 1.25663706e-6, 1e-14
PER = ("radius", "anisotropy", "anisotropy_axis", "magnetisation_direction", "location")


def run(sizes, steps, shape="sine", renorm=False):
    rng = np.random.default_rng(100 + sum(sizes))
    e = G.cluster_ensemble(np.array(sizes), 10e-9, 0.10, 2.2, rng)
    e.update(magnetisation=4e5, damping=0.1, temperature=300.0, field_shape=shape,
             field_amplitude=0.02 / MU0, field_frequency=3e8,
             seeds=rng.integers(0, 2 ** 31 - 1, size=len(sizes)))
    return e, core.simulate_ensemble(time_step=DT, end_time=(steps + 0.5) * DT, max_samples=5,
                                     interactions=True, use_implicit=False, precision="fp64",
                                     renorm=renorm, **e)


@pytest.mark.parametrize("sizes,steps,shape,renorm", [
    ([2], 1, "sine", False), ([2, 1, 3], 37, "sine", True), ([15, 16], 38, "square", False),
    ([17, 18, 2], 39, "constant", True), ([32, 33], 21, "sine", False),
    ([127, 2], 10, "sine", True), ([128], 9, "constant", False), ([129, 5], 6, "sine", False)])
def test_cached_pairs_give_the_same_bits(sizes, steps, shape, renorm, monkeypatch):
    monkeypatch.setenv("MAGPY_AMD_CLUSTER_LANES", "2")
    got = run(sizes, steps, shape, renorm)[1]
    monkeypatch.setenv("MAGPY_AMD_CLUSTER_CACHE", "0")
    plain = run(sizes, steps, shape, renorm)[1]
    monkeypatch.setenv("MAGPY_AMD_CLUSTER_LANES", "1")
    one = run(sizes, steps, shape, renorm)[1]
    assert np.all(got["status"] == 0)
    for k in ("x", "y", "z", "final_state"):
        np.testing.assert_array_equal(got[k], plain[k])
        np.testing.assert_array_equal(got[k], one[k])


def test_cached_pairs_match_oracle(monkeypatch):
    monkeypatch.setenv("MAGPY_AMD_CLUSTER_LANES", "2")
    sizes, steps = [16, 2, 19, 7], 30
    e, g = run(sizes, steps)
    for m, n in enumerate(sizes):
        b = int(e["member_offsets"][m])
        o = O.full_dynamics(*(e[k][b:b + n] for k in PER), 4e5, 0.1, 300.0, False, True, False,
                            1e-9, DT, (steps + 0.5) * DT, 5, int(e["seeds"][m]),
                            field_shape="sine", field_amplitude=0.02 / MU0, field_frequency=3e8,
                            rng="philox")
        for c in "xyz":
            assert np.allclose(g[c][b:b + n], o[c], rtol=0, atol=4e5 * 1e-10), (m, c)
