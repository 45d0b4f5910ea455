"""Device memory of ensembles of several schedules, and where their launch sets are cut.

Members of 64 anisotropies, 1,024 particles each, take their samples at steps that
differ by a step here and there.  Whatever is recorded on the way, a run that asks
for the ensemble sums alone keeps sums (24 bytes per sample and group), and one that
asks for trajectories 24 bytes per sample and particle, beside the records of one
launch set: at most 1 GiB, which is also where a set is cut.  FP32 groups with a field
table are cut at four waves per SIMD, 65,536 lanes.  The sums are the sums of the
samples (1e-12 of Ms times the particles: FP64 sums in another order).
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MU0, MS, DT = 1.25663706e-6, 4e5, 1e-14
GIB, ARRAYS = 1 << 30, 128 << 20   # the inputs of 65,536 particles and the slabs they share


def ensemble(members, size, steps, samples, precision, **kw):
    rng = np.random.default_rng(5)
    P = members * size
    ax = G.uniform_random_axes(P, rng)
    return dict(radius=np.full(P, 10e-9),
                anisotropy=np.repeat(23e3 * np.exp(0.1 * rng.normal(size=members)), size),
                anisotropy_axis=ax, magnetisation_direction=ax, location=np.zeros((P, 3)),
                member_offsets=size * np.arange(members + 1), magnetisation=MS, damping=0.1,
                temperature=300.0, field_shape="sine", field_amplitude=0.02 / MU0,
                field_frequency=3e8, seeds=rng.integers(0, 2 ** 31 - 1, size=members),
                time_step=DT, end_time=steps * DT, max_samples=samples, interactions=False,
                precision=precision, **kw)


def free():
    """Free device memory, from the HIP runtime that the library has loaded."""
    hip, f, t = ctypes.CDLL("libamdhip64.so.7"), ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


def test_sums_alone_keep_no_samples():
    print("CASE launch_set_memory sums", flush=True)
    e = ensemble(64, 1024, 2000, 1001, "fp64")
    core.simulate_ensemble(**ensemble(2, 4, 8, 5, "fp64"))   # the library's code and queues
    before = free()
    ses = core.Session(trajectories=False, **e)
    ses.advance(1)
    used, sets = before - free(), ses.info()["launches"]
    assert 2 <= sets < 64        # several groups share a launch, and the records cut the sets
    assert used <= GIB + ARRAYS
    only = ses.finish()
    before = free()
    ses = core.Session(trajectories=True, **e)
    ses.advance(1)
    samples = 1001 * 24 * 65536
    assert before - free() <= samples + GIB + ARRAYS
    out = ses.finish()
    np.testing.assert_array_equal(only["ensemble_m"], out["ensemble_m"])
    sums = np.stack([out[k].sum(axis=0) for k in "xyz"], axis=1)
    assert np.max(np.abs(sums - only["ensemble_m"])) <= 1e-12 * MS * 65536


@pytest.mark.parametrize("members,size,sets", [(64, 1024, 1), (70, 1024, 2)])
def test_field_table_sets_are_cut_at_the_lanes_of_the_card(members, size, sets):
    print("CASE launch_set_memory table", members, flush=True)
    e = ensemble(members, size, 8, 5, "fp32")
    ses = core.Session(trajectories=True, **e)
    ses.advance(1)
    assert ses.info()["launches"] == sets
    out = ses.finish()
    for m in (0, members // 2, members - 1):
        at = slice(m * size, (m + 1) * size)
        one = {k: v[at] if k in ("radius", "anisotropy", "anisotropy_axis",
                                 "magnetisation_direction", "location") else v
               for k, v in e.items()}
        one.update(member_offsets=np.array([0, size]), seeds=e["seeds"][m:m + 1])
        alone = core.simulate_ensemble(**one)
        for k in "xyz":
            np.testing.assert_array_equal(alone[k], out[k][at])
