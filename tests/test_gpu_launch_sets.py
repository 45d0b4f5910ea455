"""Members of different reduced time steps share launches.

An ensemble whose members differ in anisotropy or damping has a reduced step
per member, and sample times on step boundaries then fall on sample steps that
differ by the rounding of each.  Such members run in one launch that records the
union of their sample steps; each must give, bit for bit, what it gives alone:
FP64 and FP32 Heun (constant field, one sine field with a table row per step,
fields that differ by member), the implicit scheme, clusters, caller-given
noise, renormalisation, samples closer than a step, a resumed run, a session
advanced in blocks.  The ensemble sums are sums of the members' samples (1e-12
of Ms times the particles: FP64 sums in another order).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

core = pytest.importorskip("magpy_amd.core")
from magpy_amd import geometry as G  # noqa: E402

MU0, MS = 1.25663706e-6, 4e5
PER = ("radius", "anisotropy", "anisotropy_axis", "magnetisation_direction", "location")
CASES = {
    "fp64": dict(M=70),
    "fp64_few_waves_square": dict(M=9, shape="square"),
    "fp32_constant": dict(M=70, precision="fp32", shape="constant"),
    "fp32_sine": dict(M=70, precision="fp32"),
    "fp32_sine_renorm": dict(M=131, precision="fp32", renorm=True, S=3),
    "fp32_fields_differ": dict(M=12, precision="fp32", freqs=True),
    "fp64_fields_differ": dict(M=12, freqs=True),
    "implicit": dict(M=40, use_implicit=True, dt=5e-13),
    "clusters_fp64": dict(sizes=[2, 5, 1, 9, 3, 3], S=5),
    "clusters_fp32_constant": dict(sizes=[2, 5, 1, 9, 3, 3], precision="fp32", shape="constant"),
    "clusters_fp32_sine": dict(sizes=[2, 5, 1, 9], precision="fp32"),
    "clusters_implicit": dict(sizes=[2, 5, 1, 12], use_implicit=True, dt=5e-13),
    "noise": dict(M=11, noise=True),
    "noise_fp32": dict(M=11, noise=True, precision="fp32"),
    "dense_samples": dict(M=10, steps=30, S=101),
    "resumed": dict(M=12, start=57),
    "resumed_on_a_sample": dict(M=12, start=60),
}


def build(M=0, sizes=None, shape="sine", freqs=False, seed=3):
    sizes = np.array(sizes if sizes else [1] * M)
    rng = np.random.default_rng(seed)
    e = G.cluster_ensemble(sizes, 10e-9, 0.10, 2.2, rng)
    n = sizes.size
    e["anisotropy"] = e["anisotropy"] * np.repeat(np.exp(0.1 * rng.normal(size=n)), sizes)
    e.update(magnetisation=MS, damping=np.where(np.arange(n) % 5 == 4, 0.2, 0.1),
             temperature=300.0, field_shape=[shape] * n, field_amplitude=0.02 / MU0,
             field_frequency=(rng.choice([1e8, 3e8], size=n) if freqs else np.full(n, 3e8)),
             seeds=rng.integers(0, 2 ** 31 - 1, size=n))
    return e, sizes


def part(e, m):
    b, x = int(e["member_offsets"][m]), int(e["member_offsets"][m + 1])
    one = {k: v[b:x] if k in PER else v for k, v in e.items()}
    one.update(member_offsets=np.array([0, x - b]), seeds=e["seeds"][m:m + 1],
               damping=e["damping"][m:m + 1], field_shape=e["field_shape"][m:m + 1],
               field_frequency=e["field_frequency"][m:m + 1])
    return one, b, x


@pytest.mark.parametrize("name", list(CASES))
def test_members_equal_each_alone(name):
    print("CASE launch_sets", name, flush=True)
    c = dict(CASES[name])
    e, sizes = build(c.pop("M", 0), c.pop("sizes", None), c.pop("shape", "sine"),
                     c.pop("freqs", False))
    dt, S, steps = c.pop("dt", 1e-14), c.pop("S", 11), c.pop("steps", 200)
    start, noise = c.pop("start", 0), c.pop("noise", False)
    P = int(sizes.sum())
    kw = dict(time_step=dt, end_time=steps * dt, max_samples=S, interactions=len(set(sizes)) > 1,
              **c)
    more, own = {}, lambda b, x: {}
    if noise:
        nz = np.random.default_rng(8).normal(size=(steps + 2, P, 3))
        more, own = dict(noise=nz), lambda b, x: dict(noise=np.ascontiguousarray(nz[:, b:x]))
    if start:
        st = e["magnetisation_direction"][:, [1, 2, 0]]
        more = dict(start_step=start, start_state=st)
        own = lambda b, x: dict(start_step=start, start_state=st[b:x])  # noqa: E731
    g = core.simulate_ensemble(member_times=True, **kw, **more, **e)
    ens = np.zeros((S, 3))
    for m in range(len(sizes)):
        one, b, x = part(e, m)
        a = core.simulate_ensemble(**kw, **own(b, x), **one)
        for k in "xyz":
            np.testing.assert_array_equal(a[k], g[k][b:x], err_msg="member %d %s" % (m, k))
        np.testing.assert_array_equal(a["final_state"], g["final_state"][b:x])
        np.testing.assert_array_equal(a["time"], g["member_time"][m])
        ens += a["ensemble_m"]
    assert np.array_equal(np.isnan(ens), np.isnan(g["ensemble_m"]))
    assert np.nanmax(np.abs(ens - g["ensemble_m"])) <= 1e-12 * MS * P
    only = core.simulate_ensemble(trajectories=False, **kw, **more, **e)
    np.testing.assert_array_equal(only["ensemble_m"], g["ensemble_m"])


def test_session_blocks(monkeypatch):
    print("CASE launch_sets_session", flush=True)
    e, _ = build(M=33)
    for precision in ("fp64", "fp32"):
        kw = dict(time_step=1e-14, end_time=300e-14, max_samples=7, interactions=False,
                  precision=precision, **e)
        whole = core.simulate_ensemble(**kw)
        ses = core.Session(trajectories=True, **kw)
        for n in (1, 66, 101):
            ses.advance(n)
        st, step = ses.state()
        assert step == 168 and np.all(np.isfinite(st))
        out = ses.finish()
        for k in ("x", "y", "z", "final_state", "ensemble_m"):
            np.testing.assert_array_equal(out[k], whole[k])
        monkeypatch.setenv("MAGPY_AMD_STEPS_PER_LAUNCH", "37")
        again = core.simulate_ensemble(**kw)
        monkeypatch.delenv("MAGPY_AMD_STEPS_PER_LAUNCH")
        for k in ("x", "y", "z", "final_state", "ensemble_m"):
            np.testing.assert_array_equal(again[k], whole[k])
