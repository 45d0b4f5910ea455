"""Implicit clusters in the fixed scratch: its 64 MiB go to particles, not to helper lanes.

Members of one particle beside a dimer take two lanes each, one of them a helper without
a particle.  200,000 of them with two samples are 252 bytes a particle, 50 MB, and run;
with the helpers in the arrays they would be 100 MB.  Results equal the allocating entry
point's, bit for bit, as do clusters with helper lanes of every kind.
"""
import pytest

from test_zz_no_alloc import ensemble, lib, run, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,samples,steps", [
    ([1] * 199998 + [2], 2, 2), ([1, 2, 3, 5, 7, 9, 11, 6, 1] * 3, 5, 20), ([130, 9, 2, 1], 3, 3)])
def test_particles_alone_take_the_scratch(sizes, samples, steps):
    print("CASE noalloc implicit", len(sizes), flush=True)
    L = lib()
    sp, keep, M, P = ensemble(sizes, 41, 1, 1, True, samples, steps)
    rc_b, b = run(L.mp_ensemble_run_noalloc, sp, M, P, samples)
    assert rc_b == 0, L.mp_last_error()
    rc_a, a = run(L.mp_ensemble_run, sp, M, P, samples)
    assert rc_a == 0, L.mp_last_error()
    same(a, b)
