"""GPU: CBS_TRANSFORMS_FIXED on the fused form keeps to one split of y, whatever was measured before the switch."""
import numpy as np
import pytest

from helpers import params, random_field, sphere_ri

pytestmark = pytest.mark.gpu


def test_fixed_drops_a_measured_split():
    """cbs_autotune on a default handle takes any split; after the switch the handle is one that was fixed from the
    start, bit for bit.  A split that the caller sets afterwards stays."""
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, _lib
    ri = (88, 88, 88)
    p = params(ri, iterations=6)
    RI = sphere_ri(ri, 1.5, n_s=1.42)
    u = random_field(ri, 5)

    def fixed(s):
        _lib.check(_lib.lib.cbs_set_transforms(s._h, _lib.CBS_TRANSFORMS_FIXED))

    fresh, tuned, forced = (FORWARD_SOLVER_CONVERGENT_BORN(p) for _ in range(3))
    fixed(fresh)
    fresh.set_RI(RI)
    ref = fresh.solve_incident(u)
    for s in (tuned, forced):
        s.set_RI(RI)
        s.autotune(1, 4)
        print('measured', s.plan(), 'fixed', fresh.plan(), flush=True)
        assert s.plan()['a'] != fresh.plan()['a']      # 96^3 with one rhs: 24 us an iteration against 32
    # the measured options also go where other options were set in between
    tuned.set_options(track_norms=1)
    fixed(tuned)
    assert tuned.plan() == fresh.plan()
    tuned.set_RI(RI)                                   # the shift state starts over
    np.testing.assert_array_equal(tuned.solve_incident(u), ref)
    forced.set_options(split_a=48, tile_t=0, threads_real=0, threads_kspace=0)
    fixed(forced)
    assert forced.plan()['a'] == 48
    for s in (fresh, tuned, forced):
        s.close()
