"""GPU: a set_RI that runs out of device memory.  A real RI after a complex one makes the potential's buffer grow; if
that fails, the handle has no potential: solves are refused until the next set_RI that succeeds."""
import numpy as np
import pytest

from helpers import MB, params, take_memory

pytestmark = pytest.mark.gpu


def test_failed_growth_leaves_no_potential():
    from inverse_solver_amd import device as dv
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, _lib
    ri = (312, 312, 312)                    # 320^3: V is 262 MB of complex64, 393 MB with the real part behind it
    p = params(ri, iterations=2)
    RI = np.full(ri, 1.336)
    RI[100:200, 100:200, 100:200] = 1.38
    u = np.ones(ri, np.complex64)
    s = FORWARD_SOLVER_CONVERGENT_BORN(p)
    s.set_RI(RI + 1j * 1e-3 * (RI > 1.35))
    s.solve_incident(u)                     # the state buffers are there before memory is taken
    hold = take_memory(32 * MB)
    try:
        if dv.mem_info()[0] > 64 * MB:       # V (262 MB) is given back before the new one is asked for
            pytest.skip('device memory could not be taken')
        try:
            s.set_RI(RI)
        except _lib.CbsError as e:
            assert e.code == _lib.CBS_ERR_MEMORY
        else:
            pytest.skip('device memory was given back by something else')
        with pytest.raises(_lib.CbsError) as e:
            s.solve_incident(u)
        assert e.value.code == _lib.CBS_ERR_STATE
    finally:
        for b in hold:
            b.free()
    s.set_RI(RI)
    got = s.solve_incident(u)
    t = FORWARD_SOLVER_CONVERGENT_BORN(p)
    t.set_RI(RI)
    np.testing.assert_array_equal(got, t.solve_incident(u))
    s.close()
    t.close()


def test_footprint_counts_the_real_part():
    """A real RI's potential takes 12 bytes a voxel in every form (complex64 and the real part behind it): the unfused
    form, which does not read the real part, holds it too."""
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    ri = (40, 30, 25)
    p = params(ri, iterations=2)
    RI = np.full(ri, 1.336)
    RI[10:20, 10:20, 10:20] = 1.38
    real, cplx = {}, {}
    for form in (1, 3):
        s = FORWARD_SOLVER_CONVERGENT_BORN(p, options=dict(form=form))
        s.set_RI(RI)
        real[form] = s.footprint(2)
        s.set_RI(RI + 1j * 1e-3 * (RI > 1.35))
        cplx[form] = s.footprint(2)
        n = int(np.prod(s.simulation_size))
        s.close()
    assert real[3] == real[1] == cplx[1] + 4 * n == cplx[3] + 4 * n
