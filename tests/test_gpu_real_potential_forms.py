"""A real RI's potential is read as its real part alone by the four-pass form and the per-axis form's fused x
passes (compiled lengths and matrix-core products): the fields equal those of the same potential given as
complex64, bit for bit."""
import numpy as np
import pytest

from helpers import params
from test_gpu_potential import _set_host

pytestmark = pytest.mark.gpu


# simulation grids: 24^3 (compiled lengths, a part row block), 43 x 35 x 29, 75 x 45 x 67, 150 x 107 x 31
@pytest.mark.parametrize('ri,form', [((16, 16, 16), 'rows'), ((16, 16, 16), 'plain'), ((16, 16, 16), 'axes'),
                                     ((35, 27, 21), 'plain'), ((67, 37, 59), 'plain'), ((142, 99, 23), 'plain')])
def test_real_potential_forms(ri, form):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    from inverse_solver_amd.phantoms import bead_ri, incident_plane_waves
    p = params(ri, bt_px_target=4, iterations=7, return_reflection=False)
    RI = bead_ri(ri, 7, 1.46, 1.336)
    u = incident_plane_waves(list(ri), 3, 1.2, 0.532, 1.336, [0.1, 0.1, 0.1]).astype(np.complex64)
    out = []
    for real in (False, True):
        s = FORWARD_SOLVER_CONVERGENT_BORN(p, options=dict(form=dict(plain=1, rows=2, axes=3)[form]))
        if real:
            s.set_RI(RI)
        else:
            _set_host(s, RI, False)
        assert s.plan()['form'] == form
        out.append(s.solve_incident(u))
        s.close()
    np.testing.assert_array_equal(out[0], out[1])
