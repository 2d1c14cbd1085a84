"""GPU: vector runs of the per-axis form, whose x passes are fused with the update and whose z transforms with the
dyadic Green's multiply (three components of a z line in LDS): against the FP64 oracle and
against CBS_FORM_AXES, which runs every pass on its own."""
import numpy as np
import pytest

from helpers import params, rel, sphere_ri, random_field
from oracle.cbs import ForwardSolverConvergentBorn as Oracle

pytestmark = pytest.mark.gpu


# RI grids: 8 voxels of boundary come on top.  z of 27 (compiled), 29 (matrix cores), 216 (compiled, 8-wide tiles),
# 205 (matrix cores, two blocks a CU just fit), 430 (separate passes); ragged and odd x
@pytest.mark.parametrize('ri', [(17, 17, 19), (35, 27, 21), (10, 9, 208), (27, 5, 197), (9, 6, 422)])
@pytest.mark.parametrize('tol', [0.0, 1e-3])
def test_vector_axes(ri, tol):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    p = params(ri, bt_px_target=4, iterations=8, vector_simulation=True)
    RI = sphere_ri(ri, 0.5, n_s=1.42)
    fields = [np.stack([random_field(ri, 3 * a + j) for j in range(3)], axis=-1) for a in range(2)]
    u = np.stack(fields, axis=-1)
    out = []
    for form in (1, 3):
        s = FORWARD_SOLVER_CONVERGENT_BORN(p, options=dict(form=form))
        s.set_RI(RI)
        if tol:
            s.set_convergence(tol)
        out.append(s.solve_incident(u))
        s.close()
    assert rel(out[0], out[1]) <= 2e-6
    if tol == 0.0:
        o = Oracle(p, io_kernels=False)
        o.set_RI(RI)
        ref = np.stack([o.born_loop(f) for f in fields], axis=-1)
        err = rel(out[0], ref)
        print(ri, 'rel err', err, flush=True)
        assert err <= 1e-5


def test_fixed_transforms_keep_the_separate_passes():
    """cbs_set_transforms(FIXED): a vector run's fields are those of the separate passes bit for bit."""
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, _lib
    ri = (17, 17, 19)
    p = params(ri, bt_px_target=4, iterations=6, vector_simulation=True)
    u = np.stack([np.stack([random_field(ri, j) for j in range(3)], axis=-1)], axis=-1)
    out = []
    for form in (1, 3):
        s = FORWARD_SOLVER_CONVERGENT_BORN(p, options=dict(form=form))
        _lib.check(_lib.lib.cbs_set_transforms(s._h, _lib.CBS_TRANSFORMS_FIXED))
        s.set_RI(sphere_ri(ri, 0.5, n_s=1.42))
        out.append(s.solve_incident(u))
        s.close()
    np.testing.assert_array_equal(out[0], out[1])
