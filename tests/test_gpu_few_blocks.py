"""Launches of few blocks take other variants of the fused passes than wide batches: a single right-hand
side gives what it gives inside a batch and what the FP64 oracle gives."""
import numpy as np
import pytest

from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, get_default_parameters
from inverse_solver_amd.phantoms import bead_ri, incident_plane_waves
from oracle.cbs import ForwardSolverConvergentBorn as Oracle

pytestmark = pytest.mark.gpu


def _params(n, iters):
    ri = [m - 8 for m in n]
    bt = 4 * 0.2 * 1.336 / 0.532
    return ri, get_default_parameters(dict(size=ri, wavelength=0.532, NA=1.2, RI_bg=1.336, resolution=[0.1] * 3,
                                           vector_simulation=False, iterations_number=iters,
                                           boundary_thickness=[bt] * 3))


# grids whose single-rhs launch takes another real-space or k-space variant, or a variant of its own
@pytest.mark.parametrize('n,rhs', [([40, 40, 40], 9), ([96, 96, 96], 3), ([128, 128, 135], 2), ([192, 192, 128], 2),
                                   ([288, 288, 160], 2)])
def test_single_rhs_equals_batch(n, rhs):
    ri, p = _params(n, 6)
    s = FORWARD_SOLVER_CONVERGENT_BORN(p)
    s.set_RI(bead_ri(ri, 12, 1.42, 1.336))
    u = incident_plane_waves(ri, rhs, 1.2, 0.532, 1.336, [0.1] * 3).astype(np.complex64)
    both = s.solve_incident(u)
    one = np.concatenate([s.solve_incident(u[..., j:j + 1]) for j in range(rhs)], axis=-1)
    s.close()
    # same operations on every element: at most the compiler's choice of fused multiply-adds differs
    assert np.linalg.norm(both - one) <= 3e-7 * np.linalg.norm(one)


@pytest.mark.parametrize('n', [[40, 40, 40], [96, 96, 96]])
def test_single_rhs_oracle(n):
    ri, p = _params(n, 6)
    s = FORWARD_SOLVER_CONVERGENT_BORN(p)
    RI = bead_ri(ri, 12, 1.42, 1.336)
    s.set_RI(RI)
    u = incident_plane_waves(ri, 1, 1.2, 0.532, 1.336, [0.1] * 3).astype(np.complex128)
    got = s.solve_incident(u)[..., 0]
    s.close()
    o = Oracle(p, io_kernels=False)
    o.set_RI(RI)
    ref = o.born_loop(u[..., 0])
    assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)
