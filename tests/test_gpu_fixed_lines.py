"""GPU: Bluestein's transform and the run-time stages at lengths that the default handle transforms on the matrix cores,
which a handle with CBS_TRANSFORMS_FIXED (both solvers of every BACKWARD_SOLVER_MULTI) keeps: every compiled convolution
length and every stage radix as x and y lines, the convergence stop and the deferred increment's flush of the fused
passes, and the loops and 2D solves of the arbitrary-grid tests, with those tests' own oracles and tolerances."""
import numpy as np
import pytest

import test_gpu_anygrid as anygrid
import test_gpu_convergence as convergence
import test_gpu_field_pupil as pupil
import test_gpu_grid_sweep as sweep
from helpers import params

pytestmark = pytest.mark.gpu


def _fix(s):
    from inverse_solver_amd import _lib
    _lib.check(_lib.lib.cbs_set_transforms(s._h, _lib.CBS_TRANSFORMS_FIXED))


@pytest.fixture(autouse=True)
def fixed_handles(monkeypatch):
    """Every handle of a test is a fixed one."""
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN as S
    init = S.__init__

    def fixed_init(self, *args, **kw):
        init(self, *args, **kw)
        _fix(self)

    monkeypatch.setattr(S, '__init__', fixed_init)


# primes up to half of each compiled convolution length (48 ... 1296), the longest line first where it is prime; then
# lengths of run-time stages: 7, 11, 13, 9, 3 and 5 with powers of two from 2 to 16
BLUESTEIN = [19, 23, 31, 37, 47, 61, 79, 89, 127, 157, 191, 251, 317, 383, 509, 571, 647]
STAGES = [7, 14, 28, 56, 112, 11, 13, 49, 77, 143, 169, 63, 105, 126, 208, 364, 441]


@pytest.mark.parametrize('fx,fy', list(zip(BLUESTEIN, STAGES[::-1])) + list(zip(STAGES[::3], BLUESTEIN[::3])))
def test_lines_match_numpy(fx, fy):
    pupil.test_field_pupil_matches_numpy(fx, fy)


@pytest.mark.parametrize('even', [True, False])
@pytest.mark.parametrize('ri,bt_px', [((9, 9, 9), 7), ((28, 9, 13), 7)])   # 23^3: Bluestein; 42 x 23 x 27: stages and
def test_stop_iteration(ri, bt_px, even):                                  # Bluestein and a compiled length
    plan = convergence._stop_case(convergence._setup(ri, radius=0.4, bt_px_target=bt_px), None, even)
    assert plan['form'] == 'plain'


@pytest.mark.parametrize('ri,bt_px', [((34, 36, 44), 4), ((81, 60, 41), 8), ((30, 22, 20), 3), ((100, 120, 56), 8)])
def test_born_loop(ri, bt_px):
    anygrid.test_born_loop_any_grid(ri, bt_px)


@pytest.mark.parametrize('ri,bt_px', sweep._cases())
def test_random_grid(ri, bt_px):
    sweep.test_random_grid_matches_oracle(ri, bt_px)


def test_2d_solve_of_prime_lengths():
    anygrid.test_reference_demo_forward_geometry_2d_solve()


def test_switch_after_a_2d_solve():
    """The convolution grid's and the field grid's transforms follow a switch between two solves."""
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, _lib
    from inverse_solver_amd.phantoms import bead_ri, circle_illumination
    ri = (17, 19, 12)
    p = params(ri, iterations=6)
    RI = bead_ri(ri, 5, 1.46, 1.336)
    u = circle_illumination(ri[:2], 2, 1.2, 0.532, [0.1] * 3)
    s, t = FORWARD_SOLVER_CONVERGENT_BORN(p), FORWARD_SOLVER_CONVERGENT_BORN(p)
    s.set_RI(RI)
    ref = s.solve(u)
    _lib.check(_lib.lib.cbs_set_transforms(t._h, _lib.CBS_TRANSFORMS_FASTEST))
    t.set_RI(RI)
    t.solve(u)
    _fix(t)
    got = t.solve(u)
    s.close()
    t.close()
    for a, b in zip(got, ref):
        np.testing.assert_array_equal(a, b)
