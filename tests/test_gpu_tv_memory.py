"""GPU: device memory of the TV step.  A handle keeps what a problem's own element type needs (host data: its input and
three dual iterates, or four where iterations go two to a launch), and where the fourth does not fit the step runs
without it."""
import numpy as np
import pytest

from helpers import MB, params, take_memory

pytestmark = pytest.mark.gpu

DIMS = (200, 190, 110)
N = 200 * 190 * 110


def _problem(cplx):
    rng = np.random.default_rng(3)
    x = (rng.standard_normal(DIMS) * 0.05).astype(np.float32).astype(np.float64)
    return x + 1j * (rng.standard_normal(DIMS) * 0.02).astype(np.float32).astype(np.float64) if cplx else x


def _step(s, x, inner):
    from inverse_solver_amd.tv import tv_fista_inner_device
    return tv_fista_inner_device(s, x, 0.02, -0.03, 0.04, np.nan if np.iscomplexobj(x) else 0, True, False, inner)


def _solver():
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    return FORWARD_SOLVER_CONVERGENT_BORN(params((16, 16, 17), iterations=4))


# bytes a voxel: the input and 9 or 12 values of the element type
@pytest.mark.parametrize('cplx,inner,size', [(False, 2, 40), (False, 6, 52), (True, 2, 80), (True, 6, 104)])
def test_workspace(cplx, inner, size):
    from inverse_solver_amd import device as dv
    x = _problem(cplx)
    s = _solver()
    _step(s, x[:8, :8, :8], 3)                      # modules and streams are there
    before = dv.mem_info()[0]
    _step(s, x, inner)
    used = before - dv.mem_info()[0]
    s.close()
    assert used <= size * N + 8 * MB, used / N      # allocations are rounded up to 2 MB


def test_fourth_iterate_does_not_fit():
    from inverse_solver_amd import device as dv
    x = _problem(True)
    s = _solver()
    ref = _step(s, x, 6)                            # 104 bytes a voxel
    s.close()
    s = _solver()
    _step(s, x[:8, :8, :8], 3)
    hold = take_memory(92 * N)                      # 80 are needed with three iterates
    try:
        if dv.mem_info()[0] > 100 * N:
            pytest.skip('device memory could not be taken')
        got = _step(s, x, 6)
    finally:
        for b in hold:
            b.free()
    s.close()
    # the two kernels round alike but for the compiler's choice of fused multiply-adds: 2^-24 of the input a
    # value and iteration
    assert np.linalg.norm(got - ref) <= 6 * 2.0 ** -24 * np.linalg.norm(x)
