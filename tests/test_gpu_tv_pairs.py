"""GPU: two TV iterations a launch (tv_inner2) at the edges of its column tiles (60 wide, what 768 threads hold
in y) and of its runs of planes, with an odd and an even number of them, bounds and Dirichlet faces, against
TV_FISTA_inner_v2 in FP64.

Tolerance: an iteration rounds y and its products a few times (4 x 2^-24 of the input); div and
grad / (12 lam) together are non-expansive and the momentum at most triples a difference, so six
iterations stay within 6 x 3 x 4 x 2^-24 = 4.3e-6 of the input's norm."""
import numpy as np
import pytest

from helpers import params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dims', [(1, 1, 1), (1, 2, 7), (5, 80, 3), (60, 8, 5), (61, 9, 16), (60, 16, 33),
                                  (121, 45, 40), (100, 90, 70)])
@pytest.mark.parametrize('cplx', [False, True])
def test_tv_pairs(dims, cplx):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    from inverse_solver_amd.tv import tv_fista_inner_device
    from oracle.backward import tv_fista_inner_v2
    rng = np.random.default_rng(sum(dims))
    x = (rng.standard_normal(dims) * 0.05).astype(np.float32).astype(np.float64)
    if cplx:
        x = x + 1j * (rng.standard_normal(dims) * 0.02).astype(np.float32).astype(np.float64)
    s = FORWARD_SOLVER_CONVERGENT_BORN(params((16, 16, 17), iterations=4))
    for inner, nn, dirichlet in ((3, False, False), (4, True, False), (5, False, True), (6, True, True)):
        args = (0.02, -0.03, 0.04, np.nan if cplx else 0, nn, dirichlet, inner)
        got = tv_fista_inner_device(s, x, *args)
        ref = tv_fista_inner_v2(x, *args)
        assert np.linalg.norm(got - ref) <= 4.3e-6 * np.linalg.norm(x), (inner, nn, dirichlet)
    s.close()
