"""GPU: the fused TV iteration (tv_inner) at the edges of its 62 x 6 column tiles and of its runs
of three planes, on grids smaller than a tile, with zero, one and several iterations, bounds and
Dirichlet faces, against TV_FISTA_inner_v2 in FP64.

Tolerance: an iteration rounds y and its products a few times (4 x 2^-24 of the input); div and
grad / (12 lam) together are non-expansive and the momentum at most triples a difference, so five
iterations stay within 5 x 3 x 4 x 2^-24 = 3.6e-6 of the input's norm."""
import numpy as np
import pytest

from helpers import params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dims', [(1, 1, 1), (2, 3, 1), (61, 5, 3), (62, 6, 2), (63, 7, 4), (124, 12, 6), (125, 13, 7)])
@pytest.mark.parametrize('cplx', [False, True])
def test_tv_tiles(dims, cplx):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    from inverse_solver_amd.tv import tv_fista_inner_device
    from oracle.backward import tv_fista_inner_v2
    rng = np.random.default_rng(sum(dims))
    x = (rng.standard_normal(dims) * 0.05).astype(np.float32).astype(np.float64)
    if cplx:
        x = x + 1j * (rng.standard_normal(dims) * 0.02).astype(np.float32).astype(np.float64)
    s = FORWARD_SOLVER_CONVERGENT_BORN(params((16, 16, 17), iterations=4))
    for inner, nn, dirichlet in ((0, False, False), (1, False, False), (2, True, False), (5, False, True)):
        args = (0.02, -0.03, 0.04, np.nan if cplx else 0, nn, dirichlet, inner)
        got = tv_fista_inner_device(s, x, *args)
        ref = tv_fista_inner_v2(x, *args)
        assert np.linalg.norm(got - ref) <= 3.6e-6 * np.linalg.norm(x), (inner, nn, dirichlet)
    s.close()
