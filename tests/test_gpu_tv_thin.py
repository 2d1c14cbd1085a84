"""GPU: TV iterations on thin grids, whose blocks hold other columns than 62 x 6 (2 x 126, 6 x 62, 14 x 30, 30 x 14 and
126 x 2), one iteration and two a launch, with tiles that end inside a block, bounds and Dirichlet faces, against
TV_FISTA_inner_v2 in FP64.

Tolerance as in test_gpu_tv_tiles: three times 4 x 2^-24 of the input's norm an iteration."""
import numpy as np
import pytest

from helpers import params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dims', [(1, 500, 17), (2, 253, 4), (3, 130, 7), (6, 125, 5), (13, 95, 8), (26, 148, 11),
                                  (30, 29, 10), (500, 1, 13), (253, 2, 4), (500, 3, 3), (1, 1, 900)])
@pytest.mark.parametrize('cplx', [False, True])
def test_thin_grids(dims, cplx):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    from inverse_solver_amd.tv import tv_fista_inner_device
    from oracle.backward import tv_fista_inner_v2
    rng = np.random.default_rng(sum(dims))
    x = (rng.standard_normal(dims) * 0.05).astype(np.float32).astype(np.float64)
    if cplx:
        x = x + 1j * (rng.standard_normal(dims) * 0.02).astype(np.float32).astype(np.float64)
    s = FORWARD_SOLVER_CONVERGENT_BORN(params((16, 16, 17), iterations=4))
    for inner, nn, dirichlet in ((1, False, False), (2, True, False), (4, False, True), (5, True, False)):
        args = (0.02, -0.03, 0.04, np.nan if cplx else 0, nn, dirichlet, inner)
        got = tv_fista_inner_device(s, x, *args)
        ref = tv_fista_inner_v2(x, *args)
        assert np.linalg.norm(got - ref) <= inner * 3 * 4 * 2.0 ** -24 * np.linalg.norm(x), (inner, nn, dirichlet)
    s.close()
