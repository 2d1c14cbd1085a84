"""GPU: two TV iterations a launch (tv_inner2) on grids whose last tile is short in x, in y and in z, real and complex
(which requests its operands one plane ahead instead of two), against TV_FISTA_inner_v2 in FP64.  The tiles that
tv_tiles gives them, columns by columns by planes: 54 x 9 x 16 (complex) and 7 (real) on 161 x 161 x 61, 51 x 9 x 7 on
101 x 91 x 71, 41 x 12 x 9 and 4 on 121 x 95 x 83, 46 x 11 x 11 and 5 on 181 x 61 x 101.

Tolerance as in test_gpu_tv_pairs: three times 4 x 2^-24 of the input's norm an iteration."""
import numpy as np
import pytest

from helpers import params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dims', [(161, 161, 61), (101, 91, 71), (121, 95, 83), (181, 61, 101)])
@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('inner,nn,dirichlet', [(5, True, False), (6, False, True)])
def test_ragged_tiles(dims, cplx, inner, nn, dirichlet):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    from inverse_solver_amd.tv import tv_fista_inner_device
    from oracle.backward import tv_fista_inner_v2
    rng = np.random.default_rng(sum(dims))
    x = (rng.standard_normal(dims) * 0.05).astype(np.float32).astype(np.float64)
    if cplx:
        x = x + 1j * (rng.standard_normal(dims) * 0.02).astype(np.float32).astype(np.float64)
    s = FORWARD_SOLVER_CONVERGENT_BORN(params((16, 16, 17), iterations=4))
    args = (0.02, -0.03, 0.04, np.nan if cplx else 0, nn, dirichlet, inner)
    got = tv_fista_inner_device(s, x, *args)
    s.close()
    err = np.abs(got - tv_fista_inner_v2(x, *args))
    assert np.linalg.norm(err) <= inner * 3 * 4 * 2.0 ** -24 * np.linalg.norm(x)
    # a tile that is off in one column would hide in the norm: no value is off by a thousandth of the input's spread
    assert err.max() <= 1e-3 * 0.05
