"""GPU: the fused form's split of y and x tile on grids where one rule gives way to another, and the kernel variants of
few-block launches: every variant of one split gives the same bits."""
import numpy as np
import pytest

from helpers import params, random_field, rel

pytestmark = pytest.mark.gpu


def _solver(n, iterations=5, **options):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    ri = tuple(m - 8 for m in n)
    s = FORWARD_SOLVER_CONVERGENT_BORN(params(ri, iterations=iterations), options=options)
    RI = np.full(ri, 1.336)
    RI[ri[0] // 3:, ri[1] // 4:, ri[2] // 2:] = 1.40
    s.set_RI(RI)
    return s, ri, RI


# (grid, split, x tile): the largest of the small planes with b = 1 and the ones that leave it; b = 4 and its two ways
# out; the tile for b = 1, b = 2 and above, where 8 divides nx and 16 does not
@pytest.mark.parametrize('n,a,t', [([32, 32, 32], 32, 16), ([24, 24, 96], 24, 16), ([32, 32, 40], 16, 16),
                                   ([40, 40, 40], 20, 8), ([96, 96, 96], 24, 16), ([128, 128, 135], 32, 16),
                                   ([160, 80, 96], 40, 32), ([160, 80, 128], 20, 16), ([192, 96, 96], 48, 32),
                                   ([160, 160, 160], 40, 16), ([40, 20, 320], 20, 16), ([40, 20, 24], 20, 16),
                                   ([24, 96, 160], 24, 16), ([96, 216, 160], 24, 8)])
def test_split_and_tile(n, a, t):
    s, _, _ = _solver(n, 2)
    plan = s.plan()
    s.close()
    assert (plan['form'], plan['a'], plan['tile_t']) == ('fused', a, t)


# one rhs takes other real-space or k-space variants than the batch: 448, 576 and 512 threads; k-space tiles of 4, 8
# and 16 on 192 to 1024 threads; 160 x 80 x 128 keeps its wide tile
@pytest.mark.parametrize('n,batch', [([40, 40, 40], 24), ([96, 96, 96], 8), ([96, 48, 40], 24), ([24, 96, 160], 24),
                                     ([24, 216, 160], 16), ([160, 80, 128], 6), ([128, 64, 96], 12)])
def test_variants_give_the_same_bits(n, batch):
    s, ri, RI = _solver(n)
    u = np.stack([random_field(ri, a) for a in range(3)], axis=-1).astype(np.complex64)
    wide = np.concatenate([u] + [u[..., :1]] * (batch - 3), axis=-1)
    ref = s.solve_incident(wide)[..., :3]
    s.set_RI(RI)                              # the shift state of an odd series starts over
    few = s.solve_incident(u)
    s.set_RI(RI)
    one = s.solve_incident(u[..., 0])
    plan = s.plan()
    s.close()
    np.testing.assert_array_equal(few, ref)
    np.testing.assert_array_equal(one, ref[..., 0])
    f, _, _ = _solver(n, split_a=plan['a'], tile_t=plan['tile_t'])     # no other k-space tile
    got = f.solve_incident(u[..., 0])
    f.close()
    np.testing.assert_array_equal(got, ref[..., 0])


# the grids of test_gpu_few_blocks whose single right-hand side runs the batch's own kernels
@pytest.mark.parametrize('n', [[128, 128, 135], [192, 192, 128], [288, 288, 160]])
def test_single_rhs_oracle(n):
    from oracle.cbs import ForwardSolverConvergentBorn as Oracle
    s, ri, RI = _solver(n, 3)
    u = random_field(ri, 2)
    got = s.solve_incident(u)
    s.close()
    o = Oracle(params(ri, iterations=3), io_kernels=False, workers=16)
    o.set_RI(RI)
    assert rel(got, o.born_loop(u)) < 1e-5
