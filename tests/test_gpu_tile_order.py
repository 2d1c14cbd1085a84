"""GPU: the order of the strided line transforms' tiles, which depends on the row length (whole 128 or 512 bytes or neither) and on
the batch's size (16, 96 and 256 MiB): every tile is transformed once in each, on compiled, matrix-core, Bluestein and run-time
lines, scalar and vector."""
import numpy as np
import pytest

from helpers import params, rel, random_field, sphere_ri

pytestmark = pytest.mark.gpu


def _solver(ri, fixed, vector=False, **kw):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, _lib
    s = FORWARD_SOLVER_CONVERGENT_BORN(params(ri, vector_simulation=vector, **kw))
    if fixed:
        _lib.check(_lib.lib.cbs_set_transforms(s._h, _lib.CBS_TRANSFORMS_FIXED))
    return s


# simulation grids of 64 x 20 x 27, 64 x 23 x 29, 128 x 21 x 22 and, in the other order, 65 x 23 x 29 and 80 x 20 x 27
@pytest.mark.parametrize('ri', [(56, 12, 19), (56, 15, 21), (120, 13, 14), (57, 15, 21), (72, 12, 19)])
@pytest.mark.parametrize('fixed', [False, True])
@pytest.mark.parametrize('vector', [False, True])
def test_small_batches(ri, fixed, vector):
    from oracle.cbs import ForwardSolverConvergentBorn as Oracle
    s = _solver(ri, fixed, vector, iterations=5)
    RI = sphere_ri(ri, 0.4, n_s=1.42)
    u = [random_field(ri + ((3,) if vector else ()), a) for a in range(2)]
    s.set_RI(RI)
    got = s.solve_incident(np.stack(u, axis=-1))
    assert s.plan()['form'] == 'plain'
    s.close()
    o = Oracle(params(ri, vector_simulation=vector, iterations=5), io_kernels=False)
    o.set_RI(RI)
    for a in range(2):
        assert rel(got[..., a], o.born_loop(u[a])) < 1e-5


@pytest.mark.parametrize('fixed', [False, True])
def test_batches_across_the_orders(fixed):
    """64 x 125 x 121: 2 rhs are 15 MiB, 12 are 89, 32 are 236 and 35 are 258, tiles in one and the other order in turn: a
    rhs has the same bits in each."""
    ri = (56, 117, 113)
    s = _solver(ri, fixed, iterations=4)
    s.set_RI(sphere_ri(ri, 2.0, n_s=1.42))
    u = np.stack([random_field(ri, a) for a in range(5)] * 7, axis=-1).astype(np.complex64)
    large = s.solve_incident(u)
    for n in (32, 12, 2):
        np.testing.assert_array_equal(s.solve_incident(u[..., :n]), large[..., :n])
    s.close()
    np.testing.assert_array_equal(large[..., 5:10], large[..., :5])
