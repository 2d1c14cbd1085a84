"""GPU: the phase integration kernels bit for bit against the oracle at the edges of their chunks
(rows: 16 rows and 64 columns a wave; column: 512 steps), and one step of it over the whole range of
arguments: within a few units in the last place of the multiples of 2 pi and of pi, at the bound of
its fast remainder, above it, infinite and NaN."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _integrate(p, s1, s2):
    from inverse_solver_amd import _lib
    p, s1, s2 = (np.asfortranarray(a) for a in (p.astype(np.float32), s1.astype(np.int32), s2.astype(np.int32)))
    out = np.empty_like(p, order='F')
    dims = (C.c_uint32 * 3)(*p.shape)
    vp = lambda a: a.ctypes.data_as(C.c_void_p)
    _lib.check(_lib.lib.cbs_phase_integrate(0, vp(p), vp(s1), vp(s2), vp(out), dims, _lib.CBS_MEM_HOST))
    return out


@pytest.mark.parametrize('n1,n2,n3', [(1, 1, 1), (2, 513, 1), (64, 3, 5), (65, 17, 1), (66, 16, 2), (129, 15, 1),
                                      (130, 514, 1), (3, 1025, 2)])
def test_chunks(n1, n2, n3):
    from oracle.rytov import raster_unwrap
    rng = np.random.default_rng(n1 * n2)
    p = rng.uniform(-np.pi, np.pi, (n1, n2, n3)).astype(np.float32)
    s1, s2 = rng.integers(-1, 2, (n1, n2, n3)), rng.integers(-1, 2, (n2, n3))
    np.testing.assert_array_equal(_integrate(p, s1, s2), raster_unwrap(p, s1, s2))


def test_one_step_over_the_range():
    from oracle.rytov import raster_unwrap
    rng = np.random.default_rng(3)
    two_pi = np.float32(2.0) * np.float32(3.141592654)
    k = np.concatenate([np.arange(-5000, 5000), rng.integers(-10 ** 6, 10 ** 6, 2000)])
    near = (k * np.float64(two_pi) / 2).astype(np.float32)
    near = np.concatenate([near] + [(near.view(np.int32) + d).view(np.float32) for d in (-3, -2, -1, 1, 2, 3)])
    v = np.concatenate([rng.uniform(-20, 20, 50000), rng.uniform(-3e4, 3e4, 50000), near, [0.0, -0.0, 1e-30, -1e-30],
                        4096 * two_pi * (1 + 1e-7 * np.arange(-5, 6)), [1e9, -1e9, np.inf, -np.inf, np.nan]])
    p = np.zeros((2, 1, v.size), np.float32)
    p[1, 0] = v.astype(np.float32)
    zero = np.zeros((2, 1, v.size), np.int32)
    with np.errstate(invalid='ignore'):
        ref = raster_unwrap(p, zero, zero[0])
    np.testing.assert_array_equal(_integrate(p, zero, zero[0]), ref)
