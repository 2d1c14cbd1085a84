"""GPU: the matrix-core line transforms (fft_dense.hip) at the edges of their plans: lengths below
16, one element under, at and over the 16-row and 64-element steps, primes, every butterfly
(2 .. 8, 11, 13), squares of primes and the longest length, as the contiguous (x) and the strided
(y) lines of cbs_field_pupil against NumPy in FP64 with a random pupil, which tells every
frequency apart; and the Born loop that fuses them with the update and the Green's multiply, on
such lengths as x and z axes, scalar and vector.

Tolerance: a transform of n points is a sum of n / 2 products in 32 bits, rounded once a product:
relative error below 2^-24 sqrt(n / 2), 9e-7 at 448; four transforms and their butterflies are
held to 4e-6."""
import ctypes as C

import numpy as np
import pytest

from helpers import params, rel, random_field, sphere_ri

pytestmark = pytest.mark.gpu

LENGTHS = [2, 3, 7, 13, 15, 17, 22, 31, 33, 34, 61, 63, 65, 77, 97, 98, 121, 127, 129, 143, 169, 183, 191, 193, 208,
           255, 257, 301, 319, 321, 383, 385, 407, 443, 448]


@pytest.mark.parametrize('fx,fy', list(zip(LENGTHS, LENGTHS[::-1])))
def test_lengths_against_numpy(fx, fy):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, _lib
    nf = 3
    x = random_field((fx, fy, nf), fx + fy).astype(np.complex64)
    P = np.random.default_rng(fx * 1000 + fy).random((fx, fy)).astype(np.float32)
    s = FORWARD_SOLVER_CONVERGENT_BORN(params((fx, fy, 8), iterations=2))
    out = np.empty((fx, fy, nf), np.complex64, order='F')
    xf, Pf = np.asfortranarray(x), np.asfortranarray(P)
    vp = lambda a: a.ctypes.data_as(C.c_void_p)
    _lib.check(_lib.lib.cbs_field_pupil(s._h, vp(xf), C.c_void_p(None), nf, vp(Pf), vp(out), _lib.CBS_MEM_HOST))
    s.close()
    ax = (0, 1)
    F = np.fft.fftshift(np.fft.fft2(np.fft.ifftshift(x.astype(np.complex128), axes=ax), axes=ax), axes=ax)
    ref = np.fft.fftshift(np.fft.ifft2(np.fft.ifftshift(F * P[:, :, None], axes=ax), axes=ax), axes=ax)
    assert rel(out, ref) < 4e-6


@pytest.mark.parametrize('fixed', [False, True])
@pytest.mark.parametrize('ri,bt_px,vector', [((23, 20, 25), 3, False), ((41, 12, 55), 3, False), ((57, 57, 13), 2, True),
                                             ((89, 14, 7), 4, False), ((9, 30, 121), 3, True)])
def test_born_loop(ri, bt_px, vector, fixed):
    """fixed: the transforms of CBS_TRANSFORMS_FIXED, set before or after the potential."""
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, _lib
    from oracle.cbs import ForwardSolverConvergentBorn as Oracle
    p = params(ri, bt_px_target=bt_px, iterations=7, vector_simulation=vector)
    RI = sphere_ri(ri, 0.3 * min(ri) * 0.1, n_s=1.42)
    u = [random_field(ri + ((3,) if vector else ()), 3 + a) for a in range(3)]
    s = FORWARD_SOLVER_CONVERGENT_BORN(p)
    if fixed and vector:
        _lib.check(_lib.lib.cbs_set_transforms(s._h, _lib.CBS_TRANSFORMS_FIXED))
    s.set_RI(RI)
    if fixed and not vector:
        s.solve_incident(np.stack(u, axis=-1))
        _lib.check(_lib.lib.cbs_set_transforms(s._h, _lib.CBS_TRANSFORMS_FIXED))
        s.set_RI(RI)                     # the shift state of an odd iteration count starts over
    assert _lib.lib.cbs_set_transforms(s._h, 2) == _lib.CBS_ERR_ARG
    got = s.solve_incident(np.stack(u, axis=-1))
    s.close()
    o = Oracle(p, io_kernels=False)
    o.set_RI(RI)
    for a in range(3):
        assert rel(got[..., a], o.born_loop(u[a])) < (1e-5 if fixed else 4e-6)
