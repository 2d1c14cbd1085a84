"""GPU: matrix-core line transforms whose kernels few lengths take: 170, 185 and 190 points (ten tasks a tile, two a
wave) and 396, 402, 438 and 444 (18 tasks, three a wave), and x lines above 192 points in the pass that fuses them with
the update.

Tolerance as in test_gpu_dense_lines: a transform of n points is a sum of n / 2 products in 32 bits, rounded once a
product (2^-24 sqrt(n / 2), 9e-7 at 448); four transforms and their butterflies are held to 4e-6."""
import ctypes as C

import numpy as np
import pytest

from helpers import params, rel, random_field, sphere_ri

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('fx,fy', [(170, 396), (444, 185), (190, 402), (438, 170)])
def test_lengths_against_numpy(fx, fy):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, _lib
    nf = 2
    x = np.asfortranarray(random_field((fx, fy, nf), fx + fy).astype(np.complex64))
    P = np.asfortranarray(np.random.default_rng(fx * 1000 + fy).random((fx, fy)).astype(np.float32))
    s = FORWARD_SOLVER_CONVERGENT_BORN(params((fx, fy, 8), iterations=2))
    out = np.empty((fx, fy, nf), np.complex64, order='F')
    vp = lambda a: a.ctypes.data_as(C.c_void_p)
    _lib.check(_lib.lib.cbs_field_pupil(s._h, vp(x), C.c_void_p(None), nf, vp(P), vp(out), _lib.CBS_MEM_HOST))
    s.close()
    ax = (0, 1)
    F = np.fft.fftshift(np.fft.fft2(np.fft.ifftshift(x.astype(np.complex128), axes=ax), axes=ax), axes=ax)
    ref = np.fft.fftshift(np.fft.ifft2(np.fft.ifftshift(F * P[:, :, None], axes=ax), axes=ax), axes=ax)
    assert rel(out, ref) < 4e-6


# RI grids: 8 voxels of boundary come on top.  x of 257, 337, 443 and 444, z of 170, 190 and 402 points
@pytest.mark.parametrize('ri,vector', [((249, 5, 9), False), ((329, 4, 6), False), ((435, 6, 162), False),
                                       ((436, 5, 7), True), ((9, 5, 182), True), ((11, 4, 394), False)])
def test_born_loop(ri, vector):
    from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN
    from oracle.cbs import ForwardSolverConvergentBorn as Oracle
    p = params(ri, bt_px_target=4, iterations=7, vector_simulation=vector)
    RI = sphere_ri(ri, 0.2, n_s=1.42)
    u = [random_field(ri + ((3,) if vector else ()), 3 + a) for a in range(3)]
    s = FORWARD_SOLVER_CONVERGENT_BORN(p)
    s.set_RI(RI)
    got = s.solve_incident(np.stack(u, axis=-1))
    assert s.plan()['form'] == 'plain'
    s.close()
    o = Oracle(p, io_kernels=False)
    o.set_RI(RI)
    for a in range(3):
        assert rel(got[..., a], o.born_loop(u[a])) < 4e-6
