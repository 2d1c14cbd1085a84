"""Performance cases: the work a program that uses this package has it do.

Six kinds of call, through the package's public entry points (the class API and the C ABI
of include/cbs_hip.h on device buffers):

  loop      the Born loop of a batch of incident 3D fields (solve_incident_device), scalar
            or vector, on any simulation grid, with or without the convergence test
  dropin    set_RI and solve() of the class API, host arrays in and out, 2D fields
  field     cbs_solve_field: 2D fields in, transmitted, reflected and 3D fields out, all on
            the device
  gradient  get_gradiant_static of the reconstruction: forward solve, residual, adjoint solve
  tv        the TV proximal step of the reconstruction, real or complex potential
  unwrap    Goldstein phase unwrapping of the measured angles (the Rytov start)

Lengths are in micrometres, sizes in voxels.  Inputs come from the seed alone; ``exact``
restates each call in 64 bits with plain torch.
"""
import ctypes as C
import math

import numpy as np
import torch

from inverse_solver_amd import FORWARD_SOLVER_CONVERGENT_BORN, get_default_parameters
from inverse_solver_amd import _lib
from inverse_solver_amd.backward_solver import BACKWARD_SOLVER_MULTI
from inverse_solver_amd.backward_solver import get_default_parameters as backward_defaults
from inverse_solver_amd.rytov import unwrap_phase

LAM, N_M, NA = 0.532, 1.336, 1.2


def listed():
    return [
        # one illumination of a small bead, the smallest call: launches and latency
        dict(name='loop 40^3 x 1', kind='loop', x=32, y=32, z=32, bx=4, by=4, bz=4, angles=1, comps=1, dx=0.1,
             nmax=1.46, iters=0, absorbing=False, tol=0.0),
        # the drop-in class call of a MATLAB user: one plane wave through a bead, 2D in and out
        dict(name='dropin 96^3 x 1', kind='dropin', x=64, y=64, z=64, b=16, angles=1, iters=100, nmax=1.46),
        # TV step of a reconstruction with a real potential
        dict(name='tv real 96x96x97', kind='tv', x=96, y=96, z=97, cplx=False, inner=100, bounds=True),
        # the same with the reference's defaults, which keep the imaginary part
        dict(name='tv complex 161x161x61', kind='tv', x=161, y=161, z=61, cplx=True, inner=100, bounds=False),
        # phase maps of one tomogram, noisy enough to hold residues
        dict(name='unwrap 96^2 x 24', kind='unwrap', x=96, y=96, angles=24, noise=0.6),
        # one gradient of a tomographic reconstruction
        dict(name='gradient 96x96x97 x 24', kind='gradient', x=96, y=96, z=97, b=16, bz=19, angles=24, nmax=1.42),
        # every angle of a tomogram in one batch, the throughput case
        dict(name='loop 160^3 x 49', kind='loop', x=128, y=128, z=128, bx=16, by=16, bz=16, angles=49, comps=1,
             dx=0.1, nmax=1.48, iters=0, absorbing=False, tol=0.0),
        # a grid as a user's sample and boundary give it: 183 = 3 x 61 twice, and the prime 83
        dict(name='loop 183x183x83 x 12', kind='loop', x=161, y=161, z=61, bx=11, by=11, bz=11, angles=12, comps=1,
             dx=0.1108, nmax=1.46, iters=0, absorbing=False, tol=0.0),
        # a smooth grid that no kernel was tuned for, an absorbing sample
        dict(name='loop 100x120x75 x 12', kind='loop', x=84, y=104, z=59, bx=8, by=8, bz=8, angles=12, comps=1,
             dx=0.1, nmax=1.46, iters=0, absorbing=True, tol=0.0),
        # vector fields (the dyadic Green's function)
        dict(name='loop vector 160^3 x 8', kind='loop', x=128, y=128, z=128, bx=16, by=16, bz=16, angles=8, comps=3,
             dx=0.1, nmax=1.46, iters=0, absorbing=False, tol=0.0),
        # a cell-sized volume with the convergence test, the largest call
        dict(name='loop 576x576x320 x 4', kind='loop', x=512, y=512, z=256, bx=32, by=32, bz=32, angles=4, comps=1,
             dx=0.1, nmax=1.40, iters=0, absorbing=False, tol=1e-3),
        # a batch of 2D fields through the whole solve on the device
        dict(name='field 160^3 x 16', kind='field', x=128, y=128, z=128, b=16, angles=16, nmax=1.46, refl=True),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(['loop'] * 6 + ['tv'] * 2 + ['field', 'field', 'dropin', 'gradient', 'unwrap'])
    if kind == 'loop':
        while True:
            d = [int(round(_log(rng, 24, 320))) for _ in range(3)]
            comps = 3 if rng.random() < 0.2 else 1
            angles = int(round(_log(rng, 1, 49)))
            b = [rng.randint(3, max(3, min(16, n // 4))) for n in d]
            nmax = round(rng.uniform(1.36, 1.48), 3)
            c = dict(kind='loop', x=d[0] - 2 * b[0], y=d[1] - 2 * b[1], z=d[2] - 2 * b[2], bx=b[0], by=b[1], bz=b[2],
                     angles=angles, comps=comps, dx=0.1, nmax=nmax, iters=0, absorbing=rng.random() < 0.3,
                     tol=1e-3 if rng.random() < 0.2 else 0.0)
            if d[0] * d[1] * d[2] * angles * comps * _iterations(c) <= 4e9:
                return c
    if kind == 'tv':
        return dict(kind='tv', x=int(_log(rng, 24, 200)), y=int(_log(rng, 24, 200)), z=int(_log(rng, 15, 120)),
                    cplx=rng.random() < 0.5, inner=rng.randint(20, 100), bounds=rng.random() < 0.5)
    if kind == 'field':
        x = int(_log(rng, 32, 128))
        return dict(kind='field', x=x, y=x + rng.randint(-8, 8), z=int(_log(rng, 24, 128)), b=rng.randint(4, 16),
                    angles=int(_log(rng, 1, 16)), nmax=round(rng.uniform(1.36, 1.48), 3), refl=rng.random() < 0.5)
    if kind == 'dropin':
        x = rng.randint(24, 64)
        return dict(kind='dropin', x=x, y=x + rng.randint(-4, 4), z=rng.randint(24, 64), b=rng.randint(4, 16),
                    angles=rng.randint(1, 4), iters=2 * rng.randint(8, 50), nmax=1.46)
    if kind == 'gradient':
        x = rng.randint(32, 72)
        return dict(kind='gradient', x=x, y=x, z=2 * rng.randint(14, 30) + 1, b=rng.randint(6, 16),
                    bz=rng.randint(6, 16), angles=rng.randint(4, 24), nmax=1.42)
    n = int(_log(rng, 48, 256))
    return dict(kind='unwrap', x=n, y=n, angles=int(_log(rng, 1, 49)), noise=round(rng.uniform(0.1, 0.8), 2))


# ---------------------------------------------------------------- inputs

def _device():
    return torch.device('cuda' if torch.cuda.is_available() else 'cpu')


def _gen(seed):
    return torch.Generator(device='cpu').manual_seed(int(seed))


def _uniform(gen, n, lo, hi):
    return (torch.rand(n, generator=gen, dtype=torch.float64) * (hi - lo) + lo).tolist()


def _boundary(c):
    return [c['bx'], c['by'], c['bz']] if 'bx' in c else [c['b'], c['b'], c.get('bz', c['b'])]


def _params(c, **kw):
    """Solver parameters of a case: boundary_thickness gives the boundary in pixels as the class rounds it."""
    dx = c.get('dx', 0.1)
    unit = dx * 2 * N_M / LAM
    init = dict(size=[c['x'], c['y'], c['z']], wavelength=LAM, NA=NA, RI_bg=N_M, resolution=[dx] * 3,
                vector_simulation=c.get('comps', 1) == 3, iterations_number=c.get('iters', 0) or -1,
                boundary_thickness=[b * unit for b in _boundary(c)])
    init.update(kw)
    return get_default_parameters(init)


def _iterations(c):
    """The default iteration count for the case's size and largest index."""
    if c.get('iters', 0):
        return c['iters']
    dx, k = c.get('dx', 0.1), 2 * math.pi * N_M / LAM
    eps = 1.01 * k * k * (c['nmax'] ** 2 / N_M ** 2 - 1)
    ext = math.sqrt(sum(((n + 2 * b) * dx) ** 2 for n, b in zip((c['x'], c['y'], c['z']), _boundary(c))))
    return int(math.ceil(ext / (2 * k / eps) / 2 + 1) * 2)


def _ri(c, seed):
    """Index grid (z, y, x) in FP64: six blurred-edge spheres, the first with the largest index."""
    dev, g = _device(), _gen(seed)
    n = [c['z'], c['y'], c['x']]
    ax = [torch.arange(m, dtype=torch.float64, device=dev).reshape([-1 if j == i else 1 for j in range(3)])
          for i, m in enumerate(n)]
    out = torch.zeros(n, dtype=torch.float64, device=dev)
    for s in range(6):
        r = _uniform(g, 1, 0.12, 0.28)[0] * min(n)
        o = _uniform(g, 3, 0.25, 0.75)
        f = 1.0 if s == 0 else _uniform(g, 1, 0.3, 1.0)[0]
        d = torch.sqrt(sum((ax[i] - o[i] * n[i]) ** 2 for i in range(3)))
        out = torch.maximum(out, f * torch.clamp(r + 0.5 - d, 0, 1))
    ri = N_M + (c['nmax'] - N_M) * out
    return torch.complex(ri, 0.004 * out) if c.get('absorbing') else ri


def _waves(c, seed):
    """Transverse frequencies (cycles per um) of the angles: normal incidence, then a circle at 0.95 NA."""
    g = _gen(seed + 101)
    p0, a = _uniform(g, 1, 0, 2 * math.pi)[0], c['angles']
    k = 0.95 * NA / LAM
    return [(0.0, 0.0) if m == 0 else (k * math.cos(p0 + 2 * math.pi * m / max(1, a - 1)),
                                       k * math.sin(p0 + 2 * math.pi * m / max(1, a - 1))) for m in range(a)], p0


def _incident(c, seed):
    """Plane waves on the RI grid, complex64 [angle][component][z][y][x]; a vector wave is polarised across its
    direction."""
    dev, dx = _device(), c['dx']
    z, y, x = (((torch.arange(m, dtype=torch.float64, device=dev) - m // 2) * dx).reshape(s) for m, s in
               ((c['z'], (-1, 1, 1)), (c['y'], (1, -1, 1)), (c['x'], (1, 1, -1))))
    k0 = N_M / LAM
    out = torch.empty((c['angles'], c['comps'], c['z'], c['y'], c['x']), dtype=torch.complex64, device=dev)
    waves, p0 = _waves(c, seed)
    for m, (kx, ky) in enumerate(waves):
        kz = math.sqrt(k0 * k0 - kx * kx - ky * ky)
        ph = 2 * math.pi * (kx * x + ky * y + kz * z) + p0
        w = torch.complex(torch.cos(ph), torch.sin(ph))
        if c['comps'] == 1:
            out[m, 0] = w
        else:
            e = np.cross([kx, ky, kz], [0.6, 0.8, 0.0])
            for j in range(3):
                out[m, j] = w * float(e[j] / np.linalg.norm(e))
    return out


def _fields_2d(c, seed):
    """Input fields (angle, y, x), complex64: periodic plane waves of the field grid."""
    dx, dev = 0.1, _device()
    y = torch.arange(c['y'], dtype=torch.float64, device=dev).reshape(-1, 1)
    x = torch.arange(c['x'], dtype=torch.float64, device=dev).reshape(1, -1)
    waves, p0 = _waves(c, seed)
    out = []
    for kx, ky in waves:
        ix, iy = round(kx * dx * c['x']), round(ky * dx * c['y'])
        ph = 2 * math.pi * (ix * x / c['x'] + iy * y / c['y']) + p0
        out.append(torch.complex(torch.cos(ph), torch.sin(ph)))
    return torch.stack(out).to(torch.complex64)


def _hump(c, seed, height):
    """A smooth phase bump, (y, x)."""
    g, dev = _gen(seed + 77), _device()
    y = torch.arange(c['y'], dtype=torch.float64, device=dev).reshape(-1, 1) / c['y']
    x = torch.arange(c['x'], dtype=torch.float64, device=dev).reshape(1, -1) / c['x']
    out = 0
    for _ in range(4):
        cy, cx, w, h = (_uniform(g, 1, *r)[0] for r in ((0.3, 0.7), (0.3, 0.7), (0.08, 0.2), (0.4, 1.0)))
        out = out + height * h * torch.exp(-((y - cy) ** 2 + (x - cx) ** 2) / (2 * w * w))
    return out


def _measured(c, seed):
    """Measured fields of the gradient: the input behind a phase object, with 10 % noise."""
    u = _fields_2d(c, seed).to(torch.complex128)
    h = _hump(c, seed, 1.5)
    g = _gen(seed + 5)
    n = torch.view_as_complex(torch.randn(u.shape + (2,), generator=g, dtype=torch.float64)).to(u.device)
    return (u * torch.complex(torch.cos(h), torch.sin(h)) + 0.1 / math.sqrt(2) * n).to(torch.complex64)


def _host(t):
    """(angle, y, x) on the device -> (x, y, 1, angle) on the host, the class API's order."""
    return np.asfortranarray(t.cpu().numpy().transpose(2, 1, 0)[:, :, None, :])


def _ri_host(c, seed):
    return np.asfortranarray(_ri(c, seed).cpu().numpy().transpose(2, 1, 0))


def _tv_input(c, seed):
    ri = _ri(dict(c, nmax=1.42), seed)
    u = ri * ri / (N_M * N_M) - 1
    n = torch.randn((2,) + tuple(u.shape), generator=_gen(seed + 9), dtype=torch.float64).to(u.device)
    if c['cplx']:
        return torch.complex(u + 2e-3 * n[0], 2e-3 * n[1]).to(torch.complex64)
    return (u + 2e-3 * n[0]).to(torch.float32)


_TV_LAM = 1e-3


def _wrapped(c, seed):
    """Wrapped phase maps (x, y, angle) with noise, column-major float32."""
    g, out = _gen(seed + 3), []
    for a in range(c['angles']):
        h = _hump(c, seed + 1000 * a, 7.0).cpu()
        h = h + c['noise'] * torch.randn(h.shape, generator=g, dtype=torch.float64)
        out.append(torch.atan2(torch.sin(h), torch.cos(h)).to(torch.float32).numpy().T)
    return np.asfortranarray(np.stack(out, axis=2))


# ---------------------------------------------------------------- the calls

_KEPT = {}   # solvers of the class API by geometry: a program keeps one and gives it sample after sample


def _kept(c, make):
    key = tuple(sorted((k, v) for k, v in c.items() if k not in ('name', 'nmax')))
    if key not in _KEPT:
        _KEPT[key] = make()
    return _KEPT[key]


def _sync():
    if torch.cuda.is_available():
        torch.cuda.synchronize()


class _Solver(FORWARD_SOLVER_CONVERGENT_BORN):
    """A solver set to one sample, whose RI grid is on the device."""

    def __init__(self, c, seed, **kw):
        super().__init__(_params(c, **kw))
        ri = _ri(c, seed)
        _sync()
        self.set_RI_device(ri.data_ptr(), ri.is_complex())


def prepare(case, seed):
    c = case
    if c['kind'] == 'loop':
        u = _incident(c, seed)
        s = _Solver(c, seed)
        if c['tol']:
            s.set_convergence(c['tol'])
        return dict(c=c, s=s, u=u, out=torch.empty_like(u))
    if c['kind'] == 'dropin':
        s = _kept(c, lambda: FORWARD_SOLVER_CONVERGENT_BORN(_params(c, return_3D=True)))
        return dict(c=c, s=s, ri=_ri_host(c, seed), u=_host(_fields_2d(c, seed)))
    if c['kind'] == 'field':
        s = _Solver(c, seed)
        k = [t.to(torch.complex64).contiguous() for t in _io_kernels(c)]
        pin, pout = (p.to(torch.float32).cpu().contiguous() for p in _pupils(c))
        _sync()
        _lib.check(_lib.lib.cbs_set_io_kernels(s._h, *[C.c_void_p(t.data_ptr()) for t in k], _lib.CBS_MEM_DEVICE))
        u = _fields_2d(c, seed)
        t, f3 = torch.empty_like(u), torch.empty((c['angles'], c['z'], c['y'], c['x']), dtype=u.dtype, device=u.device)
        return dict(c=c, s=s, u=u, pin=pin, pout=pout, t=t, r=torch.empty_like(u) if c['refl'] else None, f3=f3)
    if c['kind'] == 'gradient':
        def make():
            fp = _params(c, return_transmission=True, return_reflection=True, return_3D=True)
            return BACKWARD_SOLVER_MULTI(backward_defaults(dict(forward_solver_parameters=fp, verbose=False)))
        return dict(c=c, s=_kept(c, make), ri=_ri_host(c, seed), u=_host(_fields_2d(c, seed)),
                    y=_host(_measured(c, seed)))
    if c['kind'] == 'tv':
        v = _tv_input(c, seed)
        # the step runs on a solver's handle; a reconstruction has one on the same device
        s = _kept(dict(kind='tv handle'), lambda: FORWARD_SOLVER_CONVERGENT_BORN(
            _params(dict(x=16, y=16, z=16, b=4, nmax=1.4))))
        return dict(c=c, s=s, v=v, out=torch.empty_like(v))
    return dict(c=c, w=_wrapped(c, seed))


def run(state):
    c = state['c']
    if c['kind'] == 'loop':
        state['s'].solve_incident_device(state['u'].data_ptr(), c['angles'], state['out'].data_ptr())
        return state['out']
    if c['kind'] == 'dropin':
        state['s'].set_RI(state['ri'])
        trans, _, f3 = state['s'].solve(state['u'])
        return [trans, f3]
    if c['kind'] == 'field':
        ptr = [C.c_void_p(t.data_ptr()) if t is not None else C.c_void_p(None)
               for t in (state['u'], state['pin'], state['pout'], state['t'], state['r'], state['f3'])]
        _lib.check(_lib.lib.cbs_solve_field(state['s']._h, ptr[0], c['angles'], ptr[1], ptr[2], ptr[3], ptr[4], ptr[5],
                                            _lib.CBS_MEM_DEVICE))
        return [t for t in (state['t'], state['f3'], state['r']) if t is not None]
    if c['kind'] == 'gradient':
        grad, err = state['s'].get_gradiant_static(state['ri'], state['u'], state['y'])
        return [grad, err]
    if c['kind'] == 'tv':
        dims = (C.c_uint32 * 3)(c['x'], c['y'], c['z'])
        a, b = C.c_void_p(state['v'].data_ptr()), C.c_void_p(state['out'].data_ptr())
        lo, hi = (0.0, 0.1) if c['bounds'] else (-math.inf, math.inf)
        if c['cplx']:
            _lib.check(_lib.lib.cbs_tv_prox_complex(state['s']._h, a, b, dims, _TV_LAM, lo, hi, math.nan,
                                                    int(c['bounds']), 0, c['inner'], _lib.CBS_MEM_DEVICE))
        else:
            _lib.check(_lib.lib.cbs_tv_prox(state['s']._h, a, b, dims, _TV_LAM, lo, hi, int(c['bounds']), 0,
                                            c['inner'], _lib.CBS_MEM_DEVICE))
        return state['out']
    return unwrap_phase(state['w'])


def work(case):
    """Bytes and operations of one call.  A Born iteration on a grid of N voxels is a forward and an inverse 3D
    transform (10 N log2 N) and about 60 operations a voxel of pointwise work; its transforms couple every voxel
    with every other one, so the state (8 bytes a voxel) crosses memory twice each way.  Inputs and outputs of the
    call come on top."""
    c = case
    vox = c['x'] * c['y'] * c.get('z', 1)
    if c['kind'] == 'tv':
        size = 8 if c['cplx'] else 4
        return dict(bytes=2.0 * size * vox, flops=(60.0 if c['cplx'] else 30.0) * vox * c['inner'])
    if c['kind'] == 'unwrap':
        return dict(bytes=8.0 * vox * c['angles'], flops=40.0 * vox * c['angles'])
    n = float(np.prod([m + 2 * b for m, b in zip((c['x'], c['y'], c['z']), _boundary(c))]))
    rhs = c['angles'] * c.get('comps', 1) * (2 if c['kind'] == 'gradient' else 1)
    it = _iterations(c)
    bytes_ = rhs * (32.0 * n * it + 16.0 * vox) + 8.0 * n
    flops = rhs * it * n * (10 * math.log2(n) + 60)
    if c['kind'] != 'loop':   # the convolution-grid transforms of every z plane, in and out
        m = 4.0 * c['x'] * c['y']
        flops += rhs * c['z'] * 2 * (5 * m * math.log2(m))
        bytes_ += 8.0 * 3 * m * c['z']
    return dict(bytes=bytes_, flops=flops)


# ---------------------------------------------------------------- 64-bit restatements

def _c2(a, inverse=False):
    """Centred 2D transform over the last two axes."""
    f = torch.fft.ifft2 if inverse else torch.fft.fft2
    return torch.fft.fftshift(f(torch.fft.ifftshift(a, dim=(-2, -1))), dim=(-2, -1))


def _freq(n, dx):
    return (torch.arange(n, dtype=torch.float64, device=_device()) - n // 2) / (dx * n)


def _pupils(c):
    """NA circle times the Abbe factors, (y, x), input and output."""
    k2 = _freq(c['y'], 0.1).reshape(-1, 1) ** 2 + _freq(c['x'], 0.1).reshape(1, -1) ** 2
    na = torch.sqrt(k2) < NA / LAM
    cos = torch.sqrt(torch.clamp((N_M / LAM) ** 2 - k2, min=0)) / (N_M / LAM)
    return (torch.where(na, 1 / torch.sqrt(torch.where(na, cos, torch.ones_like(cos))), torch.zeros_like(cos)),
            torch.where(na, torch.sqrt(cos), torch.zeros_like(cos)))


def _bessel(nu, x):
    """J0 or J1: Bessel's integral by the trapezoidal rule below 25, Hankel's series above (DLMF 10.9.2, 10.17.3)."""
    small, y = torch.zeros_like(x), torch.clamp(x, min=25.0)
    for m in range(64):
        tau = 2 * math.pi * m / 64
        small += torch.cos(nu * tau - torch.clamp(x, max=25.0) * math.sin(tau)) / 64
    P, Q, a = torch.ones_like(y), torch.zeros_like(y), torch.ones_like(y)
    for k in range(1, 20):
        a = a * ((4 * nu * nu - (2 * k - 1) ** 2) / (8.0 * k)) / y
        sign = -1 if k % 4 in (2, 3) else 1
        P, Q = (P, Q + sign * a) if k % 2 else (P + sign * a, Q)
    w = y - (nu / 2 + 0.25) * math.pi
    return torch.where(x < 25.0, small, torch.sqrt(2 / (math.pi * y)) * (torch.cos(w) * P - torch.sin(w) * Q))


def _hankel(samples, crop):
    """Quasi-discrete Hankel transform of order 0 on [0, 1]: radii, frequencies and the two weighted matrices."""
    dev = _device()
    c = math.pi * (torch.arange(1, samples + 2, dtype=torch.float64, device=dev) - 0.25)
    for _ in range(60):
        c = c + torch.clamp(_bessel(0, c) / _bessel(1, c), -0.05, 0.05)
    top, c = c[-1], c[:-1]
    pos = int(torch.argmin(torch.abs(c - c.max() * crop))) + 1
    j1 = torch.abs(_bessel(1, c))
    k, rv, w = 2 * math.pi / top * j1, j1, torch.sqrt(2 / top) / j1
    mat = (w[:pos, None] * w[None, :]) * _bessel(0, c[:pos, None] / top * c[None, :])
    return c / top, c[:pos], mat, k[:pos], rv


def _truncated_green(c, refocus):
    """Axially truncated Green's function (or refocusing kernel), z in real space, (z, ky, kx) centred on the
    convolution grid, as FORWARD_SOLVER_CONVERGENT_BORN's constructor defines it."""
    dev, dx, over = _device(), 0.1, 10
    out = [2 * c['x'], 2 * c['y'], c['z']]
    side = math.ceil((max(out[0], out[1]) * (math.sqrt(2) * 1.1) + over) * dx / dx)
    nz, samples = out[2] + over, 40000
    fx = _freq(side, dx)
    rho = torch.sqrt(fx[:, None] ** 2 + fx[None, :] ** 2)
    fz = _freq(nz, dx)
    k0, kmax = N_M / LAM, NA / LAM
    diag = math.hypot(side, side)
    r, k, mat, kw, rv = _hankel(samples, diag * 2 / (2 * samples))
    H = r / r.max() * rho.max() * 2
    k3 = torch.sqrt(torch.clamp(k0 * k0 - H * H, min=0))
    inside = H < kmax
    fac = (nz - over / 2) / nz
    g = (torch.sinc((k3[:, None] - fz[None, :]) * dx * nz * fac) * fac * inside[:, None]).to(torch.complex128)
    if not refocus:
        g = g / (torch.where(inside, k3, k3 + 1)[:, None] * (1j * 4 * math.pi))
    m = mat.to(torch.complex128)
    img = (m @ (g / rv[:, None])) * kw[:, None]
    t = k / k.max()
    mask = torch.where(t < 0.9, torch.ones_like(t), torch.where((t < 1) & (t > 0.9), (1 - t) * 10,
                                                                torch.zeros_like(t)))
    g = (m.T @ (img * mask[:, None] / kw[:, None])) * rv[:, None]
    lo = torch.clamp(torch.searchsorted(H, rho.reshape(-1)) - 1, 0, samples - 1)
    hi = torch.where(H[lo] < rho.reshape(-1), lo + 1, lo).clamp(max=samples - 1)
    w = torch.where(hi == lo, torch.ones_like(H[lo]), (rho.reshape(-1) - H[lo]) / (H[hi] - H[lo]))
    sx, sy = side // 2 - out[0] // 2, side // 2 - out[1] // 2
    res = torch.empty((nz, out[1], out[0]), dtype=torch.complex128, device=dev)
    for z in range(nz):
        p = ((g[lo, z] * w + g[hi, z] * (1 - w)) * (nz / (dx * dx))).reshape(side, side)
        res[z] = _c2(_c2(p, True)[sy:sy + out[1], sx:sx + out[0]])
    res = torch.fft.fftshift(torch.fft.ifft(torch.fft.ifftshift(res, dim=0), dim=0), dim=0)
    zs = nz // 2 - out[2] // 2
    return res[zs:zs + out[2]]


def _io_kernels(c):
    """Refocusing, transmission and reflection kernels, (z, ky, kx) centred on the convolution grid."""
    key = ('io', c['x'], c['y'], c['z'])
    if key not in _KEPT:
        ref = _truncated_green(c, True) * 0.01
        green = _c2(_truncated_green(c, False), True)
        _KEPT[key] = (ref, _c2(torch.conj(green)), _c2(green))
    return _KEPT[key]


class _Series:
    """The convergent Born series in 64 bits, arrays (z, y, x); ri as _ri gives it."""

    def __init__(self, c, ri):
        dev, dx = ri.device, c.get('dx', 0.1)
        b = _boundary(c)[::-1]
        n = [m + 2 * q for m, q in zip(ri.shape, b)]
        self.roi = tuple(slice(q, q + m) for m, q in zip(ri.shape, b))
        k = 2 * math.pi * N_M / LAM
        self.pot = (k * k * (ri * ri / (N_M * N_M) - 1)).to(torch.complex128)
        self.eps = 1.01 * float(self.pot.abs().max())
        self.V = torch.full(n, -1j * self.eps, dtype=torch.complex128, device=dev)
        self.V[self.roi] += self.pot
        self.iters = c.get('iters', 0) or int(math.ceil(math.sqrt(sum((m * dx) ** 2 for m in n)) /
                                                        (2 * k / self.eps) / 2 + 1) * 2)
        shape = lambda v, i: v.reshape([-1 if j == i else 1 for j in range(3)])  # noqa: E731
        self.mask, self.ramp, self.k = 1.0, 1.0, []
        for i, (m, q) in enumerate(zip(n, b)):
            d = torch.arange(m, dtype=torch.float64, device=dev)
            edge = torch.minimum(d, m - 1 - d)
            self.mask = self.mask * shape(torch.clamp(edge / (q - 0.5), max=1), i)
            ph = -math.pi * (d - m // 2) / (2 * m)
            self.ramp = self.ramp * shape(torch.complex(torch.cos(ph), torch.sin(ph)), i)
            f = torch.fft.ifftshift(torch.arange(m, dtype=torch.float64, device=dev) - m // 2) + 0.25
            self.k.append(shape(f / (dx * m), i))
        self.km, self.comps = k, c.get('comps', 1)

    def green(self, flip):
        turn = (lambda v, i: torch.roll(torch.flip(v, (i,)), 1, i)) if flip else (lambda v, i: v)
        kk = [turn(v, i) for i, v in enumerate(self.k)]
        g = 1 / (4 * math.pi ** 2 * (kk[0] ** 2 + kk[1] ** 2 + kk[2] ** 2) - self.km ** 2 - 1j * self.eps)
        return g, [v / (self.km / (2 * math.pi)) for v in kk[::-1]]

    def solve(self, u, tol=0.0):
        """u: (components, z, y, x) on the RI grid; returns Field + u there."""
        u = u.to(torch.complex128)
        full = (u.shape[0],) + tuple(self.V.shape)
        roi = (slice(None),) + self.roi
        src = torch.zeros(full, dtype=torch.complex128, device=u.device)
        src[roi] = self.pot * u
        src *= 0.5j / self.eps
        F = torch.zeros_like(src)
        f = first = ref = None
        for j in range(1, self.iters + 1):
            g, rad = self.green(j % 2)
            ramp = torch.conj(self.ramp) if j % 2 else self.ramp
            p = src if j <= 2 else (1j / self.eps) * f * self.V
            q = torch.fft.fftn(p * ramp, dim=(1, 2, 3))
            if self.comps == 3:
                k2 = self.km ** 2
                dot = (k2 / (k2 + 1j * self.eps)) * sum(rad[i] * q[i] for i in range(3))
                q = torch.stack([q[i] - rad[i] * dot for i in range(3)])
            q *= g
            q = self.V * torch.fft.ifftn(q, dim=(1, 2, 3)).mul_(torch.conj(ramp))
            f = (q if j <= 2 else f - p + q) * self.mask
            if j == 2:
                first = F.clone()
            F += f
            if tol and j == 2:
                ref = float(F.abs().square().sum())
            if tol and j >= 3 and float(f.abs().square().sum()) <= tol * tol * ref:
                break
            if j == 3:
                f = f + first
        return F[roi] + u


def _pad(a, c):
    """Field or RI grid -> convolution grid, over the last two axes."""
    out = torch.zeros(a.shape[:-2] + (2 * c['y'], 2 * c['x']), dtype=a.dtype, device=a.device)
    y0, x0 = c['y'] - c['y'] // 2, c['x'] - c['x'] // 2
    out[..., y0:y0 + c['y'], x0:x0 + c['x']] = a
    return out


def _crop(a, c):
    y0, x0 = c['y'] - c['y'] // 2, c['x'] - c['x'] // 2
    return a[..., y0:y0 + c['y'], x0:x0 + c['x']]


def _solve_2d(c, series, u, kernels, pin, pout, want):
    """The whole 2D solve of one field (y, x): transmitted, reflected and 3D fields (those wanted)."""
    ref, kt, kr = kernels
    U = _c2(u.to(torch.complex128)) * pin
    spec = _c2(_pad(_c2(U, True), c))
    f3 = series.solve(_crop(_c2(spec * ref, True), c)[None])[0]
    out = {'3d': f3}
    if want == ('3d',):
        return out
    em = _c2(_pad(f3 * series.pot * 0.001, c))
    out['t'] = _c2((_c2(_crop(_c2((em * kt).sum(0), True), c)) + U) * pout, True)
    if 'r' in want:
        out['r'] = _c2(_c2(_crop(_c2((em * kr).sum(0), True), c)) * pout, True)
    return out


def _to_host_order(t):
    """(angle, [z,] y, x) -> (x, y, [z,] 1, angle)."""
    return t.permute(*range(t.dim() - 1, 0, -1), 0).unsqueeze(-2).contiguous()


def exact(case, seed):
    c = case
    if c['kind'] == 'unwrap':
        return None   # the branch cuts decide the values, and they follow the search order
    if c['kind'] == 'tv':
        return _tv64(c, _tv_input(c, seed))
    ri = _ri(c, seed)
    if c['kind'] == 'loop':
        s, u = _Series(c, ri), _incident(c, seed)
        return torch.stack([s.solve(u[a], c['tol']) for a in range(c['angles'])])
    u = _fields_2d(c, seed)
    pin, pout = _pupils(c)
    k = _io_kernels(c)
    s = _Series(c, ri)
    if c['kind'] == 'field':
        k = [t.to(torch.complex64).to(torch.complex128) for t in k]
        pin, pout = (p.to(torch.float32).to(torch.float64) for p in (pin, pout))
        got = [_solve_2d(c, s, v, k, pin, pout, ('t', 'r', '3d')) for v in u]
        return [torch.stack([g[w] for g in got]) for w in (('t', '3d', 'r') if c['refl'] else ('t', '3d'))]
    if c['kind'] == 'dropin':
        got = [_solve_2d(c, s, v, k, pin, pout, ('t', '3d')) for v in u]
        return [_to_host_order(torch.stack([g[w] for g in got])) for w in ('t', '3d')]
    y = _measured(c, seed).to(torch.complex128)
    back = _Series(c, torch.conj(torch.flip(ri, (0,))))
    grad, err = 0, 0.0
    for v, m in zip(u, y):
        g = _solve_2d(c, s, v, k, pin, pout, ('t', '3d'))
        d = g['t'] - m
        err += float(d.abs().square().sum())
        w = torch.flip(torch.conj(_solve_2d(c, back, torch.conj(d), k, pin, pout, ('3d',))['3d']), (0,))
        grad = grad + torch.conj(g['3d']) * w
    return [(-1j * grad / c['angles']).permute(2, 1, 0).contiguous(), err]


def _tv64(c, v):
    """The FISTA proximal step on the dual, arrays (z, y, x)."""
    v = v.to(torch.complex128 if c['cplx'] else torch.float64)
    axes = (2, 1, 0)

    def project(a):
        if c['cplx']:
            re = a.real.clamp(0.0, 0.1) if c['bounds'] else a.real
            return torch.complex(re, a.imag.clamp(min=0))
        return a.clamp(0.0, 0.1) if c['bounds'] else a

    def primal(P):
        return project(v - _TV_LAM * sum(P[i] - torch.roll(P[i], 1, ax) for i, ax in enumerate(axes)))

    P = [torch.zeros_like(v) for _ in range(3)]
    R, t = P, 1.0
    for _ in range(c['inner']):
        y = primal(R)
        new = [R[i] + (y - torch.roll(y, -1, ax)) / (12 * _TV_LAM) for i, ax in enumerate(axes)]
        norm = torch.sqrt(torch.clamp(sum(p.abs() ** 2 for p in new), min=1))
        new = [p / norm for p in new]
        tn = (1 + math.sqrt(1 + 4 * t * t)) / 2
        R = [a + (t - 1) / tn * (a - b) for a, b in zip(new, P)]
        P, t = new, tn
    return primal(P)
