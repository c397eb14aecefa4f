"""Performance cases of the NUFFT: what a reconstruction program calls.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same
ranges, ``prepare`` makes the plan and the inputs on the GPU, ``run`` is one
pass through the public entry points, ``work`` counts what a pass cannot do
without, and ``exact`` evaluates the same operators in 64 bits with plain
numpy and torch.

A case is a dict of plain values:

* ``op``: ``pair`` (one forward and one adjoint), ``forward``, ``adjoint``,
  ``sense`` (one image to all coils and back), ``grad`` (a training step's
  gradients in the image and the trajectory), ``cg`` (least squares by CG),
  ``batch`` (CG of many uneven problems at once), ``tv`` (L1-TV by split
  Bregman);
* ``traj``: ``uniform``, ``radial`` (golden angle) or ``spiral`` (2-D);
* ``Nd``, ``Jd``: image and interpolator sizes, as ``64x64``; ``over``: grid
  over image size; ``M``: samples; ``coils``; ``iters``: solver iterations;
* ``problems``, ``layout``: the batch's size and the seed of its sizes.

Images are smooth-phase ellipsoid phantoms with 1 % noise, samples the
closed-form Fourier transform of such a phantom with 1 % noise.
"""
import math
import random

import numpy as np
import torch

GOLDEN_ANGLE = math.pi * (math.sqrt(5.0) - 1.0) / 2.0
# the 2-D golden means (plastic-number generator) that spread 3-D spokes
GOLDEN_MEANS = (0.46557123187676802, 0.68232780382801932)


# ----------------------------------------------------------------- cases --
def _case(name, op, traj, Nd, Jd, M, over=2.0, coils=1, iters=0):
    c = dict(op=op, traj=traj, Nd=Nd, Jd=Jd, M=M, over=over, coils=coils, iters=iters)
    return dict(c, name=name) if name else c


def _batch(name, problems, layout, iters):
    c = dict(op='batch', problems=problems, layout=layout, iters=iters)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest calls: one spectrum of a line (latency and launches)
        _case('line1d_pair', 'pair', 'uniform', '256', '6', 1000),
        # the plain 2-D example size: a small slice
        _case('plain2d_pair', 'pair', 'uniform', '64x64', '6x6', 4096),
        # one slice of a radial scan, each direction by itself
        _case('radial2d_forward', 'forward', 'radial', '256x256', '6x6', 205824),
        _case('radial2d_adjoint', 'adjoint', 'radial', '256x256', '6x6', 205824),
        # an odd field of view and sample count, another support per axis
        _case('ragged2d_pair', 'pair', 'spiral', '195x231', '5x7', 60001),
        # the benchmark volume: the largest calls
        _case('uniform3d_pair', 'pair', 'uniform', '128x128x128', '6x6x6', 2097152),
        # a ragged volume on golden-means spokes (dense centre)
        _case('radial3d_pair', 'pair', 'radial', '60x75x54', '6x5x6', 300007),
        # 8 receive coils sharing a trajectory: one gradient of a SENSE recon
        _case('sense2d_pair', 'sense', 'radial', '256x256', '6x6', 131072, coils=8),
        # the same data in a training step that learns image and trajectory
        _case('sense2d_grad', 'grad', 'radial', '256x256', '6x6', 131072, coils=8),
        # iterative reconstruction of one slice, FP64 (ten iterations: past
        # about fifteen the reference's own result depends on summation order)
        _case('radial2d_cg', 'cg', 'radial', '256x256', '6x6', 205824, iters=10),
        # a stack of independent uneven slices
        _batch('batch2d_cg', 16, 400, 10),
        # total-variation reconstruction of one slice
        _case('radial2d_tv', 'tv', 'radial', '256x256', '6x6', 205824, iters=5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(n):
    """The nearest size at or below n whose prime factors are 2 to 13."""
    while True:
        m = n
        for p in (2, 3, 5, 7, 11, 13):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n -= 1


def draw(rng):
    op = rng.choice(['pair', 'pair', 'pair', 'forward', 'adjoint', 'sense', 'grad', 'cg',
                     'batch', 'tv'])
    if op == 'batch':
        return _batch(None, rng.randint(3, 16), rng.randrange(1 << 30), rng.randint(3, 10))
    if op in ('pair', 'forward', 'adjoint'):
        d = rng.choice([1, 2, 2, 3, 3])
        lo, hi = {1: (32, 1000), 2: (24, 320), 3: (16, 120)}[d]
        M = _log_int(rng, *{1: (200, 20000), 2: (1000, 250000), 3: (5000, 1000000)}[d])
        over = rng.choice([2.0, 2.0, 2.0, 1.5])
        J = [rng.choice([6, 6, 6, 4, 5, 7, 8] if d < 3 else [6, 6, 6, 4, 5])] * d
        if rng.random() < 0.25:
            J = [rng.choice([4, 5, 6, 7] if d < 3 else [4, 5, 6]) for _ in range(d)]
    else:
        d, over, J = 2, 2.0, [6, 6]
        lo, hi = 48, 256
        M = _log_int(rng, 8000, 200000)
    N = _smooth(_log_int(rng, lo, hi))
    Nd = [N] * d
    if rng.random() < 0.5:
        Nd = [_smooth(_log_int(rng, max(lo, N // 2), min(hi, 2 * N))) for _ in range(d)]
    if over != 2.0:
        Nd = [n - n % 2 if n % 2 == 0 else _smooth(n + 1) for n in Nd]
        if any(n % 2 for n in Nd):
            over = 2.0
    traj = rng.choice(['uniform', 'radial', 'spiral'] if d == 2 else
                      ['uniform', 'radial'] if d == 3 else ['uniform'])
    return _case(None, op, traj, 'x'.join(map(str, Nd)), 'x'.join(map(str, J)), M, over,
                 coils=rng.randint(2, 8) if op in ('sense', 'grad') else 1,
                 iters=rng.randint(3, 10) if op == 'cg' else rng.randint(2, 6) if op == 'tv'
                 else 0)


def _sizes(case):
    """(Nd, Kd, Jd) of a case."""
    Nd = tuple(int(v) for v in case['Nd'].split('x'))
    Jd = tuple(int(v) for v in case['Jd'].split('x'))
    return Nd, tuple(int(round(n * case['over'])) for n in Nd), Jd


def _members(case):
    """The single cases of a batch: N of 128, 192 or 256, radial or spiral."""
    rng = random.Random(case['layout'])
    out = []
    for _ in range(case['problems']):
        N = rng.choice([128, 192, 256])
        traj = rng.choice(['radial', 'spiral'])
        M = rng.randint(64, 402) * 2 * N if traj == 'radial' else rng.randint(16384, 205824)
        out.append(_case(None, 'cg', traj, '%dx%d' % (N, N), '6x6', M, iters=case['iters']))
    return out


# ---------------------------------------------------------------- inputs --
def _trajectory(case, seed):
    """(M, d) float64 coordinates in [-pi, pi) on the host."""
    Nd, _, _ = _sizes(case)
    d, M = len(Nd), case['M']
    rng = np.random.default_rng([seed, 1])
    if case['traj'] == 'uniform':
        return rng.uniform(-np.pi, np.pi, (M, d))
    turn = rng.uniform(0.0, 2.0 * np.pi)
    if case['traj'] == 'spiral':
        t = np.arange(M) / M
        r = np.tan(t * np.arctan(np.pi))          # density about 1 / (1 + r^2)
        a = 2.0 * np.pi * max(8, max(Nd) // 8) * t + turn
        om = np.stack([r * np.cos(a), r * np.sin(a)], axis=1)
    else:
        read = 2 * max(Nd)
        spoke = np.repeat(np.arange(-(-M // read)), read)[:M]
        r = np.pi * (np.tile(np.arange(read) - read // 2, -(-M // read))[:M]) / (read // 2)
        if d == 2:
            a = spoke * GOLDEN_ANGLE + turn
            om = np.stack([r * np.cos(a), r * np.sin(a)], axis=1)
        else:
            z = 2.0 * np.mod(spoke * GOLDEN_MEANS[0], 1.0) - 1.0
            a = 2.0 * np.pi * np.mod(spoke * GOLDEN_MEANS[1], 1.0) + turn
            q = np.sqrt(1.0 - z * z)
            om = np.stack([r * q * np.cos(a), r * q * np.sin(a), r * z], axis=1)
    return np.clip(om, -np.pi, np.pi - 1e-9)


def _ellipsoids(d, seed, count=10):
    """(centre, half axes, value) of random ellipsoids in [-1, 1)^d."""
    rng = np.random.default_rng([seed, 2])
    return [(rng.uniform(-0.6, 0.6, d), rng.uniform(0.05, 0.4, d),
             rng.uniform(-1, 1) * np.exp(1j * rng.uniform(-1, 1))) for _ in range(count)]


def _noise(shape, seed):
    rng = np.random.default_rng([seed, 3])
    z = rng.standard_normal(tuple(shape) + (2,), dtype=np.float32)
    return torch.view_as_complex(torch.from_numpy(z)).cuda()


def _image(case, seed):
    """complex64 ellipsoid phantom with 1 % noise."""
    Nd, _, _ = _sizes(case)
    axes = [torch.arange(n, dtype=torch.float64, device='cuda') * (2.0 / n) - 1.0 for n in Nd]
    mesh = torch.meshgrid(*axes, indexing='ij')
    img = torch.zeros(Nd, dtype=torch.complex128, device='cuda')
    for c, a, v in _ellipsoids(len(Nd), seed):
        img += ((sum(((m - ci) / ai) ** 2 for m, ci, ai in zip(mesh, c, a))) <= 1.0) * v
    img *= torch.exp(0.7j * sum(mesh))
    rms = img.abs().square().mean().sqrt()
    return (img + 0.01 * rms * _noise(Nd, seed)).to(torch.complex64)


def _samples(case, om, seed, coils=1):
    """complex64 (M,) or (M, coils): the ellipsoids' Fourier transforms, with
    coil c seeing a shifted and scaled object, and 1 % noise."""
    Nd, _, _ = _sizes(case)
    d, M = len(Nd), om.shape[0]
    w = torch.from_numpy(om).cuda()
    out = torch.zeros((M, coils), dtype=torch.complex128, device='cuda')
    half = np.array(Nd) / 2.0
    shift = np.random.default_rng([seed, 4]).uniform(-0.1, 0.1, (coils, d))
    for c, a, v in _ellipsoids(d, seed):
        s = a * half
        rho = (w * torch.from_numpy(s).cuda()).square().sum(1).sqrt().clamp_min(1e-6)
        if d == 1:
            f = 2.0 * torch.sin(rho) / rho
        elif d == 2:
            f = 2.0 * math.pi * torch.special.bessel_j1(rho) / rho
        else:
            r = rho.clamp_min(1e-2)
            f = 4.0 * math.pi * (torch.sin(r) - r * torch.cos(r)) / r ** 3
        f = f * float(np.prod(s))
        for q in range(coils):
            at = torch.from_numpy((c + shift[q]) * half).cuda()
            out[:, q] += v * (1.0 + 0.1 * q) * f * torch.exp(-1j * (w @ at))
    rms = out.abs().square().mean().sqrt()
    out = (out + 0.01 * rms * _noise((M, coils), seed + 77)).to(torch.complex64)
    return out[:, 0].contiguous() if coils == 1 else out


def _coil_maps(Nd, coils, seed):
    """complex64 Nd + (coils,): smooth maps with unit sum of squares."""
    rng = np.random.default_rng([seed, 5])
    axes = [np.linspace(-1.0, 1.0, n, endpoint=False) for n in Nd]
    mesh = np.meshgrid(*axes, indexing='ij')
    basis = np.stack([np.ones(Nd)] + list(mesh) + [m * m for m in mesh], axis=-1)
    coef = rng.standard_normal((basis.shape[-1], coils, 2))
    coef[0, :, 0] += 3.0
    S = basis @ (coef[..., 0] + 1j * coef[..., 1])
    S /= np.sqrt(np.sum(np.abs(S) ** 2, axis=-1, keepdims=True))
    return torch.from_numpy(S.astype(np.complex64)).cuda()


def _inputs(case, seed):
    """Trajectory and tensors of a single case, without a plan."""
    s = {'case': case, 'om': _trajectory(case, seed)}
    op, coils = case['op'], case['coils']
    if op in ('pair', 'forward', 'sense', 'grad'):
        s['x'] = _image(case, seed)
    if op != 'forward':
        s['y'] = _samples(case, s['om'], seed, coils if op in ('sense', 'grad') else 1)
    if op in ('sense', 'grad'):
        s['S'] = _coil_maps(_sizes(case)[0], coils, seed)
    return s


def prepare(case, seed):
    if case['op'] == 'batch':
        from pynufft_amd.batch import BatchNUFFT
        parts = [_inputs(c, seed + 1000 * i) for i, c in enumerate(_members(case))]
        A = BatchNUFFT()
        A.plan([(p['om'],) + _sizes(p['case']) for p in parts])
        return {'case': case, 'A': A, 'y': torch.cat([p['y'] for p in parts])}
    from pynufft_amd.nufft import NUFFT
    s = _inputs(case, seed)
    Nd, Kd, Jd = _sizes(case)
    A = s['A'] = NUFFT()
    A.plan(s['om'], Nd, Kd, Jd, batch=case['coils'] if 'S' in s else None)
    if case['op'] == 'sense':
        A.set_sense(s['S'])
    if case['op'] == 'grad':
        s['x'].requires_grad_(True)
        s['om'] = torch.from_numpy(s['om'].astype(np.float32)).cuda().requires_grad_(True)
    return s


# ------------------------------------------------------------------ pass --
def run(state):
    case, A = state['case'], state['A']
    op = case['op']
    if op == 'pair':
        return {'y': A.forward(state['x']), 'x': A.adjoint(state['y'])}
    if op == 'forward':
        return A.forward(state['x'])
    if op == 'adjoint':
        return A.adjoint(state['y'])
    if op == 'sense':
        return {'y': A.forward_one2many(state['x']), 'x': A.adjoint_many2one(state['y'])}
    if op == 'grad':
        from pynufft_amd.autograd import nufft_forward
        y = nufft_forward(A, state['x'][..., None] * state['S'], state['om'])
        loss = (y - state['y']).abs().square().sum()
        gx, gom = torch.autograd.grad(loss, (state['x'], state['om']))
        return {'y': y.detach(), 'gx': gx, 'gom': gom}
    if op == 'batch':
        return A.solve(state['y'], maxiter=case['iters'], rtol=0.0)
    if op == 'cg':
        return A.solve(state['y'], 'cg', maxiter=case['iters'], rtol=0.0)
    return A.solve(state['y'], 'L1TVOLS', maxiter=case['iters'], rho=1.0)


# ------------------------------------------------------------------ work --
def work(case):
    """Inputs read once (8 bytes a coordinate) and outputs written once; 8
    operations a complex multiply-add and 5 K log2 K a transform."""
    if case['op'] == 'batch':
        parts = [work(c) for c in _members(case)]
        return {k: sum(p[k] for p in parts) for k in ('bytes', 'flops')}
    Nd, Kd, Jd = _sizes(case)
    N, K, J, d = np.prod(Nd), np.prod(Kd), np.prod(Jd), len(Nd)
    M, nb, it = case['M'], case['coils'], case['iters']
    interp, fft = 8.0 * M * J * nb, 5.0 * K * math.log2(K) * nb
    once = 8.0 * M * d
    image, samples, stack = 8.0 * N, 8.0 * M * nb, 8.0 * N * nb
    op = case['op']
    if op in ('forward', 'adjoint'):
        b, f = once + image + samples, interp + fft
    elif op == 'pair':
        b, f = once + 2 * (image + samples), 2 * (interp + fft)
    elif op == 'sense':
        b, f = once + 2 * (image + samples) + stack, 2 * (interp + fft + 8.0 * N * nb)
    elif op == 'grad':
        # the trajectory's gradient: d derivatives of every sample
        b, f = 1.5 * once + 2 * (image + samples) + stack, (2 + d) * interp + 2 * fft
    elif op == 'cg':
        b, f = once + samples + image, (2 * it + 1) * interp + it * 36.0 * K + fft
    else:
        b, f = once + samples + image, (2 * it + 2) * (interp + 2 * fft) + it * 60.0 * N * d
    return {'bytes': float(b), 'flops': float(f)}


# ---------------------------------------------------------------- 64 bits --
# Kaiser-Bessel shape per support length where the grid is twice the image
_KB_SHAPE = {2: 2.5, 3: 2.27, 4: 2.31, 5: 2.34, 6: 2.32, 7: 2.32, 8: 2.35}


class _Operators:
    """The min-max NUFFT of Fessler and Sutton in 64 bits: the Kaiser-Bessel
    scaling fitted by cosines, per-axis min-max coefficients, dense loops over
    the support."""

    def __init__(self, om, Nd, Kd, Jd):
        self.Nd, self.Kd, self.Jd = Nd, Kd, Jd
        om = om if isinstance(om, torch.Tensor) else torch.from_numpy(om).cuda()
        self.M = om.shape[0]
        self.s = torch.ones((), dtype=torch.float64, device='cuda')
        self.u, self.cell = [], []
        for a, (N, K, J) in enumerate(zip(Nd, Kd, Jd)):
            alpha = self._cosines(N, K, J)
            n = torch.arange(N, dtype=torch.float64, device='cuda') - (N - 1) / 2.0
            order = range(1 - len(alpha), len(alpha))
            sd = sum(alpha[abs(l)] * torch.cos(2.0 * math.pi / K * l * n) for l in order)
            self.s = self.s[..., None] * sd
            u, cell = self._axis(om[:, a], N, K, J, alpha, order)
            self.u.append(u)
            self.cell.append(cell)

    @staticmethod
    def _cosines(N, K, J):
        """Cosine coefficients of 1 / (Kaiser-Bessel transform), fitted in
        single precision as the plan defines them."""
        L = 13 if N > 40 else -(-N // 3)
        n = np.arange(N) - (N - 1) / 2.0
        shape = J * (_KB_SHAPE[J] if K == 2 * N else 2.34)
        z = np.sqrt((np.pi * J * n / K + 0j) ** 2 - shape ** 2)
        kb = np.real(J * np.sin(z) / z) / np.i0(shape)
        A = np.cos(np.outer(2.0 * np.pi / K * n, np.arange(L + 1))).astype(np.complex64)
        alpha = np.linalg.lstsq(A, (1.0 / kb)[:, None].astype(np.complex64), rcond=-1)[0]
        alpha = np.real(alpha[:, 0]).astype(np.float64)
        alpha[1:] /= 2.0
        return alpha

    @staticmethod
    def _axis(om, N, K, J, alpha, order):
        ratio, gam = K / N, 2.0 * math.pi / K
        j = np.arange(J)
        T = sum(alpha[abs(l)] * alpha[abs(m)] * np.sinc((j[None] - j[:, None] + l - m) / ratio)
                for l in order for m in order)
        T = torch.from_numpy(np.linalg.pinv(T, rcond=J * np.finfo(float).eps)).cuda()
        first = torch.floor(om / gam - J / 2.0).detach()
        jj = torch.arange(1, J + 1, dtype=torch.float64, device='cuda')
        arg = (om / gam - first)[:, None] - jj
        r = sum(alpha[abs(l)] * torch.sinc((arg + l) / ratio) for l in order)
        u = torch.exp(1j * (om * N / 2.0)[:, None] - 1j * gam * (N - 1) / 2.0 * arg) * (r @ T.T)
        cell = torch.remainder(first.long()[:, None] + torch.arange(1, J + 1, device='cuda'), K)
        return u, cell

    def _offsets(self):
        """(coefficient, flat cell) of every support offset."""
        def walk(a, u, cell):
            if a == len(self.Nd):
                yield u, cell
                return
            for j in range(self.Jd[a]):
                uj, cj = self.u[a][:, j], self.cell[a][:, j]
                yield from walk(a + 1, uj if u is None else u * uj,
                                cj if cell is None else cell * self.Kd[a] + cj)
        return walk(0, None, None)

    def k2y(self, k):
        """(K, nb) grid to (M, nb) samples."""
        y = 0
        for u, cell in self._offsets():
            y = y + u[:, None] * k[cell]
        return y

    def y2k(self, y):
        k = torch.zeros((math.prod(self.Kd), y.shape[1], 2), dtype=torch.float64, device='cuda')
        for u, cell in self._offsets():
            k.index_add_(0, cell, torch.view_as_real(u.conj()[:, None] * y))
        return torch.view_as_complex(k)

    def xx2k(self, x):
        """Nd + (nb,) image to (K, nb) grid."""
        d = len(self.Nd)
        k = torch.fft.fftn(x, s=self.Kd, dim=tuple(range(d)))
        return k.reshape(math.prod(self.Kd), x.shape[-1])

    def k2xx(self, k):
        d = len(self.Nd)
        x = torch.fft.ifftn(k.reshape(self.Kd + (k.shape[-1],)), dim=tuple(range(d)))
        return x[tuple(slice(n) for n in self.Nd)]

    def forward(self, x):
        return self.k2y(self.xx2k(x * self.s[..., None]))

    def adjoint(self, y):
        return self.k2xx(self.y2k(y)) * self.s[..., None]

    def cg(self, y, iters):
        r = self.y2k(y)
        k, p, rr = torch.zeros_like(r), r.clone(), r.abs().square().sum()
        for it in range(iters):
            q = self.y2k(self.k2y(p))
            a = rr / torch.sum(p.conj() * q)
            k, r = k + a * p, r - a * q
            rr, old = r.abs().square().sum(), rr
            p = r + (rr / old) * p
        return (self.k2xx(k) / self.s[..., None])[..., 0]

    def tv(self, y, iters, lam):
        """Split Bregman for sum |grad x| with the k-space quadratic solve."""
        Nd, axes = self.Nd, range(len(self.Nd))
        ones = torch.ones((self.M, 1), dtype=torch.complex128, device='cuda')
        stencil = torch.zeros(self.Kd, dtype=torch.complex128, device='cuda')
        stencil[(0,) * len(Nd)] = -2.0 * len(Nd)
        for a in axes:
            for step in (1, -1):
                stencil[tuple(step if b == a else 0 for b in axes)] = 1.0
        uker = self.xx2k(self.adjoint(ones)).abs()[:, 0] - lam * torch.fft.fftn(stencil).reshape(-1)
        Ahy = self.adjoint(y)[..., 0]
        x, res = torch.zeros_like(Ahy), torch.zeros_like(Ahy)
        dd, bb = [torch.zeros_like(x) for _ in axes], [torch.zeros_like(x) for _ in axes]
        for _ in range(iters):
            rhs = res.clone()
            for a in axes:
                e = dd[a] - bb[a]
                rhs += lam * (torch.roll(e, -1, a) - e)
            k = (self.xx2k(rhs[..., None]) + 1e-7) / (uker[:, None] + 1e-7)
            x = self.k2xx(k)[..., 0]
            zz = [torch.roll(x, 1, a) - x for a in axes]
            t = [zz[a] + bb[a] for a in axes]
            mag = sum(v.abs().square() for v in t).sqrt() + 1e-5
            keep = (mag - 1.0 / lam).clamp_min(0.0) / mag
            res = res + Ahy - self.adjoint(self.forward(x[..., None]))[..., 0]
            for a in axes:
                dd[a] = t[a] * keep
                bb[a] = bb[a] + zz[a] - dd[a]
        return x


def exact(case, seed):
    if case['op'] == 'batch':
        return torch.cat([exact(c, seed + 1000 * i).reshape(-1)
                          for i, c in enumerate(_members(case))])
    s = _inputs(case, seed)
    op = case['op']
    x = s['x'].to(torch.complex128) if 'x' in s else None
    y = s['y'].to(torch.complex128) if 'y' in s else None
    S = s['S'].to(torch.complex128) if 'S' in s else None
    om = torch.from_numpy(s['om']).cuda()
    if op == 'grad':
        x.requires_grad_(True)
        om.requires_grad_(True)
    A = _Operators(om, *_sizes(case))
    if op in ('pair', 'forward', 'adjoint'):
        out = {}
        if x is not None:
            out['y'] = A.forward(x[..., None])[:, 0]
        if y is not None:
            out['x'] = A.adjoint(y[:, None])[..., 0]
        return out if op == 'pair' else next(iter(out.values()))
    if op == 'sense':
        return {'y': A.forward(x[..., None] * S), 'x': (A.adjoint(y) * S.conj()).mean(-1)}
    if op == 'grad':
        out = A.forward(x[..., None] * S)
        gx, gom = torch.autograd.grad((out - y).abs().square().sum(), (x, om))
        return {'y': out.detach(), 'gx': gx, 'gom': gom}
    if op == 'cg':
        return A.cg(y[:, None], case['iters'])
    return A.tv(y[:, None], case['iters'], 1.0)
