"""Interpolation, gridding and P^H P with real factors against the complex
FP64 factors applied one by one, where the kernels' variants meet: supports
with a compiled variant, mixed and odd ones and sizes up to 16; boxes of a
fixed extent, axes spanned by one tile (which wrap) and cut ones; odd and even
image sizes (the sign across the grid's edge); one and several coils (more
than a pass takes); tiles of one slot, of several and of more than a
workgroup's list; empty tiles.

Tolerance (relative 2-norm): complex64 rounds a factor per axis, the phase, the
modulation and the value (2^-24 each) and sums up to J^D <= 256 products whose
absolute sum exceeds the result at most 16-fold for the random values here:
16 * 7 * 2^-24 = 7e-6, taken as 1e-5; complex128 rounds as much less (2^-53), or
2^-50 of the accumulator's bound, at most 2^20 above the result: 1e-9."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

CASES = [
    # Nd, Kd, Jd, samples, chunk
    ((8,), (15,), (3,), 40, None),
    ((9,), (20,), (16,), 200, 16),
    ((400,), (810,), (6,), 900, 32),
    ((30, 33), (60, 66), (6, 6), 3000, 64),
    ((30, 33), (64, 72), (4, 4), 3000, None),
    ((32, 32), (64, 64), (8, 8), 2000, 32),
    ((16, 20), (48, 40), (5, 7), 1500, 20),
    ((16, 20), (50, 44), (1, 2), 1500, 20),
    ((10, 64), (15, 130), (5, 3), 1200, 33),
    ((64, 7), (130, 14), (9, 5), 700, 50),
    ((24, 24), (48, 48), (16, 11), 500, 30),
    ((20, 20), (40, 40), (6, 6), 2600, 2),
    ((20, 21, 22), (40, 42, 44), (6, 6, 6), 2500, 128),
    ((20, 17, 20), (44, 36, 40), (4, 4, 4), 1500, None),
    ((8, 20, 18), (15, 42, 36), (6, 5, 3), 1500, 100),
    ((10, 9, 40), (13, 12, 80), (2, 7, 8), 900, 100),
]


def reference(st):
    """Grid cells (M, J...) and factors of every sample."""
    d, M, Kd = len(st['Kd']), int(st['M']), st['Kd']
    cell, u = np.zeros((M, 1), np.int64), np.ones((M, 1), np.complex128)
    for a in range(d):
        j = (st['base'][a][:, None] + np.arange(st['Jd'][a])) % Kd[a]
        cell = (cell[:, :, None] * Kd[a] + j[:, None, :]).reshape(M, -1)
        u = (u[:, :, None] * st['ud'][a][:, None, :]).reshape(M, -1)
    return cell, u


def clustered(rng, M, d):
    """Half the samples in a corner at the grid's edge, so that its tile has
    many rows, and some tiles none."""
    om = rng.uniform(-np.pi, np.pi, (M, d))
    om[::2] = rng.uniform(-0.05, 0.05, (len(om[::2]), d))
    om[:, 0] = np.where(om[:, 0] > 2.5, 0.1, om[:, 0])
    return om


@pytest.mark.parametrize('coils', [None, 3, 9])
@pytest.mark.parametrize('Nd, Kd, Jd, M, chunk', CASES)
def test_stages(hip, Nd, Kd, Jd, M, chunk, coils):
    from pynufft_amd import helper
    from pynufft_amd.nufft import NUFFT
    rng = np.random.default_rng(M + sum(Kd))
    om = clustered(rng, M, len(Nd))
    st = helper.plan(om, Nd, Kd, Jd, chunk_rows=chunk)
    A = NUFFT()
    A.plan(om, Nd, Kd, Jd, batch=coils, host_plan=st)
    cell, u = reference(st)
    nb = coils or 1
    k = rng.standard_normal((int(np.prod(Kd)), nb, 2)) @ [1, 1j]
    y = rng.standard_normal((M, nb, 2)) @ [1, 1j]

    def forward(k):
        return np.einsum('mj,mjc->mc', u, k[cell])

    def back(y):
        out = np.zeros((int(np.prod(Kd)), nb), np.complex128)
        np.add.at(out, cell, np.conj(u)[:, :, None] * y[:, None, :])
        return out

    kk = k.reshape(Kd + (() if coils is None else (nb,)))
    yy = y.reshape((M,) + (() if coils is None else (nb,)))
    # complex64 plans of a large apodization spread run in FP64 as a whole
    for dtype, tol in ((np.complex64, 1e-5), (np.complex128, 1e-9)):
        ki, yi = kk.astype(dtype), yy.astype(dtype)
        assert rel(A.k2y(ki).reshape(y.shape), forward(k)) < tol
        assert rel(A.y2k(yi).reshape(k.shape), back(y)) < tol
        assert rel(A.k2y2k(ki).reshape(k.shape), back(forward(k))) < tol


@pytest.mark.parametrize('dtype', [np.complex64, np.complex128])
def test_not_finite(hip, dtype):
    """A sample that is not finite reaches its support and no other tile."""
    from pynufft_amd.nufft import NUFFT
    rng = np.random.default_rng(5)
    om = rng.uniform(-np.pi, np.pi, (500, 2))
    A = NUFFT()
    A.plan(om, (40, 40), (80, 80), (6, 6))
    y = (rng.standard_normal((500, 2)) @ [1, 1j]).astype(dtype)
    good = A.y2k(y)
    for bad in (np.nan, np.inf, complex(0, -np.inf)):
        y2 = y.copy()
        y2[7] = bad
        k = A.y2k(y2)
        cells = np.ravel_multi_index(
            [((A._host['base'][a][7] + j) % 80) for a, j in
             enumerate(np.meshgrid(np.arange(6), np.arange(6), indexing='ij'))], (80, 80)).ravel()
        assert not np.isfinite(k.ravel()[cells]).any()
        same = np.isfinite(k)
        assert same.sum() >= k.size - 4 * 21 * 21 and np.array_equal(k[same], good[same])
