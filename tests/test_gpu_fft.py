"""The line FFT against numpy's FP64 FFT at the lengths where its variants
meet: compiled lengths (32 to 1024) at their ends, two- and three-radix
schedules, prime radices, the run-time kernel below, above and between them,
single radices, and line counts that fill the last workgroup partly, along
contiguous (1 coil) and strided (9 and 17 coils) axes.

Tolerance: a radix pass rounds each value a few times (2^-24 each), so the
relative 2-norm error stays below passes * 8 * 2^-24; the longest schedule
here has four passes: 2e-6."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('coils', [None, 9, 17])
@pytest.mark.parametrize('K', [2, 6, 16, 30, 32, 36, 45, 64, 121, 130, 169, 182, 200, 216, 256,
                               390, 462, 512, 625, 968, 1000, 1024, 1040, 1331, 2048, 3840])
def test_lines(hip, K, coils):
    from pynufft_amd.nufft import NUFFT
    rng = np.random.default_rng(K)
    for N in sorted({max(1, K // 2), max(1, K // 2 + 1), K}):
        A = NUFFT()
        A.plan(rng.uniform(-3, 3, (5, 1)), (N,), (K,), (2,), batch=coils)
        shape = (N,) if coils is None else (N, coils)
        x = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
        k = A.xx2k(x)
        assert rel(k, np.fft.fft(x.astype(np.complex128), K, axis=0)) < 2e-6
        assert rel(A.k2xx(k), x) < 2e-6


@pytest.mark.parametrize('Nd', [(20, 21), (195, 231), (5, 60, 3), (13, 18, 50)])
def test_axes(hip, Nd):
    from pynufft_amd.nufft import NUFFT
    rng = np.random.default_rng(sum(Nd))
    Kd = tuple(2 * n for n in Nd)
    A = NUFFT()
    A.plan(rng.uniform(-3, 3, (5, len(Nd))), Nd, Kd, (3,) * len(Nd))
    x = (rng.standard_normal(Nd) + 1j * rng.standard_normal(Nd)).astype(np.complex64)
    k = A.xx2k(x)
    assert rel(k, np.fft.fftn(x.astype(np.complex128), s=Kd, axes=range(len(Nd)))) < 2e-6
    assert rel(A.k2xx(k), x) < 2e-6
