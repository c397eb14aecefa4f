"""The real-factor records against the complex min-max factors they replace
(CPU).

Tolerances, relative to the largest factor: the phases' arguments reach
pi * K ~ 4e3, whose FP64 rounding is 5e-13 (complex128 records); complex64
records round the factor and the phase once each (2^-24), products of up to
three axes included: 3 * 2^-24 * 2."""
import numpy as np
import pytest

from pynufft_amd import helper

GEOMETRIES = [((7,), (13,), (1,)), ((64,), (64,), (5,)), ((600,), (1301,), (16,)),
              ((9, 40), (18, 96), (6, 6)), ((33, 8), (70, 16), (3, 7)),
              ((12, 13, 20), (24, 30, 41), (6, 5, 4)), ((8, 8, 8), (8, 17, 24), (2, 1, 8))]


@pytest.mark.parametrize('Nd, Kd, Jd', GEOMETRIES)
def test_records_hold_the_factors(Nd, Kd, Jd):
    d, M = len(Nd), 300
    om = np.random.default_rng(M + sum(Kd)).uniform(-np.pi, np.pi, (M, d))
    om[0], om[1] = -np.pi, 0.0
    st = helper.plan(om, Nd, Kd, Jd)
    assert helper.has_real_factors(st)
    r64, phase = helper.real_records(st, fp64=True)
    r32 = helper.real_records(st)
    sj, rows = sum(Jd), st['perm']
    word = np.ascontiguousarray(r64[:, sj]).view(np.int64)
    tail = np.ascontiguousarray(r32[:, sj + 2:]).view(np.int32)
    assert np.array_equal(tail[:, 1 + (d == 3)], rows)
    ph32 = (r32[:, sj] + 1j * r32[:, sj + 1]).astype(np.complex128)
    at = 0
    for a in range(d):
        x = word >> 16 * a & 0xffff
        t, K = st['tile'][a], Kd[a]
        first = st['base'][a][rows]
        assert np.array_equal(x, first % t if t < K else first)
        assert np.array_equal(x, tail[:, 1] if a == 2 else tail[:, 0] >> 16 * a & 0xffff)
        u = st['ud'][a][rows]
        cell = first[:, None] + np.arange(Jd[a])[None, :]
        wrapped = np.where(cell >= K, (-1.0) ** (Nd[a] - 1), 1.0)
        grid = helper.grid_modulation(Nd[a], K)[cell % K] * wrapped
        other = np.exp(1j * (om[rows].sum(1) - om[rows, a]) / 2)[:, None]
        top = np.abs(u).max()
        for rec, p, tol in ((r64, phase, 5e-12), (r32, ph32, 6 * 2.0 ** -24)):
            c = rec[:, at:at + Jd[a]].astype(np.float64)
            # the phase of the whole sample: the other axes' part divided out
            got = c * p[:, None] / other
            assert np.abs(got - u * np.conj(grid)).max() <= tol * top
        at += Jd[a]


def test_other_factors_are_refused():
    st = helper.plan(np.random.default_rng(0).uniform(-3, 3, (50, 1)), (16,), (32,), (4,))
    st['ud'] = [st['ud'][0] * np.exp(0.1j * np.arange(4))]
    assert not helper.has_real_factors(st)


def test_one_other_row_is_found():
    """A row that the sampled check misses."""
    st = helper.plan(np.random.default_rng(0).uniform(-3, 3, (9000, 1)), (16,), (32,), (4,))
    st['ud'][0][8002] *= np.exp(0.1j * np.arange(4))
    sampled = np.unique(np.linspace(0, 8999, 4096).astype(np.int64))
    assert 8002 not in sampled and helper.has_real_factors(st)
    assert helper.real_records(st) is None
