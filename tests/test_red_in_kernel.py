"""Scalar reductions folded by the loop's own launch (the last workgroup to
arrive): partial counts at the edges of the group shapes -- one workgroup, one
group of 256, just over it, groups of 64, of 128 and of 512 -- and workgroups
narrower than a wave.  MAX and MAXLOC must equal the oracle's, the SUM lie
within 1e-12 relative of its compensated sum (the bound of every SUM here)."""
import ctypes

import numpy as np
import pytest

import fake_device as T
import helpers as H
from test_variants import _force

KIND_PARALLEL, KIND_STENCIL = 0, 3

# (n, block x): interior (n - 2)^3 in workgroups of x * 1 * 1 points
PARTIALS = [(3, 64), (18, 64), (19, 64), (66, 64), (67, 64), (200, 64), (19, 8), (19, 1), (34, 32)]


def _forced(kind, bx):
    _force(kind, (bx, 1, 1), [1] + [0] * 7)


@pytest.mark.gpu
@pytest.mark.parametrize('n,bx', PARTIALS)
def test_max_and_sum(n, bx):
    _forced(KIND_STENCIL, bx)
    try:
        res = H.run_jac3d(n, 3)
    finally:
        _force(KIND_STENCIL, None, None)
    ref = H.oracle_jac3d(n, 3)
    assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps'])
    assert H.sum_close(res['sum'], ref['sum'])


@pytest.mark.gpu
@pytest.mark.parametrize('n,bx', [(16, 64), (17, 64), (65, 64), (130, 64), (17, 8)])
def test_maxloc(n, bx):
    _forced(KIND_PARALLEL, bx)
    try:
        res = H.run_adi3d(n, 2)
    finally:
        _force(KIND_PARALLEL, None, None)
    ref = H.oracle_adi3d(n, 2)
    assert np.array_equal(res['max'], ref['max']) and np.array_equal(res['loc'], ref['loc'])


def _extremes(kind, n, m, rng):
    a = rng.random((n, m)) - 0.5
    at = rng.integers(0, n * m, 5)
    if kind == 'all inf':
        a[:] = np.inf
    elif kind == 'all lowest':
        a[:] = -np.finfo(np.float64).max
    elif kind == 'all minus inf':
        a[:] = -np.inf
    elif kind == 'some of both':
        a.ravel()[at] = [np.inf, -np.inf, -np.inf, np.inf, -np.inf]
    elif kind == 'nan':   # the body's `if (a < min)` passes over them
        a.ravel()[rng.integers(0, n * m, n * m // 3)] = np.nan
    return a


@pytest.mark.gpu
@pytest.mark.parametrize('kind', ['all inf', 'all lowest', 'all minus inf', 'some of both', 'nan'])
@pytest.mark.parametrize('n,m', [(1, 1), (3, 70), (40, 301), (700, 1501)])
def test_extremes(kind, n, m):
    """MAX, MINLOC and SUM over infinities, the type's lowest value and (MINLOC)
    NaN, from initial values that may win, in one group of partials and in many."""
    a = _extremes(kind, n, m, np.random.default_rng(n * m))
    A, cols = T.array(n, m), ctypes.c_long(m)
    T.host(A, (n, m))[...] = a
    T.rt.dvmh_actual_array2_(A)
    for start in (2.0, -np.inf, np.inf):
        s, p, mx, mn = (ctypes.c_double(x) for x in (0, 1, start, start))
        loc = ctypes.c_long(-1)
        r = T.region(A, scalars=[cols])
        T.loop(r, 'libcdv_redall.so', 'loop_redall_cdv_82_cuda', A, [(0, n - 1), (0, m - 1)], [A, cols],
               reds=[(1, s), (2, p), (3, mx), (12, mn, loc)])
        T.rt.dvmh_region_end_C(r)
        flat = a.ravel()
        low = np.where(np.isnan(flat), np.inf, flat)
        assert (mn.value, loc.value) == ((low.min(), int(low.argmin())) if low.min() < start else (start, -1))
        if kind != 'nan':
            assert mx.value == max(flat.max(), start)
        if not np.isfinite(flat).all():
            with np.errstate(invalid='ignore'):
                assert np.array_equal(s.value, flat.sum(), equal_nan=True)
    T.rt.dvmh_delete_object_(A)
