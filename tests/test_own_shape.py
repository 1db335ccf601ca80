"""Loops whose configuration nobody chose run in shapes picked from their
extents: stencils and 2-D loops at the row widths where the shape changes (64,
128, and one off), a cube large enough for the LDS march, and line sweeps whose
length and number of lines leave remainders of their chunks (16) and workgroups
(64, 128).  All must equal the oracle bit for bit (the SUM within its bound)."""
import numpy as np
import pytest

import helpers as H
from test_variants import _force

KIND_PARALLEL, KIND_STENCIL = 0, 3

# register march: (rows, points per lane and row, planes, 2 = stores past the caches)
STARS = [(1, 1, 4, 1), (2, 1, 1, 1), (2, 2, 5, 2), (4, 1, 3, 2), (4, 2, 2, 1), (4, 2, 500, 2), (1, 1, 7, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize('n', [65, 66, 67, 130, 282, 283])
def test_stencil3(n):
    res, ref = H.run_jac3d(n, 2), H.oracle_jac3d(n, 2)
    assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps'])
    assert H.sum_close(res['sum'], ref['sum'])


@pytest.mark.gpu
@pytest.mark.parametrize('n', [64, 65, 66, 67, 129, 130, 131])
def test_stencil2(n):
    res, ref = H.run_jac2d(n, 3), H.oracle_jac2d(n, 3)
    assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps'])


@pytest.mark.gpu
@pytest.mark.parametrize('n', [5, 16, 17, 18, 19, 34, 63, 65, 131])
def test_lines(n):
    res, ref = H.run_adi3d(n, 2), H.oracle_adi3d(n, 2)
    assert np.array_equal(res['max'], ref['max']) and np.array_equal(res['loc'], ref['loc'])
    assert H.bits_equal(res['A'], ref['A'])


def _star(kind, rows, points, planes, nt):
    _force(kind, (64, 4, 1), [nt, 1, 2, planes, rows, points, 0, 0])


@pytest.mark.gpu
@pytest.mark.parametrize('shape', STARS)
@pytest.mark.parametrize('n', [3, 4, 18, 65, 66, 67, 131])
def test_star(n, shape):
    _star(KIND_STENCIL, *shape)
    try:
        res = H.run_jac3d(n, 3)
    finally:
        _force(KIND_STENCIL, None, None)
    ref = H.oracle_jac3d(n, 3)
    assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps'])
    assert H.sum_close(res['sum'], ref['sum'])


@pytest.mark.gpu
@pytest.mark.parametrize('n', [40, 66, 100, 131])
def test_star_float(n):
    """float, a loop that names no stencil array: every step's maximum as in the direct kernel."""
    own = H.run_jackat(3, n, 20)
    _force(KIND_PARALLEL, (32, 4, 2), [1] + [0] * 7)
    try:
        ref = H.run_jackat(3, n, 20)
    finally:
        _force(KIND_PARALLEL, None, None)
    assert own[0] == ref[0] and np.array_equal(own[1], ref[1])
