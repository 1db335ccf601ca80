"""Loops whose configuration nobody chose run in shapes picked from their
extents: stencils and 2-D loops at the row widths where the shape changes (64,
128, and one off), a cube large enough for the LDS march, and line sweeps whose
length and number of lines leave remainders of their chunks (16) and workgroups
(64, 128).  All must equal the oracle bit for bit (the SUM within its bound)."""
import numpy as np
import pytest

import helpers as H


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
