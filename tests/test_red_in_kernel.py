"""Scalar reductions folded by the loop's own launch (the last workgroup to
arrive): partial counts at the edges of the group shapes -- one workgroup, one
group of 256, just over it, groups of 64, of 128 and of 512 -- and workgroups
narrower than a wave.  MAX and MAXLOC must equal the oracle's, the SUM lie
within 1e-12 relative of its compensated sum (the bound of every SUM here)."""
import numpy as np
import pytest

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
