"""Loops with branches (programs/branches.cdv).  A condition that stands beside
the accesses to neighbours keeps the kernels that load ahead; one that guards
them does not.  Results must equal a sequential evaluation bit for bit."""
import ctypes
import os
import sys

import numpy as np
import pytest

import dvmh_amd as D
import helpers as H
from test_cdvmh import _u01
from test_variants import _force

sys.path.insert(0, os.path.join(H.REPO, 'dvm-snapshot-r6603-fork_amd', 'emit'))
import hipgen  # noqa: E402

_dp = ctypes.POINTER(ctypes.c_double)
SEED = D.SEED_BASE + 11

T = 'double t = X[i - 1][j] + X[i + 1][j] + X[i][j - 1] + X[i][j + 1];\n'
FORMS = [   # body, every neighbour is reached in every iteration
    (T + 'X[i][j] = t;', True),
    (T + 'if (t > r) r = t;\nX[i][j] = t;', True),
    (T + 'r = MAX(r, t);\nX[i][j] = t > 1 ? t : X[i][j];', True),
    (T + 'r = r > t && t > 0 ? r : t;\nif (t > 0) X[i][j] = t; else { X[i][j] = -t; }', True),
    (T + 'for (int q = 0; q < 3; q++) t *= 0.5;\nwhile (t > 4) { t -= 1; if (t < 0) break; }\nX[i][j] = t;', True),
    (T + 'switch ((int)t) { case 0: t = 1; break; default: t = 2; }\nX[i][j] = t;', True),
    (T + 'X[i][j] = weight(t);', True),
    ('/* if (i) */ ' + T + 'X[i][j] = t;   // && so on', True),
    (T + 'if (i > 1) t += X[i - 1][j];\nX[i][j] = t;', True),          # reached anyway
    ('if (i > 0) { ' + T + ' X[i][j] = t; }', False),
    ('double t = X[i + 1][j] + X[i][j + 1];\nif (i > 0) t += X[i - 1][j];\nX[i][j] = t + X[i][j - 1];', False),
    ('double t = i > 0 ? X[i - 1][j] : 0;\nX[i][j] = t + X[i + 1][j] + X[i][j - 1] + X[i][j + 1];', False),
    ('double t = X[i + 1][j] + X[i][j - 1] + X[i][j + 1];\nX[i][j] = t * (i > 0 && X[i - 1][j] > 0);', False),
    ('for (int q = 0; q < i; q++) X[i][j] += X[i - 1][j] + X[i][j - 1] + X[i + 1][j] + X[i][j + 1];', False),
    ('do { if (i < 1) break; X[i][j] += X[i - 1][j]; } while (0);', False),
    ('SELECT(i > 0, X[i][j]);\n' + T + 'X[i][j] = t;', False),           # may jump
    ('X[i][j] = weight(X[i - 1][j]);', False),                           # may be a macro that picks
    ('X[i][j] = X[i][j] > 0 || X[i - 1][j] > 0;', False),
    ('if (j == 3) goto out;\n' + T + 'X[i][j] = t;\nout: ;', False),
    ('switch (j) { case 1: X[i][j] = X[i - 1][j]; }', False),
    ('{ { ' + T + ' } if (r > 0) r = 0; }\nX[i][j] = r;', True),
    (T + 'X[i][j] = t', False),                                          # no statement: in doubt
]


@pytest.mark.parametrize('body,ahead', FORMS)
def test_what_may_be_loaded_ahead(body, ahead):
    L = hipgen.Loop({'name': 'l', 'vars': [('i', 'int'), ('j', 'int')], 'params': [('array', 'X', 'double', 2)],
                     'reductions': [('max', 'r', 'double')], 'across': {'array': 'X', 'widths': [(1, 1), (1, 1)]}, 'body': body}, 't')
    assert L.loads_ahead('X') == ahead
    assert L.flow_eligible() == ahead


@pytest.mark.parametrize('tail,march', [
    ('B[i][j][k] = t;', True), ('B[i][j][k] = exp(t) + sqrt(t);', True), ('if (t > r) r = t;\nB[i][j][k] = fabs(t);', True),
    ('B[i][j][k] = t > 1 ? MAX(t, 2.0) : t;', True), ('B[i][j][k] = t > 0 ? sqrt(t) : 0;', False), ('if (t > 1) t = sin(t);\nB[i][j][k] = t;', False),
    ('while (t > 1) t *= 0.5;\nB[i][j][k] = t;', False), ('for (int q = 0; q < 4; q++) t *= t;\nB[i][j][k] = t;', False),
    ('B[i][j][k] = weight(t);', False)])
def test_which_bodies_march(tail, march):
    """The register march where nobody tuned: not for bodies that take lanes apart for long."""
    L = hipgen.Loop({'name': 'l', 'vars': [(v, 'int') for v in 'ijk'], 'params': [('array', 'A', 'double', 3), ('array', 'B', 'double', 3)],
                     'reductions': [('max', 'r', 'double')],
                     'body': 'double t = A[i - 1][j][k] + A[i + 1][j][k] + A[i][j - 1][k] + A[i][j][k + 1];\n' + tail}, 't')
    assert (L.star_array() == 'A') == march


def test_early_end_keeps_other_kernels():
    """(a kernel whose body is a function's)"""
    L = hipgen.Loop({'name': 'l', 'vars': [('i', 'int'), ('j', 'int')], 'params': [('array', 'X', 'double', 2)],
                     'across': {'array': 'X', 'widths': [(1, 1), (1, 1)]}, 'body': T + 'if (t < 0) continue;\nX[i][j] = t;'}, 't')
    assert L.loads_ahead('X') and not L.flow_eligible()


def _grid(n):
    return _u01(SEED, np.arange(n ** 3, dtype=np.uint64)).reshape(n, n, n)


def sor_reference(n, iters, w):
    a = _grid(n).tolist()
    hist = []
    for _ in range(iters):
        eps = 0.0
        for i in range(1, n - 1):
            for j in range(1, n - 1):
                row, up, down, left, right = a[i][j], a[i - 1][j], a[i + 1][j], a[i][j - 1], a[i][j + 1]
                for k in range(1, n - 1):
                    s = row[k]
                    t = (up[k] + down[k] + left[k] + right[k] + row[k - 1] + row[k + 1]) / 6.0
                    d = abs(t - s)
                    if d > eps:
                        eps = d
                    if s > 0.05 and d > 0.001:
                        row[k] = s + (0.5 * w if d > 0.5 else w) * (t - s)
        hist.append(eps)
    return np.array(hist), np.array(a).ravel()


def edge_reference(n, iters, w):
    a = _grid(n).tolist()
    for _ in range(iters):
        for i in range(n):
            for j in range(n):
                for k in range(n):
                    t = 0.0
                    if i > 0:
                        t += a[i - 1][j][k]
                    if j > 0:
                        t += a[i][j - 1][k]
                    t += a[i][j][k - 1] if k > 0 else 0.5
                    if i < n - 1:
                        t += a[i + 1][j][k]
                    a[i][j][k] = (1 - w) * a[i][j][k] + w * t
    return None, np.array(a).ravel()


def jac_reference(n, iters, c):
    A = _grid(n)
    hist = []
    for _ in range(iters):
        m = A[1:-1, 1:-1, 1:-1]
        t = A[:-2, 1:-1, 1:-1] + A[2:, 1:-1, 1:-1] + A[1:-1, :-2, 1:-1] + A[1:-1, 2:, 1:-1] + A[1:-1, 1:-1, :-2] + A[1:-1, 1:-1, 2:]
        d = np.abs(t / 6.0 - m)
        hist.append(max(0.0, d.max()))
        A[1:-1, 1:-1, 1:-1] = np.where(d > 0.3, t / 6.0, m)
        for i in range(1, n):
            t = A[i] + c * A[i - 1]
            A[i] = np.where(t < 2.0, t, A[i])
        for k in range(1, n):
            A[:, :, k] = A[:, :, k] + c * A[:, :, k - 1]
    return np.array(hist), A.ravel()


def edge2d_reference(n, iters, _):
    A = _u01(SEED, np.arange(n ** 2, dtype=np.uint64)).reshape(n, n)
    for _ in range(iters):
        t = A.copy()
        t[1:] += A[:-1]
        t[:-1] += A[1:]
        t += np.concatenate([np.full((n, 1), 0.25), A[:, :-1]], axis=1)
        t += np.concatenate([A[:, 1:], np.full((n, 1), 0.75)], axis=1)
        A = 0.2 * t
    return None, A.ravel()


def two3d_reference(n, iters, w):
    a, b = _grid(n).tolist(), np.full((n, n, n), 0.5).tolist()
    hist = []
    for _ in range(iters):
        eps = 0.0
        for i in range(1, n - 1):
            for j in range(1, n - 1):
                for k in range(1, n - 1):
                    t = (a[i - 1][j][k] + a[i + 1][j][k] + a[i][j - 1][k] + a[i][j + 1][k] + a[i][j][k - 1] + a[i][j][k + 1]) / 6.0
                    b[i][j][k] = 0.5 * b[i - 1][j][k] + 0.25 * b[i][j][k - 1] + 0.125 * t
                    a[i][j][k] = (1 - w) * a[i][j][k] + w * (t - 0.125 * b[i][j - 1][k])
                    if t > eps:
                        eps = t
        for i in range(1, n - 1):
            for j in range(1, n - 1):
                for k in range(1, n - 1):
                    a[i][j][k] = 0.25 * (a[i - 1][j][k] + a[i][j + 1][k] + a[i][j][k - 1] + a[i][j][k])
        hist.append(eps)
    return np.array(hist), np.array(a).ravel()


REFERENCE = {'two3d': two3d_reference, 'edge2d': edge2d_reference, 'sor3d': sor_reference, 'edge3d': edge_reference, 'jac3d': jac_reference}


def run(which, n, iters, factor):
    f = getattr(D.load('libcdv_branches.so'), 'branch_' + which)
    f.restype = None
    hist = None if which.startswith('edge') else np.zeros(iters)
    out = np.zeros(n ** int(which[-2]))
    D.runtime()
    f(ctypes.c_long(n), ctypes.c_int(iters), *([] if which == 'edge2d' else [ctypes.c_double(factor)]), ctypes.c_ulonglong(SEED),
      *([] if hist is None else [H.dp(hist)]), H.dp(out))
    return hist, out


def check(which, n, iters):
    factor = {'sor3d': 1.25, 'two3d': 0.8}.get(which, 0.2)
    hist, out = run(which, n, iters, factor)
    rh, ro = REFERENCE[which](n, iters, factor)
    assert H.bits_equal(out, ro)
    assert hist is None or np.array_equal(hist, rh)


@pytest.mark.parametrize('which', sorted(REFERENCE))
def test_host_path(which):
    if D.stats()['gpu_present']:
        pytest.skip('the host path runs where no GPU is present; the GPU tests cover this case')
    check(which, 9, 2)


@pytest.mark.gpu
@pytest.mark.parametrize('which', sorted(REFERENCE))
@pytest.mark.parametrize('n', [3, 5, 10, 19, 34, 67])
def test_gpu(which, n):
    before = D.stats()['loops_gpu']
    check(which, n, 2)
    assert D.stats()['loops_gpu'] > before


@pytest.mark.gpu
@pytest.mark.parametrize('kind,block,tune', [(1, (64, 1, 1), [1, 0, 2, 0, 16, 0, 0, 0]), (1, (128, 1, 1), [1, 0, 3, 0, 0, 0, 0, 0]),
                                             (1, (64, 1, 1), [1, 0, 1, 0, 16, 1, 0, 0]), (3, (64, 4, 1), [1, 0, 1, 16, 2, 0, 0, 0]),
                                             (3, (64, 4, 1), [1, 1, 2, 8, 2, 1, 0, 0]), (3, (256, 1, 1), [1, 0, 1, 8, 4, 0, 0, 0])])
def test_variants_gpu(kind, block, tune):
    """Staged variants asked for: taken where no load leaves the array, the
    direct kernel elsewhere."""
    _force(kind, block, tune)
    try:
        check('jac3d', 34, 2)
        check('edge2d', 131, 2)
    finally:
        _force(kind, None, None)


@pytest.mark.gpu
@pytest.mark.parametrize('nt,ta,tc', [(64, 4, 8), (256, 8, 16), (256, 12, 16), (32, 16, 8)])
@pytest.mark.parametrize('n', [3, 9, 20, 35])
def test_tiles_gpu(nt, ta, tc, n):
    """The tiled wavefront, which such sweeps keep, with one column per thread,
    up to four and more; edge3d's guards close, so it runs hyperplanes."""
    _force(2, (nt, 1, 1), [1, 0, 1, 0, ta, tc, 0, 0])
    try:
        check('two3d', n, 2)
        check('edge3d', n, 2)
    finally:
        _force(2, None, None)
