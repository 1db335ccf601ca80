"""Sweeps over whole numbers whose axes all depend (programs/sweeps.cdv): every
value must equal the sequential sweep's, in the element type's own range."""
import ctypes
import os
import re

import numpy as np
import pytest

import dvmh_amd as D

FORMS = {'uchar': (np.uint8, 3), 'uint': (np.uint32, 2), 'uint3': (np.uint32, 3), 'ulong': (np.uint64, 2),
         'ulonglong': (np.uint64, 3)}


def reference(which, n, iters):
    dtype, rank = FORMS[which]
    at = np.indices((n,) * rank).astype(np.uint64)
    start = at[0] * 2654435761 + at[1] * 40503 + (at[2] * 97 if rank == 3 else 0)
    m = (1 << 64) - 1   # (sums modulo 2^64 are those modulo any shorter range)
    a = (start & 0xffffffff).astype(dtype).astype(object)
    for _ in range(iters):
        for p in np.ndindex(*(n - 2,) * rank):
            i, j, k = p[0] + 1, p[1] + 1, p[-1] + 1
            if rank == 2:
                a[i, j] = (a[i - 1, j] + 3 * a[i + 1, j] + a[i, j - 1] + 5 * a[i, j + 1] + a[i, j]) & m
            else:
                a[i, j, k] = (a[i - 1, j, k] + 3 * a[i + 1, j, k] + a[i, j - 1, k] + 5 * a[i, j + 1, k] + a[i, j, k - 1] + 7 * a[i, j, k + 1] +
                              a[i, j, k]) & m
    return a.astype(np.uint64).astype(dtype).astype(np.int64).ravel()


def check(which, n, iters):
    D.runtime()
    f = getattr(D.load('libcdv_sweeps.so'), 'sweep_' + which)
    f.restype = None
    out = np.zeros(n ** FORMS[which][1], dtype=np.int64)
    f(ctypes.c_long(n), ctypes.c_int(iters), out.ctypes.data_as(ctypes.POINTER(ctypes.c_long)))
    assert np.array_equal(out, reference(which, n, iters))


@pytest.mark.parametrize('which', sorted(FORMS))
def test_host_path(which):
    if D.stats()['gpu_present']:
        pytest.skip('the host path runs where no GPU is present; the GPU tests cover this case')
    check(which, 7, 2)


@pytest.mark.gpu
@pytest.mark.parametrize('which', sorted(FORMS))
@pytest.mark.parametrize('n', [3, 10, 11, 35])
def test_gpu(which, n):
    before = D.stats()['loops_gpu']
    check(which, n + (60 if FORMS[which][1] == 2 else 0), 2)
    assert D.stats()['loops_gpu'] > before


def test_taken_by_the_dataflow_launch():
    text = open(os.path.join(D.PKG_DIR, 'gen', 'cdv', 'sweeps_cdv_hip.hip')).read()
    assert len(set(re.findall(r'\w+_flow_kernel\b', text))) == len(FORMS)
