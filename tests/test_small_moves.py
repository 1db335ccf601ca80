"""Small moves between host and device: scalars that enter a region in a
launch's arguments (eight to a launch, 16 bytes at most, larger ones copied)
and blocks of up to 2048 bytes written back through mapped memory (one byte to
just over the limit; elements of 1 to 24 bytes, also across word borders).
Bytes are bytes: what comes back must be what was sent."""
import ctypes

import numpy as np
import pytest

import dvmh_amd as D
import helpers as H   # noqa: F401  (initialises the runtime)

L = ctypes.c_long
TARGETS = L(D.DEVICE_TYPE_HOST | D.DEVICE_TYPE_CUDA)
INOUT = L(3)


def _rt():
    rt = D.runtime()
    rt.dvmh_region_create_C.restype = L
    rt.dvmh_get_natural_base_C.restype = ctypes.c_void_p
    rt.dvmh_distribution_block_C.restype = L
    return rt


def _blocks(size):
    """(lo, hi) per axis of a 24 x 300 array: single elements, odd rows, the limit and just over it."""
    full = 2048 // size
    return [((0, 0), (0, 0)), ((23, 299), (23, 299)), ((3, 1), (3, 7)), ((2, 5), (4, 9)), ((7, 0), (7, min(299, full - 1))),
            ((0, 11), (23, 11)), ((5, 1), (12, full // 8)), ((5, 1), (12, full // 8 + 1))]


@pytest.mark.gpu
@pytest.mark.parametrize('size', [1, 2, 4, 8, 12, 16, 24])
def test_blocks_back(size):
    rt = _rt()
    hdr = (L * 64)()
    rt.dvmh_array_create_C(hdr, L(2), L(size), L(24), L(1), L(1), L(300), L(1), L(1))
    rt.dvmh_distribute_C(hdr, L(2), *[L(rt.dvmh_distribution_block_C(L(a))) for a in (1, 2)])
    base = rt.dvmh_get_natural_base_C(L(0), hdr)
    host = np.ctypeslib.as_array(ctypes.cast(base, ctypes.POINTER(ctypes.c_ubyte)), shape=(24, 300, size))
    want = np.random.default_rng(size).integers(0, 256, host.shape, dtype=np.uint8)
    for lo, hi in _blocks(size):
        host[...] = want
        rt.dvmh_actual_all2_()
        r = L(rt.dvmh_region_create_C(L(0)))
        rt.dvmh_region_register_array_C(r, INOUT, hdr, b'a')
        rt.dvmh_region_execute_on_targets_C(r, TARGETS)
        rt.dvmh_region_end_C(r)
        host[...] = 0
        rt.dvmh_get_actual_subarray_C(hdr, L(2), L(lo[0]), L(hi[0]), L(lo[1]), L(hi[1]))
        sel = (slice(lo[0], hi[0] + 1), slice(lo[1], hi[1] + 1))
        assert np.array_equal(host[sel], want[sel]), (lo, hi)
        host[sel] = 0
        assert not host.any(), (lo, hi)
        rt.dvmh_get_actual_all2_()
    rt.dvmh_delete_object_(hdr)


@pytest.mark.gpu
@pytest.mark.parametrize('sizes', [[1], [8] * 8, [8] * 9, [1, 2, 4, 8, 16, 12, 3, 24, 16, 7, 2048, 2049]])
def test_scalars_there_and_back(sizes):
    rt = _rt()
    rng = np.random.default_rng(len(sizes))
    sent = [rng.integers(0, 256, s, dtype=np.uint8) for s in sizes]
    here = [x.copy() for x in sent]
    for _ in range(2):
        for h, s in zip(here, sent):
            h[...] = s
            rt.dvmh_actual_variable2_(ctypes.c_void_p(h.ctypes.data))
        r = L(rt.dvmh_region_create_C(L(0)))
        for h in here:
            rt.dvmh_region_register_scalar_C(r, INOUT, ctypes.c_void_p(h.ctypes.data), L(h.size), b's')
        rt.dvmh_region_execute_on_targets_C(r, TARGETS)
        for h in here:
            h[...] = 0
        rt.dvmh_region_end_C(r)
        assert all(np.array_equal(h, s) for h, s in zip(here, sent))
        sent = [np.roll(s, 1) for s in sent]
    for h in here:   # the addresses may be other variables' later
        rt.dvmh_data_exit_C(ctypes.c_void_p(h.ctypes.data), L(0))
