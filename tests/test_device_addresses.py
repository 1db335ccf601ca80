"""A loop that folds its own reductions hands them to the host before its
launch has ended.  A device address that leaves the runtime after that must not
be used before the end: asking for one waits for the launch, once, and not in a
handler, whose launches come after the loop anyway.  (HIP calls faked.)"""
import pytest

import fake_device

CODE = '''
import ctypes
w, e = ctypes.c_double(1.5), ctypes.c_double()
A = T.array(16, 16, 16)
def sweep(handler='loop_sor3d_32_cuda'):
    r = T.region(A, scalars=[w])
    T.loop(r, 'libprog_sor3d.so', handler, A, [(1, 14)] * 3, [A, w], reds=[(3, e)], across=[1] * 6)
    T.rt.dvmh_region_end_C(r)
asks = [lambda: T.rt.dvmh_get_natural_base_C(T.L(1), A), lambda: T.rt.dvmh_get_device_addr_C(T.L(1), ctypes.byref(w)),
        lambda: T.rt.dvmh_fill_header_C(T.L(1), ctypes.c_void_p(0), A, (T.L * 64)(), None)]
def waits(ask):
    """Stream syncs, or launches that only set the completion word."""
    F.fake_clear()
    before = F.fake_syncs()
    ask()
    return F.fake_syncs() - before + sum(1 for n, g, b in T.launches() if (g, b) == (1, 64) and 'loop' not in n)
sweep()
'''


@pytest.mark.parametrize('poll', ['1', '0'])
def test_address_waits_for_the_launch(poll):
    polled = '''
for ask in asks:
    sweep()
    assert waits(ask) == 1
    assert [waits(a) for a in asks] == [0, 0, 0]
    sweep()
    sweep()
    assert waits(ask) == 1
assert T.rt.dvmh_get_natural_base_C(T.L(0), A)
'''
    synced = '''   # (the results came by a stream sync)
for ask in asks:
    sweep()
    assert [waits(a) for a in asks] == [0, 0, 0]
'''
    fake_device.run(CODE + (polled if poll == '1' else synced), DVMH_AMD_POLL=poll)


def test_not_where_the_launch_has_ended():
    """An element read back came in a launch behind the loop's."""
    fake_device.run(CODE + '''
sweep()
T.rt.dvmh_get_actual_subarray_C(A, T.L(3), *[T.L(x) for x in (3, 3, 3, 3, 3, 3)])
assert [waits(a) for a in asks] == [0, 0, 0]
''')


def test_not_in_a_handler():
    fake_device.run(CODE + '''
sweep()
real = T.D.load('libprog_sor3d.so').loop_sor3d_32_cuda
seen = []
@ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p)
def handler(ref, a, v):
    seen.append(waits(lambda: real(ctypes.c_void_p(ref), ctypes.c_void_p(a), ctypes.c_void_p(v))))
r = T.region(A, scalars=[w])
T.loop(r, None, handler, A, [(1, 14)] * 3, [A, w], reds=[(3, e)], across=[1] * 6)
T.rt.dvmh_region_end_C(r)
assert seen == [0], seen
''')
