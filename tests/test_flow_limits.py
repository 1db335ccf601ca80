"""Host decisions about the dataflow launch of ACROSS loops, with the HIP calls
faked (no GPU, nothing runs): the longest rows and the most tiles it is used
for, chains cut to what one launch can hold, and the workspace it is handed."""
import os
import sys

import fake_device

sys.path.insert(0, os.path.join(fake_device.PKG, 'emit'))
import hipgen  # noqa: E402

LOOPS = '''
import ctypes
w, e = ctypes.c_double(1.5), ctypes.c_double()
def sor(rows, cols, row, **kw):
    A = T.array(rows, cols, row)
    r = T.region(A, scalars=[w])
    F.fake_clear()
    T.loop(r, 'libprog_sor3d.so', 'loop_sor3d_32_cuda', A, [(1, rows - 2), (1, cols - 2), (1, row - 2)], [A, w], reds=[(3, e)],
           across=[1] * 6, **kw)
    T.rt.dvmh_region_end_C(r)
    got = T.launches()
    T.rt.dvmh_delete_object_(A)
    return got
def relax(rows, row):
    A = T.array(rows, row)
    r = T.region(A, scalars=[w])
    F.fake_clear()
    T.loop(r, 'libcdv_relax2d.so', 'loop_relax2d_cdv_33_cuda', A, [(1, rows - 2), (1, row - 2)], [A, w], reds=[(3, e), (4, e)], across=[1] * 4)
    T.rt.dvmh_region_end_C(r)
    got = T.launches()
    T.rt.dvmh_delete_object_(A)
    return got
def flows(got):
    assert not any(n == 'too large' for n, _, _ in got), got
    return [(n, g) for n, g, _ in got if 'flow_kernel' in n or 'flow_chain' in n]
'''


def test_longest_rows():
    """A face of (points + 28 or 77) / 8 blocks of 1 KB must be addressable in
    31 bits, with sixteen blocks to spare: 2^31 / 1024 - 16 blocks."""
    most = (1 << 31) // 1024 - 16
    fake_device.run(LOOPS + f'''
for blocks, taken in (({most}, True), ({most} + 1, False), ({most} * 2, False)):
    n3, n2 = 8 * blocks - 28 + 7, 8 * blocks - 77 + 7
    assert bool(flows(sor(11, 4, n3 + 2))) == taken, (3, blocks)
    assert bool(flows(relax(67, n2 + 2))) == taken, (2, blocks)
''')


def test_most_tasks():
    """A launch of 64-thread workgroups stays below 2^32 work-items: the rule
    as emitted (an array of so many rows does not fit the test's host memory)."""
    header = open(os.path.join(fake_device.REPO, 'include', 'dvmh_hip_device.h')).read()
    assert 'FLOW_TASKS_MAX = (1L << 26) - 1' in header
    for rank in (2, 3):
        X = 'X' + ''.join(f'[{v}]' for v in 'ijk'[:rank])
        L = hipgen.Loop({'name': 'l', 'vars': [(v, 'int') for v in 'ijk'[:rank]], 'params': [('array', 'X', 'double', rank)],
                         'across': {'array': 'X', 'widths': [(1, 1)] * rank}, 'batch': rank == 3, 'body': f'{X} += X[i - 1]{X[4:]};'}, 't')
        text = hipgen.gpu_loop(L)
        assert 'flowTiles * 1 <= dvmh_dev::FLOW_TASKS_MAX' in text
        assert ('flowTiles * most <= dvmh_dev::FLOW_TASKS_MAX' in text) == (rank == 3)


def test_chain_cut_to_a_launch():
    fake_device.run(LOOPS + '''
A = T.array(8194, 8194, 5)
T.rt.dvmh_amd_batch_begin_C()
es = [ctypes.c_double() for _ in range(130)]
for q in range(130):
    r = T.region(A, scalars=[w])
    T.loop(r, 'libprog_sor3d.so', 'loop_sor3d_32_cuda', A, [(1, 8192), (1, 8192), (1, 3)], [A, w], reds=[(3, es[q])], across=[1] * 6,
           chain='loop_sor3d_32_cuda_chain')
    T.rt.dvmh_region_end_C(r)
F.fake_clear()
T.rt.dvmh_amd_batch_end_C()
got = flows(T.launches())
tiles = 1024 * 1024
assert sum(g for _, g in got) == 130 * tiles and all(g % tiles == 0 and g * 64 < 1 << 32 for _, g in got), got
assert all('chain' in n for n, _ in got)
''')


def test_workspace_outlives_an_allocation_that_runs_short():
    """A handler is handed the workspace, then allocates its partials; where
    the device has no room left for them, what is freed to make some must not
    be the workspace.  After the handler it may be."""
    fake_device.run(LOOPS + '''
class Flow(ctypes.Structure):
    _fields_ = [('control', ctypes.c_void_p), ('flags', ctypes.c_void_p), ('cells', ctypes.c_void_p), ('wrapped', ctypes.c_void_p)]
A = T.array(16, 16, 16)
seen = []
@ctypes.CFUNCTYPE(None, ctypes.POINTER(T.L))
def handler(ref):
    ws, part = Flow(), ctypes.c_void_p()
    assert T.rt.dvmh_amd_flow_workspace_C(T.L(100), T.L(1 << 20), ctypes.byref(ws))
    assert F.fake_live(ws.control) and F.fake_live(ws.cells)
    # (a block the cache can give back, so that the retry finds room)
    F.fake_capacity(F.fake_used())
    refused = F.fake_refused()
    T.rt.dvmh_loop_cuda_register_red_C(T.L(ref[0]), T.L(1), ctypes.byref(part), None)
    T.rt.dvmh_loop_cuda_red_prepare_C(T.L(ref[0]), T.L(1), T.L(1 << 17), T.L(0))
    assert F.fake_refused() > refused and F.fake_live(part.value)
    assert F.fake_live(ws.control) and F.fake_live(ws.cells)
    seen.append(ws.cells)
r = T.region(A)
spare = T.array(1 << 18)
T.rt.dvmh_region_end_C(T.region(spare))
T.rt.dvmh_delete_object_(spare)
T.loop(r, None, handler, A, [(1, 14)] * 3, [], reds=[(3, e)])
T.rt.dvmh_region_end_C(r)
assert seen and F.fake_live(seen[0])
F.fake_capacity(F.fake_used())
B = T.array(1 << 17)
T.rt.dvmh_region_end_C(T.region(B))
assert not F.fake_live(seen[0])
''')
