"""Host decisions about the dataflow launch of ACROSS loops, with the HIP calls
faked (no GPU, nothing runs): the longest rows and the most tiles it is used
for, chains cut to what one launch can hold, and the workspace it is handed."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import dvmh_amd as D
import fake_device
import helpers as H

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
    return [(n[n.index('loop'):n.index('_kernel')], g) for n, g, _ in got if 'flow_kernel' in n or 'flow_chain' in n]
SOR, RELAX = 'loop_sor3d_32_flow', 'loop_relax2d_cdv_33_flow'
'''


def test_longest_rows():
    """A face of (points + 28 or 77) / 8 blocks of 1 KB must be addressable in
    31 bits, with sixteen blocks to spare: longer rows are walked part by part."""
    fake_device.run(LOOPS + f'''
most = (1 << 31) // 1024 - 16
row = 8 * most - 128
assert row + 77 <= 8 * most
for parts in (1, 2, 3):
    for n in ((row * (parts - 1) + 1, row * parts) if parts > 1 else (row,)):
        assert flows(sor(11, 4, n + 2)) == [(SOR, 2)] * parts, (3, n)
        assert flows(relax(67, n + 2)) == [(RELAX, 2)] * parts, (2, n)
''')


def test_most_tasks():
    """A launch of 64-thread workgroups stays below 2^32 work-items: the rules
    as emitted (an array of so many rows does not fit the test's host memory)."""
    header = open(os.path.join(fake_device.REPO, 'include', 'dvmh_hip_device.h')).read()
    assert 'FLOW_TASKS_MAX = (1L << 26) - 1' in header
    for rank in (2, 3):
        X = 'X' + ''.join(f'[{v}]' for v in 'ijk'[:rank])
        L = hipgen.Loop({'name': 'l', 'vars': [(v, 'int') for v in 'ijk'[:rank]], 'params': [('array', 'X', 'double', rank)],
                         'across': {'array': 'X', 'widths': [(1, 1)] * rank}, 'batch': rank == 3, 'body': f'{X} += X[i - 1]{X[4:]};'}, 't')
        text = hipgen.gpu_loop(L)
        assert 'while (flow && !(flowPart * flowB <= dvmh_dev::FLOW_TASKS_MAX &&' in text
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


def test_workspace_is_bounded():
    """Less room than the cells of all tiles take: the sweep runs in parts
    whose tiles add up; no room at all, or none allowed: hyperplanes."""
    code = LOOPS + '''
def cells(tiles, n):   # bytes, rank 3
    return tiles * 2 * ((n + 28) // 8) * 1024
n = 200
whole = 25 * 25
F.fake_capacity(F.fake_used() + (1 << 28))
first = flows(sor(n + 2, n + 2, n + 2))
assert sum(g for _, g in first) == whole
'''
    fake_device.run(code + 'assert len(first) == 1\n')
    for mb in (3, 10, 20):
        fake_device.run(code + f'''
part = max(g for _, g in first)
assert len(first) > 1 and cells(part, n) <= {mb} << 20, first
assert all(g == part for _, g in first[:-1])
assert flows(sor(n + 2, n + 2, n + 2)) == first
''', DVMH_AMD_FLOW_MB=str(mb))
    fake_device.run(LOOPS + '''
got = sor(42, 42, 42)
assert not flows(got) and any('wave012' in x for x, _, _ in got)
''', DVMH_AMD_FLOW_MB='0')
    # the device itself is short: room for the array and a little more
    fake_device.run(LOOPS + '''
A = T.array(202, 202, 202)
T.rt.dvmh_region_end_C(T.region(A, scalars=[w]))
F.fake_capacity(F.fake_used() + (80 << 20))
asked = []
for _ in range(3):
    r = T.region(A, scalars=[w])
    F.fake_clear()
    before = F.fake_asked()
    T.loop(r, 'libprog_sor3d.so', 'loop_sor3d_32_cuda', A, [(1, 200)] * 3, [A, w], reds=[(3, e)], across=[1] * 6)
    asked.append(F.fake_asked() - before)
    got = flows(T.launches())
    assert len(got) > 1 and sum(g for _, g in got) == 625, got
    T.rt.dvmh_region_end_C(r)
assert asked[0] > 1 and asked[1:] == [0, 0], asked   # not asked for again and again
''')


def test_workspace_is_given_back():
    """An array that needs the room gets it, also while captured graphs hold the
    workspace; the graphs are captured again when they recur."""
    fake_device.run(LOOPS + '''
T.rt.dvmh_amd_set_graph_C(T.L(1))
T.rt.dvmh_amd_set_graph_min_nodes_C(T.L(1))
A = T.array(102, 102, 102)
def sweep():
    r = T.region(A, scalars=[w], flags=256)
    F.fake_clear()
    T.loop(r, 'libprog_sor3d.so', 'loop_sor3d_32_cuda', A, [(1, 100)] * 3, [A, w], reds=[(3, e)], across=[1] * 6)
    T.rt.dvmh_region_end_C(r)
    return [x for x, _, _ in T.launches()]
for _ in range(4):
    got = sweep()
assert 'graph' in got and F.fake_graphs() == 1
held = F.fake_used()
F.fake_capacity(held)
B = T.array(100, 5000)   # 4 MB, less than the workspace holds
r = T.region(B)
T.rt.dvmh_region_end_C(r)
assert F.fake_graphs() == 0 and F.fake_used() <= held
F.fake_capacity(1 << 34)
for _ in range(4):
    got = sweep()
assert 'graph' in got and F.fake_graphs() == 1
''')


CHILD = f'''
import sys
sys.path[:0] = [{fake_device.PKG!r}, {fake_device.HERE!r}]
import numpy as np
import helpers as H
from test_cdvmh import _check_relax2d
for n in (20, 67, 131):
    for run in (lambda: H.run_sor3d(n, 3), lambda: H.run_sor3d_chain(n, 3, 3)):
        res, ref = run(), H.oracle_sor3d(n, 3)
        assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps']), n
for n in (66, 200, 331):
    _check_relax2d(n, 2)
rt = H.D.runtime()
rt.dvmh_amd_set_graph_C(1)
rt.dvmh_amd_set_graph_min_nodes_C(1)
before = H.D.stats()['graph_replays']
res, ref = H.run_sor3d(67, 8, flags=H.D.REGION_AMD_GRAPH), H.oracle_sor3d(67, 8)
assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps']) and H.D.stats()['graph_replays'] > before + 4
print('equal')
'''


@pytest.mark.gpu
@pytest.mark.parametrize('mb', [0, 1, 3])
def test_in_parts_gpu(mb):
    """No workspace, one for a row of tiles or so, one for some: sweeps in parts
    (replayed from a graph too), chains sweep by sweep."""
    p = subprocess.run([sys.executable, '-c', CHILD], env=dict(os.environ, DVMH_AMD_FLOW_MB=str(mb)), capture_output=True, text=True, timeout=100)
    assert p.returncode == 0 and p.stdout.strip().endswith('equal'), p.stderr[-2000:]


@pytest.mark.gpu
@pytest.mark.parametrize('cut', [1, 8, 9, 30])
def test_rows_in_parts_gpu(cut):
    """A sweep cut along its innermost axis, the parts one after another."""
    T, n = fake_device, 40
    w, e, nn, seed = ctypes.c_double(1.5), ctypes.c_double(0), ctypes.c_long(n), ctypes.c_ulonglong(D.SEED_BASE + 3)
    A = T.array(n, n, n)
    r = T.region(A, scalars=[w, nn, seed])
    T.loop(r, 'libprog_sor3d.so', 'loop_sor3d_18_cuda', A, [(0, n - 1)] * 3, [A, nn, seed])
    for part in ((1, cut), (cut + 1, n - 2)):
        T.loop(r, 'libprog_sor3d.so', 'loop_sor3d_32_cuda', A, [(1, n - 2), (1, n - 2), part], [A, w], reds=[(3, e)], across=[1] * 6)
    T.rt.dvmh_region_end_C(r)
    T.rt.dvmh_get_actual_array2_(A)
    got = T.host(A, (n ** 3,)).copy()
    T.rt.dvmh_delete_object_(A)
    ref = H.oracle_sor3d(n, 1)
    assert H.bits_equal(got, ref['A']) and e.value == ref['eps'][0]
