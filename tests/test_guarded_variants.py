"""Variants that load ahead (LDS march, fused pairs, staged line sweeps), asked
for by the tuner or a batch, on bodies that guard an access to a neighbour:
they run only where every load stays inside the array.  (HIP calls faked: what
is checked is which kernel the handler launches.)"""
import os
import sys

import pytest

import fake_device

sys.path.insert(0, os.path.join(fake_device.PKG, 'emit'))
import hipgen  # noqa: E402

CODE = '''
import ast, ctypes, os
spec = ast.literal_eval(open(os.path.join(T.PKG, 'gen', 'cdv', 'branches_cdv.loops')).read().split('\\n', 1)[1])
def named(text):
    return [l['name'] for l in spec['loops'] if text in l['body']][0]
def force(kind, block, **tune):
    t = [1, 0, 0, 0, 0, 0, 0, 0]
    for k, v in tune.items():
        t[dict(variant=2, chunk=3, a=4, b=5)[k]] = v
    T.rt.dvmh_amd_tuner_force_C(T.L(kind), (T.L * 3)(*block), (T.L * 8)(*t))
lib = 'libcdv_branches.so'
'''


def test_line_sweep():
    fake_device.run(CODE + '''
c = ctypes.c_double(0.2)
A = T.array(40, 40, 40)
name = named('A[i][j][k] = A[i][j][k] + c * A[i][j][k - 1];')
for variant, kernel in ((3, 'lvec'), (1, 'ltile')):
    force(1, (64, 1, 1), variant=variant, a=16, b=1)
    for first, staged in ((0, False), (1, True)):
        r = T.region(A, scalars=[c])
        F.fake_clear()
        T.loop(r, lib, name + '_cuda', A, [(0, 39), (0, 39), (first, 39)], [A, c], across=[0, 0, 0, 0, 1, 0])
        T.rt.dvmh_region_end_C(r)
        got = [n for n, _, _ in T.launches()]
        assert any(kernel in n for n in got) == staged and any('line2' in n for n in got) != staged, (variant, first, got)
''')


def test_march_and_pair():
    fake_device.run(CODE + '''
A, B = T.array(300, 300), T.array(300, 300)
n = T.L(300)
step, copy = named('t += j < n - 1'), named('A[i][j] = B[i][j];')
def loops(lo, hi):
    r = T.region(A, B, scalars=[n])
    for k, (name, base, params) in enumerate(((step, B, [A, n, B]), (copy, A, [A, B]))):
        T.loop(r, lib, name + '_cuda', base, [(lo, hi)] * 2, params, line=10 + k)
    T.rt.dvmh_region_end_C(r)
    return [x for x, _, _ in T.launches()]
force(3, (256, 1, 1), variant=1, a=4, chunk=8)
for lo, hi, ahead in ((0, 299, False), (1, 299, False), (0, 298, False), (1, 298, True)):
    F.fake_clear()
    got = loops(lo, hi)
    assert any('march' in x for x in got) == ahead, (lo, hi, got)
    F.fake_clear()
    T.rt.dvmh_amd_batch_begin_C()
    loops(lo, hi)
    T.rt.dvmh_amd_batch_end_C()
    got = [x for x, _, _ in T.launches()]
    assert any('pair_kernel' in x for x in got) == ahead, (lo, hi, got)
''')


def _emit(tmp_path, body, **more):
    d = {'name': 'loop_g', 'vars': [('i', 'int'), ('j', 'int')], 'params': [('array', 'A', 'double', 2), ('array', 'B', 'double', 2)],
         'body': body}
    d.update(more)
    return hipgen.gpu_loop(hipgen.Loop(d, 'g'))


@pytest.mark.parametrize('guard', [True, False])
def test_batch_and_register_sweep(tmp_path, guard):
    """As emitted: a batch's march tiles, the register-staged sweep."""
    access = 'if (i > 0) B[i][j] = A[i - 1][j];' if guard else 'B[i][j] = A[i - 1][j];'
    text = _emit(tmp_path, access, stencil=['A'], batch=True)
    assert ('if (bvariant == 1 && !(dvmh_amd_loop_reads_inside_C(lr, hdr, ' in text) == guard
    assert ('(nonunit || wide || outside)' in text) == guard
    sweep = 'if (i > 0) A[i][j] = A[i][j] + A[i - 1][j];' if guard else 'A[i][j] = A[i][j] + A[i - 1][j];'
    text = _emit(tmp_path, sweep, across={'array': 'A', 'widths': [(1, 0), (0, 0)]})
    assert ('if (lreg && !(dvmh_amd_loop_reads_inside_C(loop_ref, A_hdr, ' in text) == guard


def test_tiled_wavefront():
    """Three dependent axes: what the dataflow launch does not take (values that
    pass through a second array, guarded accesses) keeps the tiles of a tuned loop."""
    fake_device.run(CODE + '''
w, e, n = ctypes.c_double(0.5), ctypes.c_double(), T.L(40)
A, B = T.array(40, 40, 40), T.array(40, 40, 40)
def kernels(text, lo, hi, params, reds=()):
    r = T.region(A, B, scalars=[w, n])
    F.fake_clear()
    T.loop(r, lib, named(text) + '_cuda', A, [(lo, hi)] * 3, params, reds=reds, across=[1] * 6)
    T.rt.dvmh_region_end_C(r)
    return {k for k in ('flow', 'tile', 'wave012') for x, _, _ in T.launches() if k + '_kernel' in x}
two = 'B[i][j][k] = 0.5 * B[i - 1][j][k]'
for tuned in (False, True):
    if tuned:
        force(2, (256, 1, 1), variant=1, a=8, b=8)
    other = {'tile' if tuned else 'wave012'}
    assert kernels(two, 1, 38, [A, B, w], [(3, e)]) == other
    assert kernels('if (i > 0 && j > 0 && k > 0)', 1, 38, [A]) == other
    assert kernels('if (i > 0 && j > 0 && k > 0)', 0, 38, [A]) == {'wave012'}
    assert kernels('if (i < n - 1)', 0, 39, [A, n, w]) == {'wave012'}
    assert kernels('double d = fabs(t - s);', 1, 38, [A, w], [(3, e)]) == {'flow'}
''')
