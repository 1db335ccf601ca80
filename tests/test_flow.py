"""ACROSS loops whose axes all depend, run as one dataflow launch: grids of one
tile, of tiles the grid fills and does not fill, rows shorter than a block of
eight steps and just over one; repeated as a replayed graph; and past the point
where the launch tags run out.  Every point must equal the sequential sweep's."""
import os
import re
import subprocess
import sys

import numpy as np
import pytest

import dvmh_amd as D
import helpers as H
from test_cdvmh import _check_relax2d

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, 'dvm-snapshot-r6603-fork_amd')
sys.path.insert(0, os.path.join(PKG, 'emit'))
import hipgen  # noqa: E402


@pytest.mark.gpu
@pytest.mark.parametrize('n', [3, 4, 9, 10, 11, 17, 18, 19, 26, 35, 66, 101])
def test_three_axes(n):
    res, ref = H.run_sor3d(n, 3), H.oracle_sor3d(n, 3)
    assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps'])


@pytest.mark.gpu
@pytest.mark.parametrize('n', [3, 9, 10, 11, 65, 66, 67, 130, 131])
def test_two_axes(n):
    _check_relax2d(n, 3)


@pytest.mark.gpu
@pytest.mark.parametrize('n,sweeps,group', [(12, 130, 130), (19, 65, 65), (26, 64, 64)])
def test_chains_longer_than_a_launch(n, sweeps, group):
    res, ref = H.run_sor3d_chain(n, sweeps, group), H.oracle_sor3d(n, sweeps)
    assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps'])


@pytest.mark.gpu
def test_replayed_as_a_graph():
    r = D.runtime()
    r.dvmh_amd_set_graph_C(1)
    r.dvmh_amd_set_graph_min_nodes_C(1)
    replays = D.stats()['graph_replays']
    try:
        res = H.run_sor3d(43, 8, flags=D.REGION_AMD_GRAPH)
    finally:
        r.dvmh_amd_set_graph_min_nodes_C(-1)
        r.dvmh_amd_set_graph_C(0)
    ref = H.oracle_sor3d(43, 8)
    assert D.stats()['graph_replays'] - replays >= 6
    assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps'])


CHILD = f'''
import sys
sys.path[:0] = [{PKG!r}, {os.path.join(REPO, 'tests')!r}]
import numpy as np
import helpers as H
for n in (20, 43, 20):
    res, ref = H.run_sor3d(n, 6), H.oracle_sor3d(n, 6)
    assert H.bits_equal(res['A'], ref['A']) and np.array_equal(res['eps'], ref['eps']), n
print('equal')
'''


@pytest.mark.gpu
def test_tags_start_over():
    env = dict(os.environ, DVMH_AMD_FLOW_TAG=str((1 << 31) - 4))
    p = subprocess.run([sys.executable, '-c', CHILD], env=env, capture_output=True, text=True, timeout=100)
    assert p.returncode == 0 and p.stdout.strip().endswith('equal'), p.stderr[-2000:]


RELAX = 't = 0.25 * (X[i - 1][j] + X[i + 1][j] + X[i][j - 1] + X[i][j + 1]);\nX[i][j] = t;'
FORMS = [   # body after RELAX, further loop entries, runs as a dataflow launch
    ('', {}, True),
    ('Y[i][j] = t;', {}, True),                                  # another array at the loop point
    ('Y[i][j] += X[i - 1][j];', {}, True),
    ('t = Y[i - 1][j];', {}, True),                              # read anywhere
    ('Y[i][j] = Y[i - 1][j] + t;', {}, False),                   # passes between points
    ('Y[i - 1][j] = t;', {}, False),
    ('Y[j][i] = t;', {}, False),
    ('f(Y, t);', {}, False),
    ('X[i][j - 1] = t;', {}, False),                             # writes off the point
    ('t = X[i - 1][j - 1];', {}, False),                         # two offsets
    ('t = X[i - 2][j];', {}, False),
    ('g(&X[i][j]);', {}, False),
    ('X[i][j]++;', {}, True),
    ('w = t;', {}, False),                                       # assigns a scalar
    ('t = w == t;', {}, True),
    ('r = Max(r, t);', {'reductions': [('max', 'r', 'double')]}, True),
    ('r[i % 3] += t;', {'reductions': [('sum', 'r', 'double')], 'reduction_lengths': {'r': 3}}, True),
    ('', {'across': {'array': 'X', 'widths': [(1, 1), (2, 1)]}}, False),
    ('', {'across': {'array': 'X', 'widths': [(1, 1), (0, 0)]}}, False),
    ('', {'across': {'array': 'X', 'widths': [(1, 0), (0, 1)]}}, True),
]


@pytest.mark.parametrize('more,entries,flow', FORMS)
def test_which_loops_run_as_a_launch(more, entries, flow):
    """What the workgroups of the launch do not pass to each other keeps a loop
    on the hyperplane kernels, which every form still has."""
    d = {'name': 'loop_t', 'vars': [('i', 'int'), ('j', 'int')], 'steps': ['1', '1'], 'privates': ['double t'],
         'params': [('array', 'X', 'double', 2), ('array', 'Y', 'double', 2), ('scalar', 'w', 'double')],
         'across': {'array': 'X', 'widths': [(1, 1), (1, 1)]}, 'body': RELAX + '\n' + more}
    d.update(entries)
    L = hipgen.Loop(d, 't')
    assert L.flow_eligible() == flow
    text = hipgen.gpu_loop(L)
    assert ('loop_t_flow_kernel' in text) == flow
    assert re.search(r'loop_t_wave01_kernel', text)
