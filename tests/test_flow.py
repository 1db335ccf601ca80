"""ACROSS loops whose axes all depend, run as one dataflow launch: grids of one
tile, of tiles the grid fills and does not fill, rows shorter than a block of
eight steps and just over one; repeated as a replayed graph; and past the point
where the launch tags run out.  Every point must equal the sequential sweep's."""
import os
import subprocess
import sys

import numpy as np
import pytest

import dvmh_amd as D
import helpers as H
from test_cdvmh import _check_relax2d

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, 'dvm-snapshot-r6603-fork_amd')


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
