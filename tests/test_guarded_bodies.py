"""Bodies that guard an access to a neighbour (the array may end where the loop
does) keep the kernels that read only what an iteration reads: no register
march, no dataflow sweep, and no staged sweep or LDS march that nobody asked
for.  The same bodies without the guard take them."""
import os
import subprocess
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPGEN = os.path.join(REPO, 'dvm-snapshot-r6603-fork_amd', 'emit', 'hipgen.py')

V = [('i', 'int'), ('j', 'int'), ('k', 'int')]
PLAIN = 'B[i][j][k] = A[i][j][k] + A[i - 1][j][k];\n'
SWEEP = 'A[i][j][k] = A[i][j][k] + A[i - 1][j][k] + A[i][j - 1][k] + A[i][j][k - 1];\n'
LINE = 'A[i][j][k] = A[i][j][k] + A[i - 1][j][k];\n'
GUARDS = ['if (i > 0) { %s }\n', 'for (int q = 0; q < i; q++) { %s }\n', 'SELECT(i > 0, A[i][j][k]);\n %s']


def _emit(tmp_path, guard):
    g = (lambda s: guard % s) if guard else (lambda s: s)
    A, B = ('array', 'A', 'double', 3), ('array', 'B', 'double', 3)
    loops = [{'name': 'loop_st', 'vars': V, 'params': [A, B], 'stencil': ['A'], 'body': g(PLAIN)},
             {'name': 'loop_all', 'vars': V, 'params': [A], 'across': {'array': 'A', 'widths': [(1, 0)] * 3}, 'body': g(SWEEP)},
             {'name': 'loop_line', 'vars': V, 'params': [A], 'across': {'array': 'A', 'widths': [(1, 0), (0, 0), (0, 0)]}, 'body': g(LINE)}]
    spec = tmp_path / 'guard.loops'
    spec.write_text(repr({'program': 'guard', 'loops': loops}))
    subprocess.run([sys.executable, HIPGEN, str(spec), str(tmp_path)], check=True)
    return (tmp_path / 'guard_hip.hip').read_text()


@pytest.mark.parametrize('guard', [None] + GUARDS)
def test_guarded(tmp_path, guard):
    text = _emit(tmp_path, guard)
    free = guard is None
    assert ('loop_st_star_kernel' in text) == free
    assert ('loop_all_flow_kernel' in text) == free
    line = text[text.index('void loop_line_cuda('):]
    assert ('tune[DVMH_AMD_T_OWN] && A_tfm' in line) == free
    stencil = text[text.index('void loop_st_cuda('):text.index('void loop_all_cuda(')]
    assert ('280L * 280 * 280' in stencil) == free
