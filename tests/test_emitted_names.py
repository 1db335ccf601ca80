"""Emitted kernels and handlers use names a program may use too: a stencil, a
MAXLOC loop and line sweeps whose arrays and scalars carry short names (C, R, w,
c, star, walk, ..) must compile, and no name of the emitter may hide one of the
program's (which -Wshadow would report)."""
import os
import shutil
import subprocess
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, 'dvm-snapshot-r6603-fork_amd')
HIPCC = shutil.which('hipcc') or '/opt/rocm/bin/hipcc'

NAMES = [('C', 'R', 'w'), ('star', 'walk', 'c'), ('NT', 'parts', 'wave'), ('w1', 'tiles', 'fill'), ('own', 'cur', 'to'), ('nxt', 'col', 'm')]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason='no hipcc')
@pytest.mark.parametrize('A,B,s', NAMES)
def test_names(tmp_path, A, B, s):
    star = f'{B}[i][j][k] = {s} * ({A}[i - 1][j][k] + {A}[i + 1][j][k] + {A}[i][j - 1][k] + {A}[i][j][k + 1]);\n'
    loc = f'if (fabs({A}[i][j][k]) * {s} > mx) {{ mx = fabs({A}[i][j][k]) * {s}; loc = k; }}\n'
    v = [('i', 'int'), ('j', 'int'), ('k', 'int')]
    arr = [('array', A, 'double', 3), ('array', B, 'double', 3), ('scalar', s, 'double')]
    loops = [{'name': 'loop_st', 'vars': v, 'params': arr, 'stencil': [A], 'body': star},
             {'name': 'loop_loc', 'vars': v, 'params': [arr[0], arr[2]], 'reductions': [('maxloc', 'mx', 'double', 'loc', 'long')], 'body': loc},
             {'name': 'loop_line', 'vars': v, 'params': [arr[0], arr[2]], 'across': {'array': A, 'widths': [(1, 0), (0, 0), (0, 0)]},
              'body': f'{A}[i][j][k] = {A}[i][j][k] + {s} * {A}[i - 1][j][k];\n'}]
    spec = tmp_path / 'names.loops'
    spec.write_text(repr({'program': 'names', 'loops': loops}))
    subprocess.run([sys.executable, os.path.join(PKG, 'emit', 'hipgen.py'), str(spec), str(tmp_path)], check=True)
    text = (tmp_path / 'names_hip.hip').read_text()
    assert 'loop_st_star_kernel' in text
    res = subprocess.run([HIPCC, '--offload-arch=gfx950', '--cuda-device-only', '-fsyntax-only', '-std=c++17', '-Wshadow',
                          f'-I{REPO}/include', str(tmp_path / 'names_hip.hip')], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-3000:]
    hidden = [ln for ln in res.stderr.split('\n') if 'names_hip.hip' in ln and 'shadows' in ln and any(f"'{n}'" in ln for n in (A, B, s))]
    assert not hidden, hidden
