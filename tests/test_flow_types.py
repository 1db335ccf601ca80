"""ACROSS loops whose axes all depend compile for gfx950, their dataflow
kernels included, for every element type the launch is emitted for."""
import os
import shutil
import subprocess
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(REPO, 'dvm-snapshot-r6603-fork_amd', 'emit'))
import hipgen  # noqa: E402

HIPCC = shutil.which('hipcc') or '/opt/rocm/bin/hipcc'


@pytest.mark.skipif(not os.path.exists(HIPCC), reason='no hipcc')
@pytest.mark.parametrize('ctype', hipgen.FLOW_TYPES)
def test_compiles(tmp_path, ctype):
    loops = [{'name': f'loop_{r}', 'vars': [(v, 'int') for v in 'ijk'[:r]], 'params': [('array', 'X', ctype, r)], 'batch': r == 3,
              'reductions': [('max', 'm', ctype)], 'across': {'array': 'X', 'widths': [(1, 1)] * r},
              'body': {2: 'X[i][j] = (X[i - 1][j] + X[i][j - 1] + X[i + 1][j] + X[i][j + 1]) / 4;\nm = Max(m, X[i][j]);',
                       3: 'X[i][j][k] = (X[i - 1][j][k] + X[i][j - 1][k] + X[i][j][k + 1]) / 3;\nm = Max(m, X[i][j][k]);'}[r]} for r in (2, 3)]
    assert all(hipgen.Loop(d, 't').flow_eligible() for d in loops)
    spec = tmp_path / 'types.loops'
    spec.write_text(repr({'program': 'types', 'include': 'dvmh_prog_common.h', 'loops': loops}))
    subprocess.run([sys.executable, hipgen.__file__, str(spec), str(tmp_path)], check=True)
    # (the lines that keep the arithmetic as written do not matter here: -O1)
    p = subprocess.run([HIPCC, '--offload-arch=gfx950', '--cuda-device-only', '-S', '-O1', '-std=c++17', '-Xclang', '-target-feature', '-Xclang',
                        '-packed-fp32-ops', f'-I{REPO}/include',
                        f'-I{REPO}/dvm-snapshot-r6603-fork_amd/programs', str(tmp_path / 'types_hip.hip'), '-o', str(tmp_path / 'types.s')],
                       capture_output=True, text=True)
    assert p.returncode == 0, p.stderr[-2000:]
