"""Runs pieces of Python in a child process whose HIP calls go to
tests/fake_hip.cpp: what the runtime and the emitted handlers decide on the
host (which kernels, which shapes, which memory) without a GPU.  In the child,
`import fake_device as T` gives the counters of the fake (T.F) and small
wrappers of the DVMH C interface (which work on a real device as well)."""
import ctypes
import functools
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
PKG = os.path.join(REPO, 'dvm-snapshot-r6603-fork_amd')
if PKG not in sys.path:
    sys.path.insert(0, PKG)
L = ctypes.c_long
INOUT, CUDA, INT_DOUBLE = L(3), L(2), 4


@functools.lru_cache(None)
def _library():
    out = os.path.join(tempfile.mkdtemp(prefix='fake_hip_'), 'libfake_hip.so')
    subprocess.run(['g++', '-O1', '-shared', '-fPIC', '-std=c++17', '-w', '-D__HIP_PLATFORM_AMD__', '-I/opt/rocm/include',
                    os.path.join(HERE, 'fake_hip.cpp'), '-o', out, '-ldl'], check=True)
    return out


def run(code, timeout=120, **env):
    """The child's standard output; its failure is the caller's."""
    pre = f'import sys; sys.path[:0] = [{HERE!r}, {PKG!r}]\nimport fake_device as T\nF = T.F\n'
    p = subprocess.run([sys.executable, '-c', pre + code], env=dict(os.environ, FAKE_HIP=_library(), **env), capture_output=True,
                       text=True, timeout=timeout)
    assert p.returncode == 0, (p.stdout + p.stderr)[-3000:]
    return p.stdout


if 'FAKE_HIP' in os.environ:
    F = ctypes.CDLL(os.environ['FAKE_HIP'], mode=ctypes.RTLD_GLOBAL)
    F.fake_launch_name.restype = ctypes.c_char_p
    for _n in ('capacity', 'used', 'refused', 'asked', 'syncs', 'graphs', 'launches', 'launch_grid', 'launch_block'):
        getattr(F, 'fake_' + _n).restype = L
    F.fake_capacity.argtypes = F.fake_launch_name.argtypes = F.fake_launch_grid.argtypes = F.fake_launch_block.argtypes = [L]
    F.fake_live.argtypes = [ctypes.c_void_p]

import dvmh_amd as D  # noqa: E402  (behind the fake)

rt = D.runtime()
for _n in ('dvmh_region_create_C', 'dvmh_loop_create_C', 'dvmh_handler_func_C', 'dvmh_alignment_linear_C', 'dvmh_distribution_block_C'):
    getattr(rt, _n).restype = L
rt.dvmh_get_natural_base_C.restype = rt.dvmh_get_device_addr_C.restype = ctypes.c_void_p
rt.dvmh_init_lib_C(0)


def array(*dims, rt_type=INT_DOUBLE):
    hdr = (L * 64)()
    args = []
    for n in dims:
        args += [L(n), L(1), L(1)]
    rt.dvmh_array_create_C(hdr, L(len(dims)), L(-rt_type), *args)
    rt.dvmh_distribute_C(hdr, L(len(dims)), *[L(rt.dvmh_distribution_block_C(L(a + 1))) for a in range(len(dims))])
    return hdr


def region(*arrays, scalars=(), flags=0):
    r = L(rt.dvmh_region_create_C(L(flags)))
    for a in arrays:
        rt.dvmh_region_register_array_C(r, INOUT, a, b'a')
    for v in scalars:
        rt.dvmh_region_register_scalar_C(r, L(1), ctypes.byref(v), L(ctypes.sizeof(v)), b's')
    rt.dvmh_region_execute_on_targets_C(r, L(3))
    return r


def loop(r, lib, handler, base, ranges, params, reds=(), across=None, chain=None, line=1):
    """One loop of region r, performed; `handler` a name in `lib`, or a ctypes callback."""
    rt.dvmh_line_C(L(line), b'test')
    args = []
    for lo, hi in ranges:
        args += [L(lo), L(hi), L(1)]
    l = L(rt.dvmh_loop_create_C(r, L(len(ranges)), *args))
    rt.dvmh_loop_map_C(l, base, L(len(ranges)), *[L(rt.dvmh_alignment_linear_C(L(a + 1), L(1), L(0))) for a in range(len(ranges))])
    if across:
        rt.dvmh_loop_across_C(l, L(0), base, L(len(ranges)), *[L(w) for w in across])
    for func, v, *loc in reds:   # (values: double)
        rt.dvmh_loop_reduction_C(l, L(func), ctypes.byref(v), L(INT_DOUBLE), L(1), ctypes.byref(loc[0]) if loc else None,
                                 L(ctypes.sizeof(loc[0]) if loc else 0))
    fn = getattr(D.load(lib), handler) if isinstance(handler, str) else handler
    refs = [p if isinstance(p, ctypes.Array) else ctypes.byref(p) for p in params]
    rt.dvmh_loop_register_handler_C(l, CUDA, L(0), L(rt.dvmh_handler_func_C(fn, L(len(refs)), *refs)))
    if chain:
        rt.dvmh_amd_loop_register_chain_handler_C(l, L(rt.dvmh_handler_func_C(getattr(D.load(lib), chain), L(0))))
    rt.dvmh_loop_perform_C(l)


def host(a, shape, ctype=ctypes.c_double):
    """The host copy of array `a`, as numpy sees it."""
    import numpy as np
    return np.ctypeslib.as_array(ctypes.cast(rt.dvmh_get_natural_base_C(L(0), a), ctypes.POINTER(ctype)), shape=shape)


def launches():
    """(kernel, workgroups, threads) since the last fake_clear (the first of them, if very many)."""
    return [(F.fake_launch_name(i).decode(), F.fake_launch_grid(i), F.fake_launch_block(i)) for i in range(min(F.fake_launches(), 4096))]
