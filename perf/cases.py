"""The work a C-DVMH program has this runtime do, as timed cases.

Every case is one stretch of a converted program: its distributed arrays, its
regions and its parallel loops, described to libdvmh_amd through the DVMH C
interface and run by the handlers emitted for that program (the calls a
converted program makes, one by one).  A pass is a few iterations of the
program's time loop, with the get_actual of every iteration's reduction
variables that the program itself does.  Outputs are the arrays' device copies
and the reduction values of every iteration.

Two forms, as programs are run:
  plain   no setting touched: default launch configuration, results
          synchronised after every loop
  model   the cost model picks configurations, results are synchronised only
          where they are needed, repeating regions and batches become graphs
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'dvm-snapshot-r6603-fork_amd')
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import dvmh_amd as D  # noqa: E402
from dvmh_amd import costmodel as CM  # noqa: E402

_L = ctypes.c_long
_CUDA = _L(2)                       # DEVICE_TYPE_CUDA
_INT_FLOAT, _INT_DOUBLE = 3, 4      # rt_FLOAT, rt_DOUBLE
_MAX, _MIN, _SUM, _MAXLOC = 3, 4, 1, 11
_IN, _OUT, _INOUT = _L(1), _L(2), _L(3)
_TARGETS = _L(3)                    # host or GPU, as converted programs say


# ----------------------------------------------------------------- the cases
def listed():
    return [
        # a small 3-D grid, one of many in a parameter study: launches and the
        # read of each iteration's residual are all there is
        {'name': 'jac3d small', 'kind': 'jac3d', 'form': 'model', 'n0': 34, 'n1': 34, 'n2': 34, 'iters': 20},
        # the benchmark's 3-D Jacobi, MAX and SUM every iteration
        {'name': 'jac3d 384', 'kind': 'jac3d', 'form': 'model', 'n0': 384, 'n1': 384, 'n2': 384, 'iters': 10},
        # a grid of uneven sides in a program that sets nothing
        {'name': 'jac3d uneven plain', 'kind': 'jac3d', 'form': 'plain', 'n0': 201, 'n1': 187, 'n2': 239, 'iters': 10},
        # the FP32 3-D Jacobi benchmark's loops (MAX and copy, then stencil)
        {'name': 'jac3d fp32', 'kind': 'jac3f', 'form': 'model', 'n0': 320, 'n1': 320, 'n2': 320, 'iters': 8},
        # the benchmark's 2-D Jacobi: stencil, then copy and MAX, in one region
        {'name': 'jac2d 2048', 'kind': 'jac2d', 'form': 'model', 'n0': 2048, 'n1': 2048, 'iters': 20},
        # Gaussian elimination, a whole program from allocation to solution:
        # a region per pivot row, loops that shrink
        {'name': 'gauss 500', 'kind': 'gauss', 'form': 'plain', 'n0': 500},
        # 3-D over-relaxation, one sweep at a time (its residual decides on the next)
        {'name': 'sor3d 130', 'kind': 'sor3d', 'form': 'model', 'n0': 130, 'n1': 130, 'n2': 130, 'iters': 4},
        # the benchmark's 320^3 over-relaxation, ten sweeps between residuals
        {'name': 'sor3d chain 320', 'kind': 'sor3dchain', 'form': 'model', 'n0': 320, 'n1': 320, 'n2': 320, 'iters': 10},
        # the benchmark's line sweeps along every axis, both directions, MAXLOC
        {'name': 'adi3d 256', 'kind': 'adi3d', 'form': 'model', 'n0': 256, 'n1': 256, 'n2': 256, 'iters': 5},
        # the same program on a small uneven grid, nothing set
        {'name': 'adi3d uneven plain', 'kind': 'adi3d', 'form': 'plain', 'n0': 65, 'n1': 131, 'n2': 99, 'iters': 5},
        # 2-D over-relaxation (ACROSS on both axes), MAX and MIN
        {'name': 'relax2d 1000', 'kind': 'relax2d', 'form': 'plain', 'n0': 1000, 'n1': 1000, 'iters': 4},
        # many independent 2-D grids of uneven sides advanced together
        {'name': 'batched grids', 'kind': 'batched', 'form': 'model', 'count': 24, 'lo': 64, 'hi': 1024, 'iters': 8},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """A case of the listed kinds: sides spread over the logarithm of their
    range, each axis its own."""
    kind = rng.choice(['jac3d', 'jac3d', 'jac3f', 'jac2d', 'gauss', 'sor3d', 'sor3dchain', 'adi3d', 'relax2d', 'batched'])
    form = rng.choice(['model', 'plain'])
    rank, lo, hi = {'jac3d': (3, 16, 380), 'jac3f': (3, 16, 320), 'jac2d': (2, 64, 2048), 'gauss': (1, 24, 500),
                    'sor3d': (3, 12, 130), 'sor3dchain': (3, 32, 320), 'adi3d': (3, 16, 256), 'relax2d': (2, 32, 1000),
                    'batched': (0, 32, 512)}[kind]
    if kind == 'batched':
        small = int(_log_uniform(rng, lo, hi))
        return {'kind': kind, 'form': 'model', 'count': rng.randint(3, 24), 'lo': small,
                'hi': min(1024, small + rng.randint(1, 2 * small)), 'iters': 8}
    side = _log_uniform(rng, lo, hi)
    case = {'kind': kind, 'form': 'plain' if kind == 'gauss' else 'model' if kind == 'sor3dchain' else form}
    for a in range(rank):
        case['n%d' % a] = max(lo, min(hi, round(side * rng.uniform(0.75, 1.25))))
    if kind != 'gauss':
        case['iters'] = {'jac3d': 10, 'jac3f': 8, 'jac2d': 10, 'sor3d': 3, 'sor3dchain': rng.randint(4, 10), 'adi3d': 5,
                         'relax2d': 3}[kind]
    return case


def _sides(case):
    """Sides of the batched grids: evenly spread over lo..hi, then shuffled
    (small and large grids meet in one batch)."""
    c, lo, hi = case['count'], case['lo'], case['hi']
    order = np.random.RandomState(c).permutation(c)
    return [int(lo + (hi - lo) * q // max(1, c - 1)) for q in order]


def _dims(case):
    return [case['n%d' % a] for a in range(3) if 'n%d' % a in case]


def work(case):
    """Bytes: each loop's arrays read once and written once, per iteration (the
    arrays of a step that may run as one pass once for the step; the six line
    sweeps two by two, forward and back along one axis)."""
    kind, it = case['kind'], case.get('iters', 1)
    if kind == 'gauss':
        # the trailing matrix is read and written for every pivot
        n = case['n0']
        pts = sum((n - 1 - i) * (n - i) for i in range(n - 1))
        return {'bytes': 8 * n * (n + 1) * 2 + 16 * pts, 'flops': 3 * pts}
    if kind == 'batched':
        pts = sum((s - 2) ** 2 for s in _sides(case))
        return {'bytes': 24 * pts * it, 'flops': 6 * pts * it}
    d = _dims(case)
    inner = math.prod(x - 2 for x in d)
    full = math.prod(d)
    if kind == 'adi3d':
        return {'bytes': (8 + it * 3 * 16) * full, 'flops': 12 * full * it}
    per_pt, fl = {'jac3d': (16, 10), 'jac3f': (12, 9), 'jac2d': (24, 6), 'sor3d': (16, 12), 'sor3dchain': (16, 12),
                  'relax2d': (16, 10)}[kind]
    return {'bytes': per_pt * inner * it, 'flops': fl * inner * it}


# ------------------------------------------------ the converted programs' calls
_rt = None
_fns = {}


def _runtime():
    global _rt
    if _rt is None:
        _rt = CM.rt()
        for name in ('dvmh_region_create_C', 'dvmh_loop_create_C', 'dvmh_alignment_linear_C', 'dvmh_handler_func_C',
                     'dvmh_distribution_block_C'):
            getattr(_rt, name).restype = _L
        _rt.dvmh_get_natural_base_C.restype = ctypes.c_void_p
        _rt.dvmh_init_lib_C(0)
        CM.rt().dvmh_amd_model_load_C(CM.MODEL.encode())
    return _rt


def _fn(lib, name):
    if name not in _fns:
        _fns[name] = getattr(D.load(lib), name)
    return _fns[name]


def _set_form(form):
    rt = _runtime()
    model = form == 'model'
    rt.dvmh_amd_tuner_set_mode_C(2 if model else 0)
    rt.dvmh_amd_tuner_set_repeats_C(_L(2))
    rt.dvmh_amd_set_sync_mode_C(_L(1 if model else 0))
    rt.dvmh_amd_set_graph_C(1 if model else 0)


class _DeviceCopy:
    """The device copy of a distributed array, as an object torch can wrap."""

    def __init__(self, array):
        self.array = array   # keeps the array alive
        ptr = _runtime().dvmh_get_natural_base_C(_L(1), array.hdr)
        self.__cuda_array_interface__ = {'shape': tuple(array.dims), 'typestr': '<f%d' % array.size, 'data': (ptr, False),
                                         'version': 2}


class _Array:
    def __init__(self, dims, rt_type=_INT_DOUBLE):
        rt = _runtime()
        self.dims, self.size = list(dims), 4 if rt_type == _INT_FLOAT else 8
        self.hdr = (_L * 64)()
        args = []
        for x in dims:
            args += [_L(x), _L(1), _L(1)]
        rt.dvmh_array_create_C(self.hdr, _L(len(dims)), _L(-rt_type), *args)
        rt.dvmh_distribute_C(self.hdr, _L(len(dims)), *[_L(rt.dvmh_distribution_block_C(_L(a + 1))) for a in range(len(dims))])

    def __del__(self):
        _rt.dvmh_delete_object_(self.hdr)

    def host(self):
        ptr = _rt.dvmh_get_natural_base_C(_L(0), self.hdr)
        t = ctypes.c_float if self.size == 4 else ctypes.c_double
        return np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(t)), shape=tuple(self.dims))

    def device(self):
        return torch.as_tensor(_DeviceCopy(self), device='cuda')


class _Region:
    def __init__(self, arrays, scalars=(), flags=0):
        self.arrays = [(_INOUT if len(a) == 1 else a[1], a[0].hdr) for a in arrays]
        self.scalars = [(ctypes.byref(v), _L(ctypes.sizeof(v))) for v in scalars]
        self.flags = _L(flags)

    def begin(self):
        r = _L(_rt.dvmh_region_create_C(self.flags))
        for intent, hdr in self.arrays:
            _rt.dvmh_region_register_array_C(r, intent, hdr, b'a')
        for ref, size in self.scalars:
            _rt.dvmh_region_register_scalar_C(r, _IN, ref, size, b's')
        _rt.dvmh_region_execute_on_targets_C(r, _TARGETS)
        return r


class _Loop:
    """One parallel loop: the calls between its dvmh_line_C and its
    dvmh_loop_perform_C."""

    def __init__(self, lib, file, line, handler, base, ranges, params, reds=(), across=None, batch=None, chain=None, block=None):
        self.file, self.line = file, _L(line)
        rank = len(ranges)
        self.create = [_L(rank)]
        for lo, hi, step in ranges:
            self.create += [_L(lo), _L(hi), _L(step)]
        self.base, self.rank = base.hdr, _L(rank)
        self.axes = [(_L(a + 1), _L(1), _L(0)) for a in range(rank)]
        self.handler = (_fn(lib, handler + '_cuda'), _L(len(params)), *[p.hdr if isinstance(p, _Array) else ctypes.byref(p) for p in params])
        self.reds = list(reds)
        self.across = None if across is None else (_L(0), base.hdr, _L(rank), *[_L(w) for w in across])
        self.batch = None if batch is None else _fn(lib, batch)
        self.chain = None if chain is None else _fn(lib, chain)
        self.block = None if block is None else [_L(b) for b in block]

    def perform(self, region, reds=None):
        rt = _rt
        rt.dvmh_line_C(self.line, self.file)
        l = _L(rt.dvmh_loop_create_C(region, *self.create))
        rt.dvmh_loop_map_C(l, self.base, self.rank, *[_L(rt.dvmh_alignment_linear_C(*a)) for a in self.axes])
        if self.block is not None:
            rt.dvmh_loop_set_cuda_block_C(l, *self.block)
        if self.across is not None:
            rt.dvmh_loop_across_C(l, *self.across)
        for r in self.reds if reds is None else reds:
            rt.dvmh_loop_reduction_C(l, *r)
        rt.dvmh_loop_register_handler_C(l, _CUDA, _L(0), _L(rt.dvmh_handler_func_C(*self.handler)))
        if self.batch is not None:
            rt.dvmh_amd_loop_register_batch_handler_C(l, _L(rt.dvmh_handler_func_C(self.batch, _L(0))))
        if self.chain is not None:
            rt.dvmh_amd_loop_register_chain_handler_C(l, _L(rt.dvmh_handler_func_C(self.chain, _L(0))))
        rt.dvmh_loop_perform_C(l)


def _red(func, var, rt_type=_INT_DOUBLE, loc=None):
    return (_L(func), ctypes.byref(var), _L(rt_type), _L(1), ctypes.byref(loc) if loc is not None else None,
            _L(ctypes.sizeof(loc) if loc is not None else 0))


def _full(dims):
    return [(0, n - 1, 1) for n in dims]


def _interior(dims):
    return [(1, n - 2, 1) for n in dims]


def _run_region(region, *loops):
    r = region.begin()
    for l in loops:
        l.perform(r)
    _rt.dvmh_region_end_C(r)


# ----------------------------------------------------------- the programs' states
class _Jac3d:
    def __init__(self, case, seed):
        dims = _dims(case)
        self.iters = case['iters']
        self.A, self.B = _Array(dims), _Array(dims)
        self.n, self.seed = _L(max(dims)), ctypes.c_ulonglong(seed)
        _run_region(_Region([(self.A, _OUT), (self.B, _OUT)], [self.n, self.seed]),
                    _Loop('libprog_jac3d.so', b'jac3d.cdv', 21, 'loop_jac3d_21', self.A, _full(dims), [self.A, self.B, self.n, self.seed]))
        self.eps, self.s = ctypes.c_double(), ctypes.c_double()
        reds = [_red(_MAX, self.eps), _red(_SUM, self.s)]
        self.region = _Region([(self.A,), (self.B,)])
        self.loops = [_Loop('libprog_jac3d.so', b'jac3d.cdv', 41, 'loop_jac3d_41', self.B, _interior(dims), [self.A, self.B], reds),
                      _Loop('libprog_jac3d.so', b'jac3d.cdv', 54, 'loop_jac3d_54', self.A, _interior(dims), [self.A, self.B], reds)]
        self.done = 0

    def run(self):
        rt = _rt
        eps, s = ctypes.byref(self.eps), ctypes.byref(self.s)
        hist = np.empty((self.iters, 2))
        for it in range(self.iters):
            self.eps.value = self.s.value = 0.0
            rt.dvmh_actual_variable2_(eps)
            rt.dvmh_actual_variable2_(s)
            r = self.region.begin()
            rt.dvmh_shadow_renew_C((self.B if self.done % 2 else self.A).hdr, _L(0), _L(0))
            self.loops[self.done % 2].perform(r)
            rt.dvmh_region_end_C(r)
            rt.dvmh_get_actual_variable2_(eps)
            rt.dvmh_get_actual_variable2_(s)
            hist[it] = self.eps.value, self.s.value
            self.done += 1
        return {'A': self.A.device(), 'B': self.B.device(), 'hist': hist}


def _float_grid(dims, seed):
    """4 + i + j + k, as the FP32 benchmark starts, and a seeded part in [0, 1)."""
    g = torch.Generator().manual_seed(seed)
    x = torch.rand(tuple(dims), generator=g, dtype=torch.float32)
    for a, n in enumerate(dims):
        x += torch.arange(n, dtype=torch.float32).reshape([-1 if b == a else 1 for b in range(len(dims))])
    return x + 4


class _Jac3f:
    def __init__(self, case, seed):
        dims = _dims(case)
        self.iters = case['iters']
        self.A, self.B = _Array(dims, _INT_FLOAT), _Array(dims, _INT_FLOAT)
        self.B.host()[...] = _float_grid(dims, seed).numpy()
        _rt.dvmh_actual_array2_(self.A.hdr)
        _rt.dvmh_actual_array2_(self.B.hdr)
        self.eps = ctypes.c_float()
        self.region = _Region([(self.A,), (self.B,)])
        _run_region(self.region)   # both arrays to the GPU
        self.loops = [_Loop('libprog_jackat.so', b'jac3d_perf.c', 60, 'loop_jac3kat_max', self.A, _interior(dims), [self.A, self.B],
                            [_red(_MAX, self.eps, _INT_FLOAT)]),
                      _Loop('libprog_jackat.so', b'jac3d_perf.c', 72, 'loop_jac3kat_st', self.B, _interior(dims), [self.A, self.B])]

    def run(self):
        rt = _rt
        eps = ctypes.byref(self.eps)
        hist = np.empty(self.iters, dtype=np.float32)
        for it in range(self.iters):
            self.eps.value = 0.0
            rt.dvmh_actual_variable2_(eps)
            r = self.region.begin()
            self.loops[0].perform(r)
            rt.dvmh_shadow_renew_C(self.A.hdr, _L(0), _L(0))
            self.loops[1].perform(r)
            rt.dvmh_region_end_C(r)
            rt.dvmh_get_actual_variable2_(eps)
            hist[it] = self.eps.value
        return {'A': self.A.device(), 'B': self.B.device(), 'hist': hist}


class _Jac2d:
    def __init__(self, case, seed):
        dims = _dims(case)
        self.iters = case['iters']
        self.A, self.B = _Array(dims), _Array(dims)
        self.n, self.seed = _L(max(dims)), ctypes.c_ulonglong(seed)
        lib, file = 'libprog_jac2d.so', b'jac2d.cdv'
        _run_region(_Region([(self.A, _OUT), (self.B, _OUT)], [self.n, self.seed]),
                    _Loop(lib, file, 23, 'loop_jac2d_23', self.A, _full(dims), [self.A, self.B, self.n, self.seed]))
        self.eps = ctypes.c_double()
        self.region = _Region([(self.A,), (self.B,)], flags=D.REGION_AMD_GRAPH if case['form'] == 'model' else 0)
        self.loops = [_Loop(lib, file, 38, 'loop_jac2d_38', self.B, _interior(dims), [self.A, self.B]),
                      _Loop(lib, file, 43, 'loop_jac2d_43', self.A, _interior(dims), [self.A, self.B], [_red(_MAX, self.eps)])]

    def run(self):
        rt = _rt
        eps = ctypes.byref(self.eps)
        hist = np.empty(self.iters)
        for it in range(self.iters):
            self.eps.value = 0.0
            rt.dvmh_actual_variable2_(eps)
            r = self.region.begin()
            rt.dvmh_shadow_renew_C(self.A.hdr, _L(0), _L(0))
            self.loops[0].perform(r)
            self.loops[1].perform(r)
            rt.dvmh_region_end_C(r)
            rt.dvmh_get_actual_variable2_(eps)
            hist[it] = self.eps.value
        return {'A': self.A.device(), 'B': self.B.device(), 'hist': hist}


class _Gauss:
    """The whole program, host arrays in and out."""

    def __init__(self, case, seed):
        self.n, self.seed = case['n0'], seed
        self.wb, self.x, self.out = np.ones(self.n), np.empty(self.n), np.empty((self.n, self.n + 1))
        self.fn = _fn('libcdv_gauss.so', 'gauss')

    def run(self):
        self.fn(_L(self.n), ctypes.c_ulonglong(self.seed), *[ctypes.c_void_p(a.ctypes.data) for a in (self.wb, self.x, self.out)])
        return {'x': self.x, 'out': self.out}


_OMEGA = 1.5


class _Sor3d:
    def __init__(self, case, seed):
        dims = _dims(case)
        self.iters, self.chained = case['iters'], case['kind'] == 'sor3dchain'
        self.A = _Array(dims)
        self.n, self.seed, self.w = _L(max(dims)), ctypes.c_ulonglong(seed), ctypes.c_double(_OMEGA)
        lib, file = 'libprog_sor3d.so', b'sor3d.cdv'
        _run_region(_Region([(self.A, _OUT)], [self.n, self.seed]),
                    _Loop(lib, file, 18, 'loop_sor3d_18', self.A, _full(dims), [self.A, self.n, self.seed]))
        self.eps = [ctypes.c_double() for _ in range(self.iters if self.chained else 1)]
        self.reds = [[_red(_MAX, e)] for e in self.eps]
        graph = case['form'] == 'model' and not self.chained
        self.region = _Region([(self.A,)], [self.w], flags=D.REGION_AMD_GRAPH if graph else 0)
        self.loop = _Loop(lib, file, 32, 'loop_sor3d_32', self.A, _interior(dims), [self.A, self.w], across=[1] * 6,
                          chain='loop_sor3d_32_cuda_chain' if self.chained else None)

    def run(self):
        rt = _rt
        hist = np.empty(self.iters)
        if self.chained:
            rt.dvmh_amd_batch_begin_C()
            for q in range(self.iters):
                self.eps[q].value = 0.0
                r = self.region.begin()
                self.loop.perform(r, self.reds[q])
                rt.dvmh_region_end_C(r)
            rt.dvmh_amd_batch_end_C()
            for q in range(self.iters):
                rt.dvmh_get_actual_variable2_(ctypes.byref(self.eps[q]))
                hist[q] = self.eps[q].value
        else:
            eps = ctypes.byref(self.eps[0])
            for it in range(self.iters):
                self.eps[0].value = 0.0
                rt.dvmh_actual_variable2_(eps)
                r = self.region.begin()
                self.loop.perform(r, self.reds[0])
                rt.dvmh_region_end_C(r)
                rt.dvmh_get_actual_variable2_(eps)
                hist[it] = self.eps[0].value
        return {'A': self.A.device(), 'hist': hist}


_COEF = 0.3


class _Adi3d:
    """A pass is the program from its initial field on (the sweeps amplify)."""

    def __init__(self, case, seed):
        dims = _dims(case)
        self.iters = case['iters']
        self.a = _Array(dims)
        self.n, self.seed, self.c = _L(max(dims)), ctypes.c_ulonglong(seed), ctypes.c_double(_COEF)
        lib, file = 'libprog_adi3d.so', b'adi3d.cdv'
        self.init = (_Region([(self.a, _OUT)], [self.n, self.seed]),
                     _Loop(lib, file, 20, 'loop_adi3d_20', self.a, _full(dims), [self.a, self.n, self.seed]))
        self.mx, self.loc = ctypes.c_double(), _L()
        self.region = _Region([(self.a,)], [self.c, self.n], flags=D.REGION_AMD_GRAPH if case['form'] == 'model' else 0)
        self.loops = []
        for axis in range(3):
            for back in (0, 1):
                ranges, across = _full(dims), [0] * 6
                ranges[axis] = (dims[axis] - 2, 0, -1) if back else (1, dims[axis] - 1, 1)
                across[2 * axis + back] = 1
                line = 34 + 10 * axis + 5 * back
                self.loops.append(_Loop(lib, file, line, 'loop_adi3d_%d' % line, self.a, ranges, [self.a, self.c], across=across))
        self.loops.append(_Loop(lib, file, 64, 'loop_adi3d_64', self.a, _full(dims), [self.a, self.n],
                                [_red(_MAXLOC, self.mx, loc=self.loc)]))
        _run_region(*self.init)

    def run(self):
        rt = _rt
        mx, loc = ctypes.byref(self.mx), ctypes.byref(self.loc)
        hist, locs = np.empty(self.iters), np.empty(self.iters, dtype=np.int64)
        _run_region(*self.init)
        for it in range(self.iters):
            self.mx.value, self.loc.value = -1.0, -1
            rt.dvmh_actual_variable2_(mx)
            rt.dvmh_actual_variable2_(loc)
            _run_region(self.region, *self.loops)
            rt.dvmh_get_actual_variable2_(mx)
            rt.dvmh_get_actual_variable2_(loc)
            hist[it], locs[it] = self.mx.value, self.loc.value
        return {'a': self.a.device(), 'hist': hist, 'loc': locs}


class _Relax2d:
    def __init__(self, case, seed):
        dims = _dims(case)
        self.iters = case['iters']
        self.A = _Array(dims)
        self.n, self.seed, self.w = _L(max(dims)), ctypes.c_ulonglong(seed), ctypes.c_double(_OMEGA)
        lib, file = 'libcdv_relax2d.so', b'relax2d.cdv'
        _run_region(_Region([(self.A, _OUT)], [self.n, self.seed]),
                    _Loop(lib, file, 20, 'loop_relax2d_cdv_20', self.A, _full(dims), [self.A, self.n, self.seed], block=(64, 2, 1)))
        self.res, self.mn = ctypes.c_double(), ctypes.c_double()
        self.region = _Region([(self.A,)], [self.w], flags=D.REGION_AMD_GRAPH if case['form'] == 'model' else 0)
        self.loop = _Loop(lib, file, 33, 'loop_relax2d_cdv_33', self.A, _interior(dims), [self.A, self.w],
                          [_red(_MAX, self.res), _red(_MIN, self.mn)], across=[1] * 4)

    def run(self):
        rt = _rt
        res, mn = ctypes.byref(self.res), ctypes.byref(self.mn)
        hist = np.empty((self.iters, 2))
        for it in range(self.iters):
            self.res.value, self.mn.value = 0.0, 1e300
            rt.dvmh_actual_variable2_(res)
            rt.dvmh_actual_variable2_(mn)
            _run_region(self.region, self.loop)
            rt.dvmh_get_actual_variable2_(res)
            rt.dvmh_get_actual_variable2_(mn)
            hist[it] = self.res.value, self.mn.value
        return {'A': self.A.device(), 'hist': hist}


class _Batched:
    def __init__(self, case, seed):
        self.iters, self.count = case['iters'], case['count']
        lib, file = 'libprog_batched.so', b'batched.cdv'
        self.grids = []
        for g, side in enumerate(_sides(case)):
            dims = [side, side]
            A, B, n, sd, eps = _Array(dims), _Array(dims), _L(side), ctypes.c_ulonglong(seed + 1000003 * g), ctypes.c_double()
            _run_region(_Region([(A, _OUT), (B, _OUT)], [n, sd]),
                        _Loop(lib, file, 21, 'loop_batched_init', A, _full(dims), [A, B, n, sd]))
            self.grids.append((A, eps, ctypes.byref(eps), _Region([(A,), (B,)]),
                               _Loop(lib, file, 31, 'loop_batched_st', B, _interior(dims), [A, B], batch='loop_batched_st_cuda_batch'),
                               _Loop(lib, file, 36, 'loop_batched_max', A, _interior(dims), [A, B], [_red(_MAX, eps)],
                                     batch='loop_batched_max_cuda_batch'), B))

    def run(self):
        rt = _rt
        hist = np.empty((self.iters, self.count))
        for it in range(self.iters):
            rt.dvmh_amd_batch_begin_C()
            for A, eps, ref, region, st, mx, _ in self.grids:
                eps.value = 0.0
                rt.dvmh_actual_variable2_(ref)
                r = region.begin()
                rt.dvmh_shadow_renew_C(A.hdr, _L(0), _L(0))
                st.perform(r)
                mx.perform(r)
                rt.dvmh_region_end_C(r)
            rt.dvmh_amd_batch_end_C()
            for g, (_, eps, ref, *_rest) in enumerate(self.grids):
                rt.dvmh_get_actual_variable2_(ref)
                hist[it, g] = eps.value
        return {'A': [g[0].device() for g in self.grids], 'hist': hist}


_STATES = {'jac3d': _Jac3d, 'jac3f': _Jac3f, 'jac2d': _Jac2d, 'gauss': _Gauss, 'sor3d': _Sor3d, 'sor3dchain': _Sor3d, 'adi3d': _Adi3d,
           'relax2d': _Relax2d, 'batched': _Batched}


def prepare(case, seed):
    _set_form(case['form'])
    return _STATES[case['kind']](case, seed)


def run(state):
    return state.run()


# ------------------------------------------------------------- values in 64 bits
def _wrap(x):
    return (x & 0xFFFFFFFFFFFFFFFF) - ((x & 0x8000000000000000) << 1)


def _shr(z, k):
    return (z >> k) & ((1 << (64 - k)) - 1)


def _u01(seed, n):
    """The programs' seeded generator (SplitMix64 finaliser, top 53 bits)."""
    z = (n + 1) * _wrap(0x9E3779B97F4A7C15) + _wrap(seed)
    z = (z ^ _shr(z, 30)) * _wrap(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _wrap(0x94D049BB133111EB)
    z = z ^ _shr(z, 31)
    return _shr(z, 11).double() * (1.0 / 9007199254740992.0)


def _grid(dims, n, seed, border=None):
    """Element (i, j, ..) from its index in a grid of side n; border value where
    an index is 0 or n - 1."""
    dev = 'cuda'
    idx = torch.zeros(tuple(dims), dtype=torch.int64, device=dev)
    edge = torch.zeros(tuple(dims), dtype=torch.bool, device=dev)
    for a, size in enumerate(dims):
        i = torch.arange(size, device=dev).reshape([-1 if b == a else 1 for b in range(len(dims))])
        idx = idx * n + i
        edge |= (i == 0) | (i == n - 1)
    x = _u01(seed, idx)
    return x if border is None else torch.where(edge, torch.full_like(x, border), x)


def _mid(x, *shift):
    """The interior of x, shifted."""
    return x[tuple(slice(1 + s, x.shape[a] - 1 + s) for a, s in enumerate(shift))]


def _star(x, offsets):
    t = _mid(x, *offsets[0])
    for o in offsets[1:]:
        t = t + _mid(x, *o)
    return t


_STAR3 = [(-1, 0, 0), (1, 0, 0), (0, -1, 0), (0, 1, 0), (0, 0, -1), (0, 0, 1)]
_STAR2 = [(-1, 0), (1, 0), (0, -1), (0, 1)]


def _fronts(dims):
    """The interior's flat indices, one tensor per hyperplane of constant index sum."""
    strides = [math.prod(dims[a + 1:]) for a in range(len(dims))]
    flat = torch.zeros([n - 2 for n in dims], dtype=torch.int64, device='cuda')
    level = torch.zeros([n - 2 for n in dims], dtype=torch.int64, device='cuda')
    for a, n in enumerate(dims):
        i = torch.arange(1, n - 1, device='cuda').reshape([-1 if b == a else 1 for b in range(len(dims))])
        flat, level = flat + i * strides[a], level + i - 1
    order = torch.sort(level.reshape(-1), stable=True)
    counts = torch.bincount(order.values).tolist()
    return torch.split(flat.reshape(-1)[order.indices], counts), strides


def _exact_jac3d(case, seed):
    dims = _dims(case)
    A = _grid(dims, max(dims), seed, 0.0)
    B = A.clone()
    hist = []
    for it in range(case['iters']):
        src, dst = (A, B) if it % 2 == 0 else (B, A)
        t = _star(src, _STAR3 + [(0, 0, 0)]) / 7.0
        _mid(dst, 0, 0, 0).copy_(t)
        hist.append([(t - _mid(src, 0, 0, 0)).abs().max().clamp(min=0), t.sum()])
    return {'A': A, 'B': B, 'hist': np.array([[float(v) for v in h] for h in hist])}


def _exact_jac3f(case, seed):
    dims = _dims(case)
    B = _float_grid(dims, seed).cuda().double()
    A = torch.zeros_like(B)
    hist = []
    for _ in range(case['iters']):
        b, a = _mid(B, 0, 0, 0), _mid(A, 0, 0, 0)
        hist.append(float((b - a).abs().max()))
        a.copy_(b)
        b.copy_(_star(A, _STAR3) / 6.0)
    return {'A': A, 'B': B, 'hist': np.array(hist)}


def _jacobi2d(A, iters):
    B = A.clone()
    hist = []
    for _ in range(iters):
        a, b = _mid(A, 0, 0), _mid(B, 0, 0)
        b.copy_(0.25 * _star(A, _STAR2))
        hist.append(float((b - a).abs().max()))
        a.copy_(b)
    return A, B, np.array(hist)


def _exact_jac2d(case, seed):
    dims = _dims(case)
    A, B, hist = _jacobi2d(_grid(dims, max(dims), seed, 1.0), case['iters'])
    return {'A': A, 'B': B, 'hist': hist}


def _exact_batched(case, seed):
    out, hists = [], []
    for g, side in enumerate(_sides(case)):
        A, _, hist = _jacobi2d(_grid([side, side], side, seed + 1000003 * g, 1.0), case['iters'])
        out.append(A)
        hists.append(hist)
    return {'A': out, 'hist': np.stack(hists, axis=1)}


def _exact_gauss(case, seed):
    n = case['n0']
    idx = torch.arange(n * (n + 1), device='cuda').reshape(n, n + 1)
    A = _u01(seed, idx)
    A.diagonal()[:] += float(n)
    for i in range(n - 1):
        A[i + 1:, i + 1:] -= A[i + 1:, i:i + 1] * A[i, i + 1:] / A[i, i]
    x = torch.empty(n, dtype=torch.float64, device='cuda')
    x[n - 1] = A[n - 1, n] / A[n - 1, n - 1]
    for j in range(n - 2, -1, -1):
        A[:j + 1, n] -= A[:j + 1, j + 1] * x[j + 1]
        x[j] = A[j, n] / A[j, j]
    return {'x': x.cpu().numpy(), 'out': A.cpu().numpy()}


def _exact_sor3d(case, seed):
    dims = _dims(case)
    A = _grid(dims, max(dims), seed, 0.0)
    f = A.reshape(-1)
    fronts, st = _fronts(dims)
    hist = []
    for _ in range(case['iters']):
        before = A.clone()
        for p in fronts:
            t = f[p - st[0]] + f[p + st[0]] + f[p - st[1]] + f[p + st[1]] + f[p - st[2]] + f[p + st[2]]
            f[p] = (_OMEGA / 6.0) * t + (1.0 - _OMEGA) * f[p]
        hist.append(float((A - before).abs().max()))
    return {'A': A, 'hist': np.array(hist)}


def _exact_relax2d(case, seed):
    dims = _dims(case)
    A = _grid(dims, max(dims), seed, 1.0)
    f = A.reshape(-1)
    fronts, st = _fronts(dims)
    hist = []
    for _ in range(case['iters']):
        before = A.clone()
        for p in fronts:
            s = f[p]
            t = 0.25 * (f[p - st[0]] + f[p + st[0]] + f[p - st[1]] + f[p + st[1]])
            f[p] = s + _OMEGA * (t - s)
        hist.append([float((_mid(A, 0, 0) - _mid(before, 0, 0)).abs().max()), float(_mid(A, 0, 0).min())])
    return {'A': A, 'hist': np.array(hist)}


def _exact_adi3d(case, seed):
    dims = _dims(case)
    n = max(dims)
    a = _grid(dims, n, seed)
    hist = []
    for _ in range(case['iters']):
        for axis in range(3):
            x = a.transpose(0, axis)
            for i in range(1, dims[axis]):
                x[i] += _COEF * x[i - 1]
            for i in range(dims[axis] - 2, -1, -1):
                x[i] += _COEF * x[i + 1]
        hist.append(float(a.abs().max()))
    return {'a': a, 'hist': np.array(hist), 'loc': None}


_EXACT = {'jac3d': _exact_jac3d, 'jac3f': _exact_jac3f, 'jac2d': _exact_jac2d, 'gauss': _exact_gauss, 'sor3d': _exact_sor3d,
          'sor3dchain': _exact_sor3d, 'adi3d': _exact_adi3d, 'relax2d': _exact_relax2d, 'batched': _exact_batched}


def exact(case, seed):
    return _EXACT[case['kind']](case, seed)
