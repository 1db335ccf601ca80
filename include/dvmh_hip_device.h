/*
 * Device-side helpers for HIP loop handlers emitted for libdvmh_amd (gfx950).
 *
 *   View       array access A[i][j][k] through the natural base and the
 *              per-axis element strides of dvmh_fill_header_C; any axis
 *              permutation of the device layout is just another stride set.
 *   DiagView   the same for a layout whose two fastest storage axes are
 *              diagonalised (planes stored anti-diagonal by anti-diagonal), the
 *              index map of rts/dvmh/include/dvmhlib_device.h:56-98.
 *   MarchView2/3, TileView3, LineView
 *              the same syntax over copies staged in LDS: a rolling window of
 *              three planes of a read-only stencil array (march variant of
 *              PARALLEL loops), a tile with halo of an ACROSS array (tiled
 *              wavefront), and a chunk of one line of an ACROSS array (tiled
 *              line sweep along the innermost axis).
 *   StarView, flowTile
 *              the same syntax over a point and its neighbours in registers,
 *              and the dataflow wavefront that walks them (ACROSS loops whose
 *              axes all depend).
 *   starMarch  a march of a read-only star stencil whose planes live in registers
 *              (PARALLEL loops), read through a StarView.
 *   reductions wave64 shuffle trees plus one LDS step across the waves of a
 *              workgroup; every thread of the workgroup must call them.
 *   xcdTile    XCD-aware renumbering of workgroups: the hardware deals
 *              consecutive workgroup ids round-robin over the 8 XCDs, so
 *              renumbering gives each XCD (and its L2) a contiguous run of tiles.
 *
 * The role of the reference's cdvmh/include/cdvmh_helpers.h (DvmhArrayHelper,
 * DvmhDiagonalizedArrayHelper) and rts/dvmh/include/dvmhlib_{warp,block}_red.h,
 * written for 64-wide wavefronts.
 */
#ifndef DVMH_HIP_DEVICE_H
#define DVMH_HIP_DEVICE_H

#include <hip/hip_runtime.h>

#include <type_traits>

#include "dvmhlib_types.h"
#include "dvmhlib_const.h"
#include "dvmh_amd.h"

namespace dvmh_dev {

// ------------------------------------------------------------------ resources
// Registers per thread of a compiled kernel (0 if the runtime cannot say): the
// figure handlers pass to dvmh_loop_cuda_get_config_C so the block is fitted to
// the register file, as the reference's handlers pass the counts ptxas reports
// (driver/src/dvm_comp:400-432 -> rts/dvmh/loop.cpp:2177-2194).
static inline int kernelRegs(const void *kernel) {
    hipFuncAttributes a;
    if (hipFuncGetAttributes(&a, kernel) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return a.numRegs > 0 ? a.numRegs : 0;
}

// ------------------------------------------------------------------ views
template <typename T, typename I, int R, bool UNIT>
struct View {
    T *base;
    I s[R];
    __device__ __forceinline__ View<T, I, R - 1, UNIT> operator[](I i) const {
        View<T, I, R - 1, UNIT> v;
        v.base = base + i * s[0];
#pragma unroll
        for (int k = 0; k < R - 1; k++) v.s[k] = s[k + 1];
        return v;
    }
};

template <typename T, typename I, bool UNIT>
struct View<T, I, 1, UNIT> {
    T *base;
    I s[1];
    __device__ __forceinline__ T &operator[](I i) const { return UNIT ? base[i] : base[i * s[0]]; }
};

// A device address held as an integer (descriptor tables of batch kernels) as
// a pointer the compiler knows to be global memory: the cast through address
// space 1 lets its loads and stores compile to global_* rather than flat_*
// instructions (no LDS/scratch aperture check, no LGKM counter wait).
template <typename T>
__device__ __forceinline__ T *globalPtr(long a) {
    return (T *)(__attribute__((address_space(1))) T *)a;
}

template <typename T, typename I, int R, bool UNIT>
__device__ __forceinline__ View<T, I, R, UNIT> makeView(T *base, const I *strides) {
    View<T, I, R, UNIT> v;
    v.base = base;
#pragma unroll
    for (int k = 0; k < R; k++) v.s[k] = strides[k];
    return v;
}

// ------------------------------------------------------------------ LDS march views
// A read-only stencil array staged in LDS as a rolling window of three planes
// of the outermost loop axis (planes i-1, i, i+1 of the point being computed).
// A plane holds `rows` x `cols` elements: the workgroup's tile of the inner
// axes plus a halo of one on each side; row 0 / column 0 hold array indices
// j0 / k0.  `A[i'][j'][k']` with |i' - i| <= 1 reads the LDS copy, so a loop
// body written against the global array runs unchanged.
template <typename T, typename I>
struct MarchRow {
    const T *p;
    I k0;
    __device__ __forceinline__ const T &operator[](I k) const { return p[k - k0]; }
};

template <typename T, typename I>
struct MarchPlane {
    const T *p;
    I cols, j0, k0;
    __device__ __forceinline__ MarchRow<T, I> operator[](I j) const { return MarchRow<T, I>{p + (j - j0) * cols, k0}; }
};

__device__ __forceinline__ int marchSlot(int cur, int delta) {
    int s = cur + delta;
    return s < 0 ? s + 3 : (s > 2 ? s - 3 : s);
}

// rank 3: planes of rows x cols
template <typename T, typename I>
struct MarchView3 {
    const T *lds;
    I rows, cols, j0, k0;
    I iCur;
    int sCur;
    __device__ __forceinline__ MarchPlane<T, I> operator[](I i) const {
        return MarchPlane<T, I>{lds + (I)marchSlot(sCur, (int)(i - iCur)) * rows * cols, cols, j0, k0};
    }
};

// rank 2: planes are single rows of cols elements
template <typename T, typename I>
struct MarchView2 {
    const T *lds;
    I cols, k0;
    I iCur;
    int sCur;
    __device__ __forceinline__ MarchRow<T, I> operator[](I i) const {
        return MarchRow<T, I>{lds + (I)marchSlot(sCur, (int)(i - iCur)) * cols, k0};
    }
};

// A tile of a rank-3 array staged in LDS (read and written): element (0,0,0)
// holds array index (i0, j0, k0), planes of rows x cols elements.
template <typename T, typename I>
struct TileRow {
    T *p;
    I k0;
    __device__ __forceinline__ T &operator[](I k) const { return p[k - k0]; }
};

template <typename T, typename I>
struct TilePlane {
    T *p;
    I cols, j0, k0;
    __device__ __forceinline__ TileRow<T, I> operator[](I j) const { return TileRow<T, I>{p + (j - j0) * cols, k0}; }
};

template <typename T, typename I>
struct TileView3 {
    T *p;
    I rows, cols, i0, j0, k0;
    __device__ __forceinline__ TilePlane<T, I> operator[](I i) const {
        return TilePlane<T, I>{p + (i - i0) * rows * cols, cols, j0, k0};
    }
};

// One line of an ACROSS array staged in LDS, for bodies that index it as
// X[i][j][k + d] with the loop's own i, j and |d| <= 1 along the line: the
// leading subscripts select nothing (they are the line the thread owns), the
// last one maps array index k to slot (k - kb) * dir of the line's chunk.
template <typename T, typename I, int D>
struct LineView {
    T *p;
    I kb, dir;
    __device__ __forceinline__ LineView<T, I, D - 1> operator[](I) const { return LineView<T, I, D - 1>{p, kb, dir}; }
};

template <typename T, typename I>
struct LineView<T, I, 1> {
    T *p;
    I kb, dir;
    __device__ __forceinline__ T &operator[](I k) const { return p[(k - kb) * dir]; }
};

// A thread's chunk of its own line of an ACROSS array held in a local buffer
// (the line sweep with register staging, lines along a non-innermost axis):
// for X[i][j][k] with the loop's own indices, the subscript on axis AX selects
// slot (x - x0) * DIR + 1 of the buffer, the others select nothing (they are
// the thread's line).  With the chunk's steps unrolled every slot index is a
// compile-time constant, so the buffer is promoted to registers.
template <typename T, typename I, int D, int AX, int DIR>
struct RegLineView {
    T *buf;
    I x0, slot;
    __device__ __forceinline__ RegLineView<T, I, D - 1, AX - 1, DIR> operator[](I x) const {
        return RegLineView<T, I, D - 1, AX - 1, DIR>{buf, x0, AX == 0 ? (x - x0) * DIR + 1 : slot};
    }
};

template <typename T, typename I, int AX, int DIR>
struct RegLineView<T, I, 1, AX, DIR> {
    T *buf;
    I x0, slot;
    __device__ __forceinline__ T &operator[](I x) const { return buf[AX == 0 ? (x - x0) * DIR + 1 : slot]; }
};

// Diagonal position inside an Rx x Ry plane (x fastest).  Also compiled for
// the host, so the layout-transform kernels, the handlers and host-side checks
// share one definition.
template <typename I>
__host__ __device__ __forceinline__ I convertXY(I x, I y, I Rx, I Ry, int slash) {
    I idx;
    if (!slash) {
        I d = x + y;
        if (Rx == Ry) {
            if (d < Rx) idx = y + (1 + d) * d / 2;
            else idx = Rx * (Rx - 1) + x - (2 * Rx - d - 1) * (2 * Rx - d - 2) / 2;
        } else if (Rx < Ry) {
            if (d < Rx) idx = y + (1 + d) * d / 2;
            else if (d < Ry) idx = (1 + Rx) * Rx / 2 + Rx - x - 1 + Rx * (d - Rx);
            else idx = Rx * Ry - Ry + y - (Rx + Ry - d - 1) * (Rx + Ry - d - 2) / 2;
        } else {
            if (d < Ry) idx = x + (1 + d) * d / 2;
            else if (d < Rx) idx = (1 + Ry) * Ry / 2 + (Ry - y - 1) + Ry * (d - Ry);
            else idx = Rx * Ry - Rx + x - (Rx + Ry - d - 1) * (Rx + Ry - d - 2) / 2;
        }
    } else {
        if (Rx == Ry) {
            I e = x + Rx - 1 - y;
            if (e < Rx) idx = Rx - 1 - y + (e + 1) * e / 2;
            else idx = Rx * (Rx - 1) + x - (Rx - x + y) * (Rx - x + y - 1) / 2;
        } else if (Rx < Ry) {
            I e = x + Ry - 1 - y;
            if (e < Rx) idx = Ry - 1 - y + (e + 1) * e / 2;
            else if (e < Ry) idx = (1 + Rx) * Rx / 2 + Rx - x - 1 + Rx * (e - Rx);
            else idx = Rx * Ry - 1 - y - (Rx + y - x) * (Rx + y - x - 1) / 2;
        } else {
            I e = x + Ry - 1 - y;
            if (e < Ry) idx = x + (1 + e) * e / 2;
            else if (e < Rx) idx = (1 + Ry) * Ry / 2 + y + Ry * (x - y - 1);
            else idx = Rx * Ry - Rx + x - (Rx + y - x) * (Rx + y - x - 1) / 2;
        }
    }
    return idx;
}

// Header extension of a diagonalised array (dvmh_fill_header_C's extendedParams).
template <typename I>
struct DiagInfo {
    int xAxis, yAxis, slash;   // 1-based original axes
    I xFirst, xLen, yFirst, yLen;
};

template <typename T, typename I, int R, int D>
struct DiagView {
    T *base;
    I s[R];
    I off, x, y;
    DiagInfo<I> di;
    __device__ __forceinline__ DiagView<T, I, R, D + 1> operator[](I i) const {
        DiagView<T, I, R, D + 1> v;
        v.base = base;
#pragma unroll
        for (int k = 0; k < R; k++) v.s[k] = s[k];
        v.di = di;
        v.off = off + i * s[D];
        v.x = (di.xAxis == D + 1) ? i : x;
        v.y = (di.yAxis == D + 1) ? i : y;
        return v;
    }
};

template <typename T, typename I, int R>
struct DiagView<T, I, R, R - 1> {
    T *base;
    I s[R];
    I off, x, y;
    DiagInfo<I> di;
    __device__ __forceinline__ T &operator[](I i) const {
        I o = off + i * s[R - 1];
        I xx = (di.xAxis == R) ? i : x, yy = (di.yAxis == R) ? i : y;
        return base[o + convertXY<I>(xx - di.xFirst, yy - di.yFirst, di.xLen, di.yLen, di.slash)];
    }
};

template <typename T, typename I, int R>
__device__ __forceinline__ DiagView<T, I, R, 0> makeDiagView(T *base, const I *strides, const DiagInfo<I> &di) {
    DiagView<T, I, R, 0> v;
    v.base = base;
#pragma unroll
    for (int k = 0; k < R; k++) v.s[k] = strides[k];
    v.off = 0;
    v.x = 0;
    v.y = 0;
    v.di = di;
    return v;
}

// ------------------------------------------------------------------ reductions
// Lane shuffle of any reduction element type (1, 2, 4 or 8 bytes, signed or
// unsigned, integer or floating), bit for bit.
template <typename T>
__device__ __forceinline__ T shflDown(T v, int o) {
    static_assert(sizeof(T) == 1 || sizeof(T) == 2 || sizeof(T) == 4 || sizeof(T) == 8, "reduction element size");
    if constexpr (sizeof(T) == 8) {
        long long x;
        __builtin_memcpy(&x, &v, 8);
        x = __shfl_down(x, o, 64);
        __builtin_memcpy(&v, &x, 8);
    } else {
        int x = 0;
        __builtin_memcpy(&x, &v, sizeof(T));
        x = __shfl_down(x, o, 64);
        __builtin_memcpy(&v, &x, sizeof(T));
    }
    return v;
}

struct OpSum {
    template <typename T> __device__ __forceinline__ T operator()(T a, T b) const { return a + b; }
};
struct OpProd {
    template <typename T> __device__ __forceinline__ T operator()(T a, T b) const { return a * b; }
};
struct OpMax {
    template <typename T> __device__ __forceinline__ T operator()(T a, T b) const { return a < b ? b : a; }
};
struct OpMin {
    template <typename T> __device__ __forceinline__ T operator()(T a, T b) const { return a > b ? b : a; }
};
struct OpAnd {
    template <typename T> __device__ __forceinline__ T operator()(T a, T b) const { return a & b; }
};
struct OpOr {
    template <typename T> __device__ __forceinline__ T operator()(T a, T b) const { return a | b; }
};
struct OpXor {
    template <typename T> __device__ __forceinline__ T operator()(T a, T b) const { return a ^ b; }
};

// Initial values of a reduction array (N elements), passed to a kernel by value.
template <typename T, int N>
struct RedVec {
    T v[N];
};
template <typename T, int N>
__host__ __device__ inline RedVec<T, N> redVec(const T (&a)[N]) {
    RedVec<T, N> r;
    for (int i = 0; i < N; i++) r.v[i] = a[i];
    return r;
}

// Reduce over the workgroup; the result is valid in thread 0.  Fixed order:
// shuffle tree inside each wave, then wave results in wave order.
template <typename T, typename Op>
__device__ __forceinline__ T blockReduce(T v, Op op) {
    __shared__ T part[16];
    const int nthreads = blockDim.x * blockDim.y * blockDim.z;
    const int t = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
    const int lane = t & 63, wave = t >> 6;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        T other = shflDown(v, o);
        if (lane + o < 64 && t + o < nthreads) v = op(v, other);
    }
    __syncthreads();
    if (lane == 0) part[wave] = v;
    __syncthreads();
    if (t == 0) {
        const int nw = (nthreads + 63) >> 6;
        for (int w = 1; w < nw; w++) v = op(v, part[w]);
    }
    __syncthreads();
    return v;
}

// MAXLOC / MINLOC: larger (smaller) value wins, equal values keep the lower loc.
template <typename T, typename L, bool MAXF>
__device__ __forceinline__ void blockReduceLoc(T &v, L &loc) {
    __shared__ T pv[16];
    __shared__ L pl[16];
    const int nthreads = blockDim.x * blockDim.y * blockDim.z;
    const int t = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
    const int lane = t & 63, wave = t >> 6;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        T ov = shflDown(v, o);
        L ol = shflDown(loc, o);
        if (lane + o < 64 && t + o < nthreads) {
            bool take = MAXF ? (v < ov || (!(ov < v) && ol < loc)) : (v > ov || (!(ov > v) && ol < loc));
            if (take) { v = ov; loc = ol; }
        }
    }
    __syncthreads();
    if (lane == 0) { pv[wave] = v; pl[wave] = loc; }
    __syncthreads();
    if (t == 0) {
        const int nw = (nthreads + 63) >> 6;
        for (int w = 1; w < nw; w++) {
            bool take = MAXF ? (v < pv[w] || (!(pv[w] < v) && pl[w] < loc)) : (v > pv[w] || (!(pv[w] > v) && pl[w] < loc));
            if (take) { v = pv[w]; loc = pl[w]; }
        }
    }
    __syncthreads();
}

// ------------------------------------------------------------------ in-kernel finish
// Folding a loop's partials in the loop's own kernel: the workgroup that
// arrives last at a counter folds them and writes the results to host memory,
// so a loop with scalar reductions is one launch.  Partials are folded in
// groups of consecutive workgroups (a counter each), the groups' results by
// the last group, always in the same order, so results are deterministic.
//
// What workgroups exchange goes through agent-scope relaxed atomics (they
// bypass the L2 of the XCD they run on) with a wait for the stores to complete
// before the arrival is counted.  A release fence instead would write back the
// XCD's whole L2 in every workgroup (measured 3.3x on the 384^3 Jacobi kernel).
// Measured against the separate finish launch (8-20 us of GPU time and a
// launch gap per loop), per iteration of 3-D Jacobi: 34^3 27.3 -> 19.8 us,
// 201x187x239 92 -> 85, 384^3 227 -> 215.  The waits lengthen the kernel
// itself by 3 us (80 workgroups), 6 (7,000) and 13 (37,000).
template <typename T, int SCOPE>
__device__ __forceinline__ void scopedStore(T *p, T v) {
    static_assert(sizeof(T) == 1 || sizeof(T) == 4 || sizeof(T) == 8, "reduction element size");
    if constexpr (sizeof(T) == 8) {
        unsigned long long x;
        __builtin_memcpy(&x, &v, 8);
        __hip_atomic_store((unsigned long long *)p, x, __ATOMIC_RELAXED, SCOPE);
    } else if constexpr (sizeof(T) == 4) {
        unsigned x;
        __builtin_memcpy(&x, &v, 4);
        __hip_atomic_store((unsigned *)p, x, __ATOMIC_RELAXED, SCOPE);
    } else {
        unsigned char x;
        __builtin_memcpy(&x, &v, 1);
        __hip_atomic_store((unsigned char *)p, x, __ATOMIC_RELAXED, SCOPE);
    }
}

template <typename T>
__device__ __forceinline__ void agentStore(T *p, T v) { scopedStore<T, __HIP_MEMORY_SCOPE_AGENT>(p, v); }

template <typename T>
__device__ __forceinline__ T agentLoad(const T *p) {
    T v;
    if constexpr (sizeof(T) == 8) {
        const unsigned long long x = __hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_memcpy(&v, &x, 8);
    } else if constexpr (sizeof(T) == 4) {
        const unsigned x = __hip_atomic_load((const unsigned *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_memcpy(&v, &x, 4);
    } else {
        const unsigned char x = __hip_atomic_load((const unsigned char *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_memcpy(&v, &x, 1);
    }
    return v;
}

// Every store of this wave so far has completed at the scope it was made for.
__device__ __forceinline__ void storesDone() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ int linearTid() { return threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z); }

// Called by the workgroup's first wave once its lane 0 has stored a partial:
// true in the wave that arrives as the last of `count` (which zeroes the
// counter for the next launch).
__device__ __forceinline__ bool lastArrival(unsigned *counter, unsigned count) {
    unsigned last = 0;
    if (linearTid() == 0) {
        storesDone();
        last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == count - 1;
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" ::: "memory");   // no load of the others' partials moves above the arrival
    }
    return __builtin_amdgcn_readfirstlane(last) != 0;
}

// The first wave folds slots[0, n), n >= 1; lane 0 ends with the result: lane l
// folds l, l + W, ... in order (W lanes in the wave, four loads in flight), then
// a shuffle tree.
template <typename T, typename Op>
__device__ __forceinline__ T foldSlots(const T *slots, int n, Op op) {
    const int threads = blockDim.x * blockDim.y * blockDim.z;
    const int W = threads < 64 ? threads : 64;
    const int lane = linearTid();
    T v = agentLoad(slots + (lane < n ? lane : 0));
    for (int i = lane + W; i < n; i += 4 * W) {
        T x[4];
#pragma unroll
        for (int q = 0; q < 4; q++) x[q] = agentLoad(slots + (i + q * W < n ? i + q * W : 0));
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (i + q * W < n) v = op(v, x[q]);
    }
    const int have = n < W ? n : W;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const T other = shflDown(v, o);
        if (lane + o < have) v = op(v, other);
    }
    return v;
}

// The same for MAXLOC / MINLOC records (equal values keep the lower loc).
template <typename T, typename L, bool MAXF>
__device__ __forceinline__ void foldSlotsLoc(const T *slots, const L *locs, int n, T &v, L &loc) {
    const int threads = blockDim.x * blockDim.y * blockDim.z;
    const int W = threads < 64 ? threads : 64;
    const int lane = linearTid();
    auto take = [](T a, L la, T b, L lb) { return MAXF ? (a < b || (!(b < a) && lb < la)) : (a > b || (!(b > a) && lb < la)); };
    v = agentLoad(slots + (lane < n ? lane : 0));
    loc = agentLoad(locs + (lane < n ? lane : 0));
    for (int i = lane + W; i < n; i += 4 * W) {
        T x[4];
        L y[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            x[q] = agentLoad(slots + (i + q * W < n ? i + q * W : 0));
            y[q] = agentLoad(locs + (i + q * W < n ? i + q * W : 0));
        }
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (i + q * W < n && take(v, loc, x[q], y[q])) { v = x[q]; loc = y[q]; }
    }
    const int have = n < W ? n : W;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const T ov = shflDown(v, o);
        const L ol = shflDown(loc, o);
        if (lane + o < have && take(v, loc, ov, ol)) { v = ov; loc = ol; }
    }
}

// Results to host memory, then (all of them complete) the completion word.
template <typename T>
__device__ __forceinline__ void hostStore(T *p, T v) { scopedStore<T, __HIP_MEMORY_SCOPE_SYSTEM>(p, v); }

__device__ __forceinline__ void publishDone(const DvmhAmdRedFinish &f) {
    if (!f.done) return;
    storesDone();
    __hip_atomic_store(f.done, f.doneSeq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ------------------------------------------------------------------ dataflow wavefront
// ACROSS loops whose axes all depend (rank 2 or 3) in one launch.  A wave owns
// a tile of the leading axes -- 8 x 8 points for rank 3, 64 for rank 2, one
// lane per point -- and walks the innermost axis; lane (p, q) runs one step
// behind lanes (p - 1, q) and (p, q - 1), so at every step each lane's lower
// neighbours are the previous step's results and its upper ones are still old:
// the order of the sequential sweep.  Tiles are taken in the order of their
// diagonal from a ticket counter, so a tile only ever waits for tiles that are
// running or done, whatever the launch's residency.
//
// The rows of a tile pass through LDS in blocks of eight steps, three of them
// at a time.  A row is held at the step its elements are walked at (element r
// of row (p, q) in slot r + p + q and the tile's phase), so in every step all
// lanes use the same slots, at offsets known to the compiler, and a finished
// block of steps is stored at once.  A block's loads and stores move eight
// aligned elements of eight rows per instruction; two blocks' loads are in
// flight while one is walked.  Rows a tile needs from its lower neighbours come
// through cells in device memory, 1 KB per face and block of steps, written and
// read by one instruction: a value in halves, each beside a 32-bit tag that no
// earlier launch used, so one load tells whether it is there.
//
// Bound by the chain of dependent steps: 0.13 us a step for rank 2 (eight
// dependent FP64 operations and a lane shift), 0.165 for rank 3 (one neighbour
// through LDS), and along a diagonal of tiles, per tile, the lanes' skew plus
// about 4 us until a finished block is seen by the next tile; chains of large
// grids by the same with several sweeps in flight (they move 26 bytes a point
// and sweep, 3.5 TB/s of the 6.3 a copy reaches).  Measured,
// one sweep with reductions: 2-D 998^2 0.38 ms (a launch per hyperplane: 9.2),
// 3-D 128^3 0.145 ms (a launch per tile-plane: 0.43), 318^3 0.48 ms (1.84; 0.76
// with rows moved unaligned and a cell's halves in two stores).
template <int RANK> struct FlowShape;
template <> struct FlowShape<3> {
    // row (p, q), -1 <= p, q <= 8, at (p + 1) * BP + (q + 1) * QP: the 32 lanes
    // of an LDS cycle in 32 different bank pairs
    static constexpr int PA = 8, PB = 8, BP = 264, QP = 25, LDS = 9 * 264 + 9 * 25 + 24;
};
template <> struct FlowShape<2> {
    static constexpr int PA = 64, PB = 1, BP = 25, QP = 0, LDS = 65 * 25 + 24;
};

// The element at the loop point (slot 0) and its neighbours along axis a, one
// below (slot 1 + 2 a) and one above (slot 2 + 2 a), as X[i][j][k].
template <typename T, typename I, int R, int AX = 0>
struct StarView {
    T *v;
    I at[R];
    int slot;
    __device__ __forceinline__ decltype(auto) operator[](I x) const {
        const I d = x - at[AX];
        const int s = d < 0 ? 1 + 2 * AX : (d > 0 ? 2 + 2 * AX : slot);
        if constexpr (AX + 1 == R) {
            return (v[s]);
        } else {
            StarView<T, I, R, AX + 1> n;
            n.v = v;
#pragma unroll
            for (int a = 0; a < R; a++) n.at[a] = at[a];
            n.slot = s;
            return n;
        }
    }
};

// The element of an array at the loop point, kept in a register: X[i][j][k]
// with the loop's own indices only.
template <typename T, int R>
struct PointView {
    T *v;
    template <typename I>
    __device__ __forceinline__ decltype(auto) operator[](I) const {
        if constexpr (R == 1) return (*v);
        else return PointView<T, R - 1>{v};
    }
};

template <typename T, typename I, int RANK>
struct FlowArgs {
    T *base;
    I s[RANK];              // element strides (the innermost is 1)
    I lo[RANK], cnt[RANK];  // the loop
    I rlo[RANK], rhi[RANK]; // array indices the body may read: loads are clamped into them
    int ntA, ntB, sweeps;
    DvmhAmdFlow ws;
};

struct FlowTask {
    int sweep, ta, tb;
    unsigned tag;           // of the task's sweep
};

// Tiles on diagonal d of an ntA x ntB grid.
__device__ __forceinline__ int flowDiagonal(int d, int ntA, int ntB) {
    const int hi = d < ntA - 1 ? d : ntA - 1, lo = d - ntB + 1 > 0 ? d - ntB + 1 : 0;
    return d < 0 || hi < lo ? 0 : hi - lo + 1;
}

// The wave's task: tickets in the order of ta + tb + 2 * sweep, which every
// task a task waits for precedes.  The control word holds the tag of the last
// sweep so far (high half) and the next ticket; the taker of the last ticket
// sets it up for the next launch.
__device__ __forceinline__ FlowTask flowTake(int ntA, int ntB, int sweeps, const DvmhAmdFlow &ws) {
    unsigned ticket = 0, epoch = 0;
    if (threadIdx.x == 0) {
        const unsigned long long c = __hip_atomic_fetch_add(ws.control, 1ULL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ticket = (unsigned)c;
        epoch = (unsigned)(c >> 32);
        if (ticket == (unsigned)ntA * (unsigned)ntB * (unsigned)sweeps - 1) {
            const unsigned long long next = epoch + (unsigned)sweeps;
            __hip_atomic_store(ws.control, next << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (next >> 31) __hip_atomic_store(ws.wrapped, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    ticket = __builtin_amdgcn_readfirstlane(ticket);
    epoch = __builtin_amdgcn_readfirstlane(epoch);
    const int lane = threadIdx.x;
    int t = (int)ticket, key = 0;
    for (int k0 = 0;; k0 += 64) {
        int n = 0;
        for (int s = 0; s < sweeps; s++) n += flowDiagonal(k0 + lane - 2 * s, ntA, ntB);
        int upTo = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int below = __shfl_up(upTo, o, 64);
            if (lane >= o) upTo += below;
        }
        const unsigned long long past = __ballot(upTo > t);
        if (past) {
            const int at = __builtin_ctzll(past);
            t -= __shfl(upTo - n, at, 64);
            key = k0 + at;
            break;
        }
        t -= __shfl(upTo, 63, 64);
    }
    int s = 0;
    for (;; s++) {
        const int n = flowDiagonal(key - 2 * s, ntA, ntB);
        if (t < n) break;
        t -= n;
    }
    const int d = key - 2 * s;
    const int a = (d - ntB + 1 > 0 ? d - ntB + 1 : 0) + t;
    return FlowTask{__builtin_amdgcn_readfirstlane(s), __builtin_amdgcn_readfirstlane(a), __builtin_amdgcn_readfirstlane(d - a),
                    epoch + (unsigned)s + 1};
}

// Cells: 64 values a lane each, the value's halves each beside the tag, moved
// by one 16-byte access per lane at agent scope (each 8-byte word is written
// whole; a reader checks both tags).
typedef unsigned FlowWords __attribute__((ext_vector_type(4)));
constexpr int FLOW_CELLS_BYTES = 64 * 16;

template <typename T>
struct FlowCells {
    FlowWords w;
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t at(const void *p, unsigned bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00027000);
    }
    static constexpr int AGENT = 16;   // cache policy: agent scope (sc1)
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t from, int offset) {
        w = __builtin_amdgcn_raw_buffer_load_b128(from, threadIdx.x * 16, offset, AGENT);
    }
    __device__ __forceinline__ bool holds(unsigned tag) const { return (w[1] == tag) & (w[3] == tag); }
    __device__ __forceinline__ T value() const {
        const unsigned x[2] = {w[0], w[2]};
        T v;
        __builtin_memcpy(&v, x, sizeof(T));
        return v;
    }
    static __device__ __forceinline__ void store(__amdgpu_buffer_rsrc_t to, int offset, T v, unsigned tag) {
        unsigned x[2] = {0, 0};
        __builtin_memcpy(x, &v, sizeof(T));
        __builtin_amdgcn_raw_buffer_store_b128(FlowWords{x[0], tag, x[1], tag}, to, threadIdx.x * 16, offset, AGENT);
    }
};

// Blocks of a face's cells: one per block of steps of the tile, at most this many.
__host__ __device__ inline long flowBlocks(int rank, long n) { return (n + (rank == 3 ? 14 : 63) + 7 + 7) >> 3; }

// A face is addressed by 32-bit byte offsets, up to sixteen blocks past its
// last (those read as no cell); the points of a row that are walked in one launch.
constexpr long FLOW_BLOCKS_MAX = (1L << 31) / FLOW_CELLS_BYTES - 16;
constexpr long FLOW_ROW_MAX = FLOW_BLOCKS_MAX * 8 - 128;
// Tiles and sweeps of a launch: a wave each, and a launch has fewer than 2^32 work-items.
constexpr long FLOW_TASKS_MAX = (1L << 26) - 1;

// Lane l gets lane l - 1's x, lane 0 gets `first` (whole wave active).
template <typename T>
__device__ __forceinline__ T laneBelow(T x, T first) {
    int w[2] = {0, 0}, o[2] = {0, 0};
    __builtin_memcpy(w, &x, sizeof(T));
    __builtin_memcpy(o, &first, sizeof(T));
    constexpr int WAVE_SHR1 = 0x138;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) + 3) / 4; i++) w[i] = __builtin_amdgcn_update_dpp(o[i], w[i], WAVE_SHR1, 0xf, 0xf, false);
    T r;
    __builtin_memcpy(&r, w, sizeof(T));
    return r;
}

// Lane l gets lane l + 1's x, lane 63 gets `last` (whole wave active).
template <typename T>
__device__ __forceinline__ T laneAbove(T x, T last) {
    int w[2] = {0, 0}, o[2] = {0, 0};
    __builtin_memcpy(w, &x, sizeof(T));
    __builtin_memcpy(o, &last, sizeof(T));
    constexpr int WAVE_SHL1 = 0x130;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) + 3) / 4; i++) w[i] = __builtin_amdgcn_update_dpp(o[i], w[i], WAVE_SHL1, 0xf, 0xf, false);
    T r;
    __builtin_memcpy(&r, w, sizeof(T));
    return r;
}

// Lane `lane`'s x in every lane.
template <typename T>
__device__ __forceinline__ T laneOf(T x, int lane) {
    int w[2] = {0, 0};
    __builtin_memcpy(w, &x, sizeof(T));
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) + 3) / 4; i++) w[i] = __builtin_amdgcn_readlane(w[i], lane);
    T r;
    __builtin_memcpy(&r, w, sizeof(T));
    return r;
}

// The first active lane's x, as a scalar.
__device__ __forceinline__ unsigned long firstLane(unsigned long x) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)x);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(x >> 32));
    return (unsigned long)hi << 32 | lo;
}

// An element per lane at the scalar address `base` + `step` bytes plus the lane's
// own 32-bit byte offset: the per-step part of the address costs scalar
// instructions only (4- and 8-byte types).
template <typename T>
struct LaneRow {
    __amdgpu_buffer_rsrc_t rs;
    char *base;
    unsigned lane;
    __device__ __forceinline__ LaneRow(char *b, unsigned l) : rs(__builtin_amdgcn_make_buffer_rsrc(b, 0, -1, 0x00027000)), base(b), lane(l) {}
    __device__ __forceinline__ T load(int step) const {
        T v;
        if constexpr (sizeof(T) == 8) {
            const auto w = __builtin_amdgcn_raw_buffer_load_b64(rs, (int)lane, step, 0);
            __builtin_memcpy(&v, &w, 8);
        } else if constexpr (sizeof(T) == 4) {
            const auto w = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)lane, step, 0);
            __builtin_memcpy(&v, &w, 4);
        } else {
            v = *(const T *)(base + step + lane);
        }
        return v;
    }
    __device__ __forceinline__ void store(int step, T v) const {
        if constexpr (sizeof(T) == 8) {
            decltype(__builtin_amdgcn_raw_buffer_load_b64(rs, 0, 0, 0)) w;
            __builtin_memcpy(&w, &v, 8);
            __builtin_amdgcn_raw_buffer_store_b64(w, rs, (int)lane, step, 0);
        } else if constexpr (sizeof(T) == 4) {
            decltype(__builtin_amdgcn_raw_buffer_load_b32(rs, 0, 0, 0)) w;
            __builtin_memcpy(&w, &v, 4);
            __builtin_amdgcn_raw_buffer_store_b32(w, rs, (int)lane, step, 0);
        } else {
            *(T *)(base + step + lane) = v;
        }
    }
};

// x is in its register here (its load is issued before, not sunk to its use).
template <typename T>
__device__ __forceinline__ void readHere(T &x) {
    if constexpr (sizeof(T) < 4) {   // (no register of its own width)
        int w = x;
        asm volatile("" : "+v"(w));
        x = (T)w;
    } else {
        asm volatile("" : "+v"(x));
    }
}

// ------------------------------------------------------------------ star march
// One wave marches nz planes (axis 0) over R rows (axis 1) of 64 * C points of
// axis 2, point l + 64 c in lane l, and runs body(v, t0, t1, t2) at every loop
// point; v[0] is the element there, v[1 + 2 a] and v[2 + 2 a] its neighbours
// below and above along axis a.
//
// Every plane a point needs stays in the registers of the lane that owns the
// point: the planes below, at and above it, and the one being loaded.  The rows
// beside the R rows and the two columns beside the tile are loaded for the
// current plane only, neighbours along a row come from the lane beside.  No LDS
// and no barrier: the loads of the next planes stay in flight across the
// arithmetic (with planes staged in LDS, two barriers a plane drained them).
// Bound by memory.  Without a reduction: 256^3 doubles, 268 MB read and written,
// 37 us (7.3 TB/s, partly from the last-level cache; planes in LDS 78, direct
// 76), 201 x 187 x 239 24 us (45), 128^3 9 (26); 384^3, beyond that cache, 175
// (200).  With MAX and SUM folded in the launch: 201 x 187 x 239 30 us, 384^3 182.
// Loads are clamped into [rlo, rhi], the indices the body may read.
// (Rank 2 has too little to keep: the same march over rows of 2-D grids is no
// faster than the direct kernel, 2048^2 23 us both, 1024^2 15 against 14.)
template <typename T, typename I, int R, int C, typename Body>
__device__ __forceinline__ void starMarch(const T *__restrict__ base, I s0, I s1, const I (&lo)[3], const I (&cnt)[3],
        const I (&rlo)[3], const I (&rhi)[3], I tz, I nz, I ty, I tx, Body body) {
    const int lane = (int)(threadIdx.x & 63);
    auto clampTo = [&](I x, int a) { return x < rlo[a] ? rlo[a] : (x > rhi[a] ? rhi[a] : x); };
    I col[C], row[R + 2];
#pragma unroll
    for (int c = 0; c < C; c++) col[c] = clampTo(lo[2] + tx + lane + 64 * c, 2);
    const I side = clampTo(lane < 32 ? lo[2] + tx - 1 : lo[2] + tx + 64 * C, 2);
#pragma unroll
    for (int r = 0; r < R + 2; r++) row[r] = clampTo(lo[1] + ty - 1 + r, 1) * s1;
    T own[4][R][C], beside[2][2][C], edge[2][R];
    auto loadOwn = [&](int q, I t) {
        const T *p = base + clampTo(lo[0] + t, 0) * s0;
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < C; c++) own[q][r][c] = p[row[r + 1] + col[c]];
    };
    auto loadBeside = [&](int q, I t) {
        const T *p = base + clampTo(lo[0] + t, 0) * s0;
#pragma unroll
        for (int c = 0; c < C; c++) {
            beside[q][0][c] = p[row[0] + col[c]];
            beside[q][1][c] = p[row[R + 1] + col[c]];
        }
#pragma unroll
        for (int r = 0; r < R; r++) edge[q][r] = p[row[r + 1] + side];
    };
    auto step = [&](I t, int below, int at, int above, int h) {
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < C; c++) {
                T v[7];
                const T x = own[at][r][c];
                v[0] = x;
                v[1] = own[below][r][c];
                v[2] = own[above][r][c];
                v[3] = r == 0 ? beside[h][0][c] : own[at][r == 0 ? 0 : r - 1][c];
                v[4] = r == R - 1 ? beside[h][1][c] : own[at][r == R - 1 ? r : r + 1][c];
                v[5] = laneBelow(x, c == 0 ? edge[h][r] : laneOf(own[at][r][c == 0 ? 0 : c - 1], 63));
                v[6] = laneAbove(x, c == C - 1 ? edge[h][r] : laneOf(own[at][r][c == C - 1 ? c : c + 1], 0));
                const I tk = tx + lane + 64 * c, tj = ty + r;
                if (tk >= 0 && tk < cnt[2] && tj < cnt[1]) body(v, t, tj, tk);
            }
    };
    loadOwn(0, tz - 1);
    loadOwn(1, tz);
    loadOwn(2, tz + 1);
    loadBeside(0, tz);
    const I end = tz + nz;
    for (I t = tz; t < end; t += 4) {
        loadOwn(3, t + 2);
        loadBeside(1, t + 1);
        step(t, 0, 1, 2, 0);
        if (t + 1 >= end) break;
        loadOwn(0, t + 3);
        loadBeside(0, t + 2);
        step(t + 1, 1, 2, 3, 1);
        if (t + 2 >= end) break;
        loadOwn(1, t + 4);
        loadBeside(1, t + 3);
        step(t + 2, 2, 3, 0, 0);
        if (t + 3 >= end) break;
        loadOwn(2, t + 5);
        loadBeside(0, t + 4);
        step(t + 3, 3, 0, 1, 1);
    }
}

// Walks the task's tile.  body(v, t0, t1, t2) runs the loop body at position
// (t0, t1, t2) of the loop (t2 unused for rank 2) with v the star around it.
// CHAIN: several sweeps of the array in one launch; its elements then pass
// between workgroups, so they are loaded and stored at agent scope, and a
// tile's flag says how many chunks of which sweep are in memory.
template <typename T, typename I, int RANK, bool CHAIN, typename Body>
__device__ __forceinline__ void flowTile(const FlowArgs<T, I, RANK> &f, const FlowTask &task, T *ring, Body &&body) {
    using S = FlowShape<RANK>;
    constexpr int K = RANK - 1, SKEW = S::PA + S::PB - 2, SLOTS = 24;
    const int lane = threadIdx.x, g = lane >> 3, e = lane & 7;   // transfers: eight rows of eight elements
    const int p = RANK == 3 ? g : lane, q = RANK == 3 ? e : 0;   // the lane's own row
    const int ta = task.ta, tb = task.tb;
    const I a0 = (I)ta * S::PA, b0 = (I)tb * S::PB;
    const int na = f.cnt[0] - a0 < S::PA ? (int)(f.cnt[0] - a0) : S::PA;
    const int nb = RANK == 2 ? 1 : (f.cnt[1] - b0 < S::PB ? (int)(f.cnt[1] - b0) : S::PB);
    const int n = (int)f.cnt[K];
    // a tile begins up to seven steps late, so that what the next tile needs
    // in a block of steps is what this one does in a block
    const int phase = -(ta + tb) & 7;
    const int blocks = (n + na + nb - 2 + phase + 7) >> 3;   // blocks of steps
    auto clampTo = [](I x, I lo, I hi) { return x < lo ? lo : (x > hi ? hi : x); };
    auto rowOff = [&](int pp, int qq) -> I {
        I o = clampTo(f.lo[0] + a0 + pp, f.rlo[0], f.rhi[0]) * f.s[0];
        if constexpr (RANK == 3) o += clampTo(f.lo[1] + b0 + qq, f.rlo[1], f.rhi[1]) * f.s[1];
        return o;
    };
    auto rowAt = [](int pp, int qq) { return (pp + 1) * S::BP + (qq + 1) * S::QP; };
    // Rows a lane moves: transfer it < 8 the tile's own, 8 and 9 the ones above
    // it, 10 and 11 the ones below (at the array's lower edges; elsewhere those
    // come in cells).  Row (pp, qq) holds element r in slot r + pp + qq + phase.
    auto rowP = [&](int it) { return RANK == 2 ? (it < 8 ? it * 8 + g : it == 8 ? S::PA : -1) : it < 8 ? it : it == 8 ? S::PA : it == 10 ? -1 : g; };
    auto rowQ = [&](int it) { return RANK == 2 ? 0 : it == 9 ? S::PB : it == 11 ? -1 : g; };
    const bool edgeA = ta == 0, edgeB = RANK == 3 && tb == 0;
    auto uses = [&](int it) { return RANK == 3 || it < 9 || it == 10 ? it < 10 || (it == 10 ? edgeA : edgeB) : false; };
    // A transfer moves eight elements of a row that are aligned in memory (64
    // bytes of FP64): slots 8 c - 8 + ahead .. + 7 for chunk c, where `ahead`,
    // 0 .. 7, is the row's own
    I off[12];      // element index of slot 0
    int ahead[12];  // plus the lane's element of the chunk
    auto eachRow = [&](auto &&fn) {
#pragma unroll
        for (int it = 0; it < 12; it++)
            if (RANK == 3 || it < 9 || it == 10) fn(it);
    };
    eachRow([&](int it) {
        off[it] = rowOff(rowP(it), rowQ(it)) + f.lo[K] - (I)(rowP(it) + rowQ(it) + phase);
        ahead[it] = (int)(-(long)((uintptr_t)f.base / sizeof(T) + off[it]) & 7) + e;
    });
    // slot of the ring that a lane's element of chunk c is in
    auto slotOf = [&](int it, int c8) {
        const unsigned x = (unsigned)(c8 + ahead[it]);
        return x < x - SLOTS ? x : x - SLOTS;   // c8 < 24: at most one turn
    };
    auto chunk8 = [](int c) { return (unsigned)(c + 2) % 3u * 8u; };   // 8 c - 8, in the ring
    // two chunks' loads are in flight while a block is walked (a block of steps
    // takes less than a round trip to memory), in two sets of registers
    struct Ahead {
        T v[12];
    } even{}, odd{};
    // (issued on every path, past the row's ends from its nearest element, so
    // that the waits know how many younger loads may stay in flight)
    auto issue = [&](Ahead &h, int c) {
        eachRow([&](int it) {
            if (uses(it)) {
                const I first = off[it] + (I)(rowP(it) + rowQ(it) + phase) - f.lo[K];
                const T *x = f.base + (first + clampTo(off[it] - first + 8 * c - 8 + ahead[it], f.rlo[K], f.rhi[K]));
                h.v[it] = CHAIN ? agentLoad(x) : *x;
            }
        });
    };
    auto commit = [&](const Ahead &h, int c) {
        const int c8 = chunk8(c);
        eachRow([&](int it) {
            if (uses(it) && (RANK == 3 || it < 8 || g == 0)) ring[rowAt(rowP(it), rowQ(it)) + slotOf(it, c8)] = h.v[it];
        });
    };
    // cells of a tile's upper faces, 64 per block of steps: lane (g, e) holds what
    // row g of the face did at step e
    const long tile = (long)ta * f.ntB + tb;
    const unsigned faceBytes = (unsigned)flowBlocks(RANK, n) * FLOW_CELLS_BYTES;
    char *const cells = (char *)f.ws.cells;
    auto face = [&](long t, int which) { return FlowCells<T>::at(cells + (t * (RANK - 1) + which) * (long)faceBytes, faceBytes); };
    const bool fromA = ta > 0, fromB = RANK == 3 && tb > 0;
    const bool toA = ta + 1 < f.ntA, toB = RANK == 3 && tb + 1 < f.ntB;
    const auto inA = face(fromA ? tile - f.ntB : tile, 0), outA = face(tile, 0);
    const auto inB = face(fromB ? tile - 1 : tile, RANK - 2), outB = face(tile, RANK - 2);
    const bool rowA = fromA && (RANK == 3 ? g < nb : g == 0), rowB = fromB && g < na;
    auto inRow = [&](int r) { return (unsigned)r < (unsigned)n; };
    // block m needs the neighbour's block m + lag (one less where its phase is 0): the
    // element lane (0, g) or (g, 0) runs above at step e, 8 m + e - g - phase
    const int lag = S::PA / 8 - (phase == 7 ? 1 : 0);
    FlowCells<T> cA{}, cB{};
    auto fetch = [&](int m) {
        cA.load(inA, (m + lag) * FLOW_CELLS_BYTES);
        if constexpr (RANK == 3) cB.load(inB, (m + lag) * FLOW_CELLS_BYTES);
    };
    auto missing = [&](int m) {
        const bool in = inRow(8 * m + e - g - phase);
        bool miss = in & rowA & !cA.holds(task.tag);
        if constexpr (RANK == 3) miss |= in & rowB & !cB.holds(task.tag);
        return __any(miss);
    };
    // chain: the flags of the tiles whose previous sweep this one reads (itself
    // and the two above); each sweep has its own, as several sweeps of a tile
    // run at a time
    unsigned long long *const flag = f.ws.flags;
    const long tiles = (long)f.ntA * f.ntB, flagged = task.sweep * tiles + tile;
    long watch = -1;
    if constexpr (CHAIN) {
        const long before = flagged - tiles;
        if (task.sweep > 0) watch = lane == 0 ? before : lane == 1 && ta + 1 < f.ntA ? before + f.ntB : lane == 2 && tb + 1 < f.ntB ? before + 1 : -1;
    }
    unsigned long long seen = 0;
    // chunk c may be loaded: the chunk stored at step block c + 1 is in memory
    auto await = [&](int c) {
        if constexpr (CHAIN) {
            if (task.sweep == 0) return;
            const unsigned long long need = (unsigned long long)(task.tag - 1) << 32 | (unsigned)(c + 2);
            while (__any(watch >= 0 && seen < need)) {
                if (watch >= 0 && seen < need) seen = __hip_atomic_load(flag + watch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            asm volatile("" ::: "memory");   // no element is loaded before its flag
        }
    };
    auto publish = [&](int count) {
        if (lane == 0) __hip_atomic_store(flag + flagged, (unsigned long long)task.tag << 32 | (unsigned)count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };

    await(1);
    issue(even, 0);
    issue(odd, 1);
    commit(even, 0);
    commit(odd, 1);
    fetch(0);
    await(3);
    issue(even, 2);
    issue(odd, 3);
    const bool mine = p < na && q < nb, whole = na == S::PA && nb == S::PB;
    T *const row = ring + rowAt(p, q);
    T prev = f.base[rowOff(p, q) + clampTo(f.lo[K] - 1, f.rlo[K], f.rhi[K])];   // the element before the first point
    readHere(prev);   // (waited for here, not by every block of steps)
    asm volatile("" ::: "memory");
    // upper neighbours are read two steps ahead (an LDS read takes longer than
    // what is left of a step once its operands are there); slots 1 and 2 of a
    // row with little ahead come with chunk 2, in block 0
    T c{}, kp{}, ip{}, jp{}, kp2{}, ip2{}, jp2{};
    auto first = [&]() {
        c = row[0], kp = row[1], kp2 = row[2];
        ip = row[S::BP + 1], ip2 = row[S::BP + 2];
        if constexpr (RANK == 3) jp = row[S::QP + 1], jp2 = row[S::QP + 2];
    };
    // every lane inside the loop at every step of block m
    auto inner = [&](int m) { return whole && 8 * m >= SKEW + phase && 8 * m + 7 < n + phase; };
    // eight steps; IN: every lane is inside the loop in all of them
    auto walk = [&](int m, auto in) {
        const T *before = row + (unsigned)(m + 2) % 3u * 8, *after = row + (unsigned)(m + 1) % 3u * 8;
        T *now = row + (unsigned)m % 3u * 8;
        // lower neighbours: what the lanes before did a step ago (their prev),
        // at the tile's edge the row below (there since the block began: read
        // ahead too); along the first axis of a rank 3 tile they are eight
        // lanes away: through LDS
        constexpr int EDGE = RANK == 3 ? S::QP : S::BP;
        T edge = before[7 - EDGE], edge1 = now[-EDGE], edge2{};
#pragma unroll
        for (int u = 0; u < 8; u++) {
            T low{};
            if constexpr (RANK == 3) low = (u == 0 ? before + 7 : now + u - 1)[-S::BP];
            const T *up = u < 5 ? now + u + 3 : after + u - 5;
            const T kp3 = up[0], ip3 = up[S::BP];
            T jp3{};
            if constexpr (RANK == 3) jp3 = up[S::QP];
            if (u < 6) edge2 = now[u + 1 - EDGE];
            T v[1 + 2 * RANK];
            v[0] = c;
            if constexpr (RANK == 3) {
                readHere(low);
                const T left = laneBelow(prev, prev);
                v[1] = low;
                v[3] = q == 0 ? edge : left;
                v[4] = jp;
            } else {
                v[1] = laneBelow(prev, edge);
            }
            v[2] = ip;
            v[1 + 2 * K] = prev;
            v[2 + 2 * K] = kp;
            const int r = 8 * m + u - p - q - phase;
            if (decltype(in)::value || (mine & inRow(r))) {
                body(v, a0 + p, RANK == 3 ? b0 + q : (I)r, (I)r);
                now[u] = v[0];
                prev = v[0];
            }
            asm volatile("" ::: "memory");   // the next step's lanes read what this one wrote
            c = kp;
            kp = kp2;
            kp2 = kp3;
            ip = ip2;
            ip2 = ip3;
            jp = jp2;
            jp2 = jp3;
            edge = edge1;
            edge1 = edge2;
        }
    };
    // next: the set that holds chunk m + 2 and takes m + 4
    auto block = [&](int m, Ahead &next) {
        // chunk m - 1 is done: out to memory, its slots take chunk m + 2
        const int c8 = chunk8(m + 2);
        T out[8];
#pragma unroll
        for (int it = 0; it < 8; it++) out[it] = ring[rowAt(rowP(it), rowQ(it)) + slotOf(it, c8)];
        asm volatile("" ::: "memory");
        commit(next, m + 2);
        if (CHAIN && m >= 1) {
            // the stores of the blocks before: at least nine younger loads follow them
            asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
            publish(m);
        }
        if (m < blocks) {
            if (missing(m)) {
                do {
                    fetch(m);
                    readHere(cA.w);
                    readHere(cB.w);
                    asm volatile("" ::: "memory");
                } while (missing(m));
            }
            T *to = ring + (unsigned)(8 * m + e + SLOTS - 1) % SLOTS;   // the lanes above read them a slot lower
            if (rowA) to[rowAt(-1, RANK == 3 ? g : 0)] = cA.value();
            if (RANK == 3 && rowB) to[rowAt(g, -1)] = cB.value();
        }
        const int s8 = 8 * m - 16;   // slots s8 + ahead
        T *const x = f.base + s8;
        auto put = [](T *to, T v) {
            if (CHAIN) agentStore(to, v);
            else *to = v;
        };
        if (inner(m - 2) & inner(m - 1)) {
#pragma unroll
            for (int it = 0; it < 8; it++) put(x + (off[it] + ahead[it]), out[it]);
        } else {
#pragma unroll
            for (int it = 0; it < 8; it++)
                if ((rowP(it) < na) & (rowQ(it) < nb) & inRow(s8 + ahead[it] - rowP(it) - rowQ(it) - phase)) put(x + (off[it] + ahead[it]), out[it]);
        }
        fetch(m + 1);   // before the row loads, so that waiting for it leaves those in flight
        await(m + 4);
        issue(next, m + 4);
        if (m < blocks) {
            asm volatile("" ::: "memory");
            if (m == 0) first();
            if (inner(m)) walk(m, std::true_type());
            else walk(m, std::false_type());
            // the upper faces' rows: what lanes (PA - 1, .) and (., PB - 1) did in this block
            const T *done = ring + (unsigned)m % 3u * 8 + e;
            if (toA) FlowCells<T>::store(outA, m * FLOW_CELLS_BYTES, done[rowAt(S::PA - 1, RANK == 3 ? g : 0)], task.tag);
            if (RANK == 3 && toB) FlowCells<T>::store(outB, m * FLOW_CELLS_BYTES, done[rowAt(g, S::PB - 1)], task.tag);
            asm volatile("" ::: "memory");
        }
    };
    for (int m = 0; m < blocks + 2; m += 2) {
        block(m, even);
        block(m + 1, odd);   // (one too many of an odd number stores nothing)
    }
    if (CHAIN) {
        storesDone();
        publish(0x7fffffff);
    }
}

// ------------------------------------------------------------------ scheduling
// Workgroup id -> logical tile id such that each XCD gets a contiguous range.
__device__ __forceinline__ long xcdTile(long wg, long n, int enable) {
    if (!enable) return wg;
    const long X = 8;
    long per = n / X, rem = n % X;
    long x = wg % X, q = wg / X;
    return x < rem ? x * (per + 1) + q : rem * (per + 1) + (x - rem) * per + q;
}

}  // namespace dvmh_dev

#endif
