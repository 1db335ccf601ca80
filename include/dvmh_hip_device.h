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
// of row (p, q) in slot r + p + q), so in every step all lanes use the same
// slots, at offsets known to the compiler, and a finished block of steps is
// stored at once.  A block's loads and stores move 64 bytes of eight rows per
// instruction; two blocks' loads are in flight while one is walked.  Rows a
// tile needs from its lower neighbours come through cells in device memory: a
// value in halves, each in an 8-byte word with a 32-bit tag that no earlier
// launch used, so one load tells whether it is there.
//
// Bound by the chain of dependent steps: 0.12 us a step for rank 2 (eight
// dependent FP64 operations and a lane shift), 0.155 for rank 3 (one neighbour
// through LDS), and along a diagonal of tiles, per tile, the lanes' skew plus
// about 4 us until a finished block is seen by the next tile.  Measured, one
// sweep with reductions: 2-D 998^2 0.38 ms (a launch per hyperplane: 9.2), 3-D
// 128^3 0.154 ms (a launch per tile-plane: 0.43), 318^3 0.76 ms (1.84).
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

// A cell: the value's bytes in 32-bit parts, each beside the tag.
template <typename T>
struct FlowCell {
    static constexpr int WORDS = sizeof(T) > 4 ? 2 : 1;
    unsigned long long w[WORDS];
    __device__ __forceinline__ void load(const unsigned long long *p) {
#pragma unroll
        for (int i = 0; i < WORDS; i++) w[i] = __hip_atomic_load(p + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ bool holds(unsigned tag) const {
        bool h = true;
#pragma unroll
        for (int i = 0; i < WORDS; i++) h &= (unsigned)(w[i] >> 32) == tag;
        return h;
    }
    __device__ __forceinline__ T value() const {
        unsigned x[2] = {(unsigned)w[0], (unsigned)w[WORDS - 1]};
        T v;
        __builtin_memcpy(&v, x, sizeof(T));
        return v;
    }
    static __device__ __forceinline__ void store(unsigned long long *p, T v, unsigned tag) {
        unsigned x[2] = {0, 0};
        __builtin_memcpy(x, &v, sizeof(T));
#pragma unroll
        for (int i = 0; i < WORDS; i++)
            __hip_atomic_store(p + i, (unsigned long long)tag << 32 | x[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};

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

// x is in its register here (its load is issued before, not sunk to its use).
template <typename T>
__device__ __forceinline__ void readHere(T &x) { asm volatile("" : "+v"(x)); }

// Walks the task's tile.  body(v, t0, t1, t2) runs the loop body at position
// (t0, t1, t2) of the loop (t2 unused for rank 2) with v the star around it.
// CHAIN: several sweeps of the array in one launch; its elements then pass
// between workgroups, so they are loaded and stored at agent scope, and a
// tile's flag says how many blocks of which sweep are in memory.
template <typename T, typename I, int RANK, bool CHAIN, typename Body>
__device__ __forceinline__ void flowTile(const FlowArgs<T, I, RANK> &f, const FlowTask &task, T *ring, Body &&body) {
    using S = FlowShape<RANK>;
    constexpr int K = RANK - 1, SKEW = S::PA + S::PB - 2, SLOTS = 24;
    const int lane = threadIdx.x, g = lane >> 3, e = lane & 7;   // block transfers: eight rows of eight elements
    const int p = RANK == 3 ? g : lane, q = RANK == 3 ? e : 0;   // the lane's own row
    const int ta = task.ta, tb = task.tb;
    const I a0 = (I)ta * S::PA, b0 = (I)tb * S::PB;
    const int na = f.cnt[0] - a0 < S::PA ? (int)(f.cnt[0] - a0) : S::PA;
    const int nb = RANK == 2 ? 1 : (f.cnt[1] - b0 < S::PB ? (int)(f.cnt[1] - b0) : S::PB);
    const int n = (int)f.cnt[K];
    const int blocks = (n + na + nb - 2 + 7) >> 3;   // blocks of steps
    auto clampTo = [](I x, I lo, I hi) { return x < lo ? lo : (x > hi ? hi : x); };
    auto rowOff = [&](int pp, int qq) -> I {
        I o = clampTo(f.lo[0] + a0 + pp, f.rlo[0], f.rhi[0]) * f.s[0];
        if constexpr (RANK == 3) o += clampTo(f.lo[1] + b0 + qq, f.rlo[1], f.rhi[1]) * f.s[1];
        return o;
    };
    auto rowAt = [](int pp, int qq) { return (pp + 1) * S::BP + (qq + 1) * S::QP; };
    // the row a lane moves in transfer `it` of a block
    auto rowP = [&](int it) { return RANK == 3 ? it : it * 8 + g; };
    auto rowQ = [&](int) { return RANK == 3 ? g : 0; };
    // rows moved block by block: the tile's 64, the ones above it and, at the
    // array's lower edges, the ones below it (elsewhere those come in cells)
    const bool edgeA = ta == 0, edgeB = RANK == 3 && tb == 0;
    I off[8];
#pragma unroll
    for (int it = 0; it < 8; it++) off[it] = rowOff(rowP(it), rowQ(it));
    const I offA = rowOff(S::PA, g), offB = RANK == 3 ? rowOff(g, S::PB) : 0;
    const I offLA = rowOff(-1, g), offLB = RANK == 3 ? rowOff(g, -1) : 0;
    const int gq = RANK == 3 ? g : 0;   // second coordinate of a face row of the first axis
    // two blocks' loads are in flight while a block is walked (a block of steps
    // takes less than a round trip to memory), in two sets of registers
    struct Ahead {
        T own[8], vA, vB, vLA, vLB;
    } even{}, odd{};
    // (issued on every path, past the row's end from its last element, so that
    // the waits know how many younger loads may stay in flight)
    auto issue = [&](Ahead &h, int b) {
        const I k = f.lo[K] + 8 * b + e;
        auto ld = [&](I o, int skew) -> T {
            const T *x = f.base + (o + clampTo(k - skew, f.rlo[K], f.rhi[K]));
            return CHAIN ? agentLoad(x) : *x;
        };
#pragma unroll
        for (int it = 0; it < 8; it++) h.own[it] = ld(off[it], rowP(it) + rowQ(it));
        h.vA = ld(offA, S::PA + gq);
        if constexpr (RANK == 3) h.vB = ld(offB, g + S::PB);
        if (edgeA) h.vLA = ld(offLA, gq - 1);
        if constexpr (RANK == 3) if (edgeB) h.vLB = ld(offLB, g - 1);
    };
    auto commit = [&](const Ahead &h, int b) {
        T *to = ring + (b % 3) * 8 + e;
#pragma unroll
        for (int it = 0; it < 8; it++) to[rowAt(rowP(it), rowQ(it))] = h.own[it];
        if constexpr (RANK == 3) {
            to[rowAt(S::PA, g)] = h.vA;
            to[rowAt(g, S::PB)] = h.vB;
            if (edgeA) to[rowAt(-1, g)] = h.vLA;
            if (edgeB) to[rowAt(g, -1)] = h.vLB;
        } else if (g == 0) {
            to[rowAt(S::PA, 0)] = h.vA;
            if (edgeA) to[rowAt(-1, 0)] = h.vLA;
        }
    };
    // cells of a tile's upper faces: PB rows of n towards ta + 1, PA rows towards tb + 1
    constexpr int W = FlowCell<T>::WORDS;
    const long tiles = (long)f.ntA * f.ntB, tile = (long)ta * f.ntB + tb;
    unsigned long long *const cellsA = f.ws.cells, *const cellsB = f.ws.cells + tiles * S::PB * n * W;
    const bool fromA = ta > 0, fromB = RANK == 3 && tb > 0;
    const bool toA = ta + 1 < f.ntA, toB = RANK == 3 && tb + 1 < f.ntB;
    // lane (g, e) fetches element 8 m + e - g of face row g: what lane (0, g)
    // (or (g, 0)) needs at step e of block m
    const bool rowA = fromA && g < nb, rowB = fromB && g < na;
    auto inRow = [&](int r) { return (unsigned)r < (unsigned)n; };
    auto cellOf = [&](unsigned long long *c, long t, int rows, int r) { return c + ((t * rows + g) * n + r) * W; };
    unsigned long long *const inA = cellOf(cellsA, tile - f.ntB, S::PB, 0), *const inB = cellOf(cellsB, tile - 1, S::PA, 0);
    unsigned long long *const outA = cellOf(cellsA, tile, S::PB, 0), *const outB = cellOf(cellsB, tile, S::PA, 0);
    // (every lane loads something, some the first cell in vain: a load in a
    // branch would have to be waited for at the branch's end)
    FlowCell<T> cA{}, cB{};
    auto fetch = [&](int m) {
        const int r = 8 * m + e - g;
        cA.load(rowA & inRow(r) ? inA + r * W : cellsA);
        if constexpr (RANK == 3) cB.load(rowB & inRow(r) ? inB + r * W : cellsA);
    };
    auto missing = [&](int m) {
        const bool in = inRow(8 * m + e - g);
        bool miss = in & rowA & !cA.holds(task.tag);
        if constexpr (RANK == 3) miss |= in & rowB & !cB.holds(task.tag);
        return __any(miss);
    };
    // chain: the flags of the tiles whose previous sweep this one reads (itself
    // and the two above); each sweep has its own, as several sweeps of a tile
    // run at a time
    unsigned long long *const flag = f.ws.flags;
    const long flagged = task.sweep * tiles + tile;
    long watch = -1;
    if constexpr (CHAIN) {
        const long before = flagged - tiles;
        if (task.sweep > 0) watch = lane == 0 ? before : lane == 1 && ta + 1 < f.ntA ? before + f.ntB : lane == 2 && tb + 1 < f.ntB ? before + 1 : -1;
    }
    unsigned long long seen = 0;
    auto await = [&](int b) {
        if constexpr (CHAIN) {
            if (task.sweep == 0) return;
            const int most = (n + SKEW + 7) >> 3;
            const unsigned long long need = (unsigned long long)(task.tag - 1) << 32 | (unsigned)(b + 1 < most ? b + 1 : most);
            while (__any(watch >= 0 && seen < need)) {
                if (watch >= 0 && seen < need) seen = __hip_atomic_load(flag + watch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            asm volatile("" ::: "memory");   // no element is loaded before its flag
        }
    };
    auto publish = [&](int count) {
        if (lane == 0) __hip_atomic_store(flag + flagged, (unsigned long long)task.tag << 32 | (unsigned)count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };

    await(0);
    issue(even, 0);
    commit(even, 0);
    await(1);
    issue(odd, 1);
    await(2);
    issue(even, 2);
    // the lower edge rows' elements before the first block's
    if (lane == 0) {
        if (edgeA) ring[rowAt(-1, 0) + SLOTS - 1] = f.base[rowOff(-1, 0) + f.lo[K]];
        if (edgeB) ring[rowAt(0, -1) + SLOTS - 1] = f.base[rowOff(0, -1) + f.lo[K]];
    }
    fetch(0);
    const bool mine = p < na && q < nb, whole = na == S::PA && nb == S::PB;
    T *const row = ring + rowAt(p, q);
    T prev = f.base[rowOff(p, q) + clampTo(f.lo[K] - 1, f.rlo[K], f.rhi[K])];   // the element before the first point
    readHere(prev);   // (waited for here, not by every block of steps)
    asm volatile("" ::: "memory");
    // upper neighbours are read two steps ahead (an LDS read takes longer than
    // what is left of a step once its operands are there)
    T c = row[0], kp = row[1], ip = row[S::BP + 1], jp{}, kp2 = row[2], ip2 = row[S::BP + 2], jp2{};
    if constexpr (RANK == 3) {
        jp = row[S::QP + 1];
        jp2 = row[S::QP + 2];
    }
    // eight steps; GUARD: some lanes are outside the loop in some of them
    auto walk = [&](int m, auto guard) {
        const T *before = row + (m + 2) % 3 * 8, *after = row + (m + 1) % 3 * 8;
        T *now = row + m % 3 * 8;
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
                const T beside = laneBelow(prev, prev);
                v[1] = low;
                v[3] = q == 0 ? edge : beside;
                v[4] = jp;
            } else {
                v[1] = laneBelow(prev, edge);
            }
            v[2] = ip;
            v[1 + 2 * K] = prev;
            v[2 + 2 * K] = kp;
            const int r = 8 * m + u - p - q;
            if (!decltype(guard)::value || (mine && r >= 0 && r < n)) {
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
    // every lane inside the loop at every step of block m
    auto inner = [&](int m) { return whole && 8 * m >= SKEW && 8 * m + 7 < n; };
    // next: the set that holds block m + 1 and takes m + 3
    auto block = [&](int m, Ahead &next) {
        T out[8];   // block m - 1, on its way to memory
#pragma unroll
        for (int it = 0; it < 8; it++) out[it] = ring[rowAt(rowP(it), rowQ(it)) + (m + 2) % 3 * 8 + e];
        asm volatile("" ::: "memory");
        commit(next, m + 1);
        if (CHAIN && m >= 2) {
            storesDone();   // those of block m - 2, a block of steps ago
            publish(m - 1);
        }
        if (m < blocks) {
            if (missing(m)) {
                do {
                    fetch(m);
#pragma unroll
                    for (int i = 0; i < W; i++) {
                        readHere(cA.w[i]);
                        readHere(cB.w[i]);
                    }
                } while (missing(m));
            }
            T *to = ring + (unsigned)(8 * m + e + SLOTS - 1) % SLOTS;   // the lanes above read them a slot lower
            const bool in = inRow(8 * m + e - g);
            if (in & rowA) to[rowAt(-1, g)] = cA.value();
            if (RANK == 3 && (in & rowB)) to[rowAt(g, -1)] = cB.value();
        }
        if (m > 0) {
            T *x = f.base + f.lo[K] + 8 * (m - 1) + e;
            auto put = [](T *to, T v) {
                if (CHAIN) agentStore(to, v);
                else *to = v;
            };
            if (inner(m - 1)) {
#pragma unroll
                for (int it = 0; it < 8; it++) put(x + (off[it] - rowP(it) - rowQ(it)), out[it]);
            } else {
#pragma unroll
                for (int it = 0; it < 8; it++) {
                    const int skew = rowP(it) + rowQ(it);
                    if ((rowP(it) < na) & (rowQ(it) < nb) & inRow(8 * (m - 1) + e - skew)) put(x + (off[it] - skew), out[it]);
                }
            }
        }
        fetch(m + 1);   // before the row loads, so that waiting for it leaves those in flight
        await(m + 3);
        issue(next, m + 3);
        if (m < blocks) {
            asm volatile("" ::: "memory");
            if (inner(m)) walk(m, std::false_type());
            else walk(m, std::true_type());
            // the upper faces' rows: what lanes (PA - 1, .) and (., PB - 1) did in this block
            const T *done = ring + m % 3 * 8 + e;
            const int rA = 8 * m + e - (S::PA - 1) - g;
            if (toA & (g < nb) & inRow(rA)) FlowCell<T>::store(outA + rA * W, done[rowAt(S::PA - 1, gq)], task.tag);
            if constexpr (RANK == 3) {
                const int rB = 8 * m + e - (S::PB - 1) - g;
                if (toB & (g < na) & inRow(rB)) FlowCell<T>::store(outB + rB * W, done[rowAt(g, S::PB - 1)], task.tag);
            }
            asm volatile("" ::: "memory");
        }
    };
    for (int m = 0; m < blocks + 1; m += 2) {
        block(m, odd);
        block(m + 1, even);   // (one too many of an odd number stores nothing)
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
