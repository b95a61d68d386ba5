// solver_common.hpp -- device building blocks shared by the single-system
// PCG (pcg.hip) and the batched persistent PCG (batch.hip): coherent loads,
// the last-block reduction handshake, and the CSR / node-block sliced row
// engines.
#pragma once

#include "sfem_internal.hpp"

namespace sfem {
namespace {

constexpr double kEps64 = 2.220446049250313e-16;  // FP64 unit roundoff x 2

// Global-address-space view of a device pointer.  Pointers read from memory
// (the batch descriptors) are generic to the compiler, which then emits flat
// loads; accessing through these views gives global loads and stores.
#define SFEM_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ const SFEM_GLOBAL T* glb(const T* p) { return (const SFEM_GLOBAL T*)p; }
template <typename T>
__device__ __forceinline__ SFEM_GLOBAL T* glb(T* p) { return (SFEM_GLOBAL T*)p; }

constexpr int kThreads = 256;

// ------------------------------------------------------------ helpers --
__device__ __forceinline__ double ld_coherent(const double* p) {
    unsigned long long v =
        __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __longlong_as_double((long long)v);
}

// Agent-coherent store of a block's partial result: it bypasses the XCD's L2
// (per-XCD L2s are not coherent with each other) so the last block, on any
// XCD, reads it with ld_coherent.
__device__ __forceinline__ void st_coherent(double* p, double v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until this wave's outstanding vector memory operations, stores
// included, have completed (GFX9 s_waitcnt: vmcnt(0), expcnt and lgkmcnt
// left at their maxima).
__device__ __forceinline__ void wait_vm_complete() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// True in every thread of the block that arrives last.  Thread 0 must have
// written this block's partials with st_coherent before the call; it waits for
// those stores to complete before its counter increment.  Unlike
// __threadfence() this does not write back and invalidate the whole L2, which
// would evict the vector every other block is still gathering from.
// The arrivals are spread over 8 counters: block b arrives on counter b % 8,
// the last block of each of those groups then on the top counter.  One
// agent-scope counter for every block serialises the arrivals (about 12 ns
// each on MI355X, 50 us for 4,096 blocks); spread over 8 counters 256 bytes
// apart they cost about 1.3 ns each.  The last block resets every counter.
__device__ __forceinline__ bool last_block_arrive(Arrivals* a) {
    __shared__ int is_last;
    __syncthreads();
    if (threadIdx.x == 0) {
        wait_vm_complete();
        const unsigned G = gridDim.x, g = blockIdx.x % 8u;
        const unsigned groups = G < 8u ? G : 8u, in_group = (G - g + 7u) / 8u;
        bool last = __hip_atomic_fetch_add(&a->c[64 * g], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                    in_group - 1u;
        if (last)
            last = __hip_atomic_fetch_add(&a->c[64 * 8], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                   groups - 1u;
        if (last)
            for (int k = 0; k < 9; ++k)
                __hip_atomic_store(&a->c[64 * k], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        is_last = last;
    }
    __syncthreads();
    return is_last;
}

// Fixed-order sums of nparts partial W-tuples (stride W) by one block:
// thread t adds parts t, t + 256, t + 512, ... in that order (component by
// component), then the block sums.  The coherent loads go out U parts at a
// time (each one a round trip past the L2; at most 8 values in flight, so
// the kernels that end in this reduction keep their register budget), the
// additions stay in order.
template <int W>
__device__ __forceinline__ void thread_partials(const double* partials, int nparts, double (&s)[W]) {
    constexpr int U = W >= 8 ? 1 : 8 / W;
#pragma unroll
    for (int k = 0; k < W; ++k) s[k] = 0.0;
    int i = threadIdx.x;
    for (; i + (U - 1) * kThreads < nparts; i += U * kThreads) {
        double v[U][W];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < W; ++k) v[u][k] = ld_coherent(partials + (int64_t)W * (i + u * kThreads) + k);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < W; ++k) s[k] += v[u][k];
    }
    for (; i < nparts; i += kThreads)
#pragma unroll
        for (int k = 0; k < W; ++k) s[k] += ld_coherent(partials + (int64_t)W * i + k);
}

// Fixed-order sum of nparts partial triples (stride 3) by one block.
__device__ __forceinline__ void sum_partials3(const double* partials, int nparts, double* a, double* b, double* c,
                                              double* sh) {
    double s[3];
    thread_partials<3>(partials, nparts, s);
    *a = block_sum_256(s[0], sh);
    *b = block_sum_256(s[1], sh + 4);
    *c = block_sum_256(s[2], sh);
}

// Sum over a block of NW wavefronts, in every thread (sh: NW slots); the
// order is fixed: butterfly per wavefront, then the wavefronts pairwise.
template <int NW>
__device__ __forceinline__ double block_sum_waves(double v, double* sh) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double t[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) t[i] = sh[i];
#pragma unroll
    for (int h = NW / 2; h > 0; h >>= 1)
#pragma unroll
        for (int i = 0; i < h; ++i) t[i] += t[i + h];
    __syncthreads();
    return t[0];
}

// Sums of nparts partial W-tuples (stride W) an earlier kernel on the stream
// left, by a block of NW wavefronts, in every thread.  Every block of a
// kernel that needs the sums calls it for itself and gets the same bits.
template <int W, int NW>
__device__ __forceinline__ void sum_parts_all(const double* __restrict__ partials, int nparts, double (&out)[W],
                                              double* sh) {
    double s[W];
#pragma unroll
    for (int k = 0; k < W; ++k) s[k] = 0.0;
#pragma unroll 2
    for (int i = threadIdx.x; i < nparts; i += NW * 64)
#pragma unroll
        for (int k = 0; k < W; ++k) s[k] += partials[(int64_t)W * i + k];
#pragma unroll
    for (int k = 0; k < W; ++k) out[k] = block_sum_waves<NW>(s[k], sh);
}

// Logical block id: consecutive logical blocks land on the same XCD (the
// hardware deals workgroups round-robin over the 8 XCDs), so each XCD's L2
// sees a contiguous part of the rows and of the gathered vector.
__device__ __forceinline__ int64_t logical_block() {
    const int64_t g = gridDim.x, b = blockIdx.x;
    if (g % 8) return b;
    return (b % 8) * (g / 8) + b / 8;
}

template <typename T>
__device__ __forceinline__ T fmaT(T a, T b, T c) { return fma(a, b, c); }

// ------------------------------------------------------- operator rows --
// CSR, G lanes per row.  Returns the row sum in every lane of the group.
template <int G, typename TV, typename ACC, typename Gather>
__device__ __forceinline__ ACC csr_row(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                       const TV* __restrict__ val, int64_t row, int lane, Gather gx) {
    ACC s = 0;
    const int32_t e = rowptr[row + 1];
#pragma unroll 4  // the loads of four strides in flight; the same order of operations
    for (int32_t k = rowptr[row] + lane; k < e; k += G) s = fmaT<ACC>((ACC)val[k], gx(col[k]), s);
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    return s;
}

// csr_row plus sum_k |val_k x_k| (the scale of the rounding error of the row
// sum, for the attainable-residual estimate).
template <int G, typename Gather>
__device__ __forceinline__ double csr_row_abs(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                              const double* __restrict__ val, int64_t row, int lane, Gather gx,
                                              double* aout) {
    double s = 0.0, a = 0.0;
    const int32_t e = rowptr[row + 1];
#pragma unroll 4
    for (int32_t k = rowptr[row] + lane; k < e; k += G) {
        const double v = val[k], x = gx(col[k]);
        s = fma(v, x, s);
        a = fma(fabs(v), fabs(x), a);
    }
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) {
        s += __shfl_xor(s, off, 64);
        a += __shfl_xor(a, off, 64);
    }
    *aout = a;
    return s;
}

// Matrix streams are read once per SpMV: with NT the loads carry the
// non-temporal hint so they do not evict the gathered vector from the caches.
template <bool NT, typename V>
__device__ __forceinline__ V ld_stream(const V* p) {
    if constexpr (NT) return __builtin_nontemporal_load(glb(p));
    else return *glb(p);
}

// Operator value sources of the sliced format.  Vals<double> / Vals<float>
// read one plane array; Vals<SplitVal> reads the FP32 rounding of each FP64
// value plus a 16-bit correction and rebuilds v = hi + lo * ulp(hi) * 2^-16
// exactly in FP64 (|v' - v| <= 2^-39 |v|): 6 bytes per value.
struct SplitVal {};

// `raw` loads a value as stored and `decode` turns it into the arithmetic
// type, so a caller can issue many loads before it uses any of them.
template <typename TV>
struct Vals {
    const TV* v;
    using Raw = TV;
    template <bool NT>
    __device__ __forceinline__ Raw raw(int64_t i) const { return ld_stream<NT>(v + i); }
    __device__ __forceinline__ TV decode(Raw r) const { return r; }
    template <bool NT>
    __device__ __forceinline__ TV get(int64_t i) const { return ld_stream<NT>(v + i); }
};

template <>
struct Vals<SplitVal> {
    const float* hi;
    const int16_t* lo;
    struct Raw {
        float h;
        int l;
    };
    template <bool NT>
    __device__ __forceinline__ Raw raw(int64_t i) const {
        return Raw{ld_stream<NT>(hi + i), (int)ld_stream<NT>(lo + i)};
    }
    __device__ __forceinline__ double decode(Raw r) const {
        // ulp(h) * 2^-16 = 2^(exponent(h) - 23 - 16); below the normal range
        // (|h| < 2^-87, where lo is 0 by construction) the scale is 0
        const float scale = __int_as_float(max((__float_as_int(r.h) & 0x7F800000) - (39 << 23), 0));
        return fma((double)r.l, (double)scale, (double)r.h);
    }
    template <bool NT>
    __device__ __forceinline__ double get(int64_t i) const { return decode(raw<NT>(i)); }
};

// Node-block sliced format: this lane's block row of slice `sl`.
template <int BS, typename TV, typename ACC, bool NT = false, typename Gather>
__device__ __forceinline__ void sell_row(const int64_t* __restrict__ sl_ptr, const int32_t* __restrict__ sl_w,
                                         const int32_t* __restrict__ scol, Vals<TV> vals, int64_t sl, int lane,
                                         Gather gx, ACC out[BS]) {
    constexpr int B2 = BS * BS;
    const int64_t base = glb(sl_ptr)[sl];
    const int w = glb(sl_w)[sl];
#pragma unroll
    for (int j = 0; j < BS; ++j) out[j] = 0;
#pragma unroll 2
    for (int k = 0; k < w; ++k) {
        const int64_t slot = base + (int64_t)k * 64;
        const int64_t c = ld_stream<NT>(scol + slot + lane);
        ACC xv[BS];
#pragma unroll
        for (int i = 0; i < BS; ++i) xv[i] = gx(c * BS + i);
        const int64_t v = slot * B2 + lane;
#pragma unroll
        for (int j = 0; j < BS; ++j)
#pragma unroll
            for (int i = 0; i < BS; ++i)
                out[j] = fmaT<ACC>((ACC)vals.template get<NT>(v + (j * BS + i) * 64), xv[i], out[j]);
    }
}

// A slice shared by a block of 4 wavefronts: wavefront `part` takes the block
// columns part, part + 4, ... of the slice's 64 block rows (sell_combine adds
// the four sums).  load() issues what does not depend on the gathered vector:
// the first PRE column ids and PV columns of values; a column past the row's
// end repeats its last one, and apply() drops it.  PRE is 8 (all ids of a Hex8
// row) where the values take 32 bits: 96x24x24, mixed, 72 -> 69 ms; with
// 64-bit values the registers cost a wavefront per SIMD (64x16x16, FP64,
// 24.8 -> 26.8 ms).
template <int BS, typename TV, bool NT = false>
struct SharedSlice {
    using Raw = typename Vals<TV>::Raw;
    static constexpr int B2 = BS * BS, SPLIT = kThreads / 64, PRE = sizeof(Raw) == 4 ? 8 : 4, PV = 2;
    const int32_t* scol;
    Vals<TV> vals;
    int64_t base = 0;
    int w = 0, part, lane;
    int32_t pc[PRE] = {};
    Raw pv[PV][B2] = {};

    __device__ __forceinline__ SharedSlice(const int32_t* scol_, Vals<TV> vals_) : scol(scol_), vals(vals_) {
        part = threadIdx.x >> 6;
        lane = threadIdx.x & 63;
    }
    __device__ __forceinline__ int64_t column(int u) const {
        return base + (int64_t)min(part + u * SPLIT, w - 1) * 64;
    }
    __device__ __forceinline__ void load(const int64_t* __restrict__ sl_ptr, const int32_t* __restrict__ sl_w,
                                         int64_t sl) {
        base = glb(sl_ptr)[sl];
        w = glb(sl_w)[sl];
        if (w <= 0) return;
#pragma unroll
        for (int u = 0; u < PRE; ++u) pc[u] = ld_stream<NT>(scol + column(u) + lane);
#pragma unroll
        for (int u = 0; u < PV; ++u)
#pragma unroll
            for (int m = 0; m < B2; ++m) pv[u][m] = vals.template raw<NT>(column(u) * B2 + lane + m * 64);
    }
    // acc += this wavefront's columns; gx(c, x) gathers block row c
    template <typename ACC, typename Gather>
    __device__ __forceinline__ void apply(Gather gx, ACC (&acc)[BS]) const {
        if (w <= 0) return;
#pragma unroll
        for (int u = 0; u < PRE; ++u) {
            if (u == 4 && u * SPLIT >= w) return;
            const bool in = part + u * SPLIT < w;
            Raw rv[B2];
#pragma unroll
            for (int m = 0; m < B2; ++m)
                rv[m] = u < PV ? pv[u < PV ? u : 0][m] : vals.template raw<NT>(column(u) * B2 + lane + m * 64);
            ACC xv[BS];
            gx((int64_t)pc[u], xv);
#pragma unroll
            for (int i = 0; i < BS; ++i) xv[i] = in ? xv[i] : ACC(0);
#pragma unroll
            for (int j = 0; j < BS; ++j)
#pragma unroll
                for (int i = 0; i < BS; ++i) acc[j] = fmaT<ACC>((ACC)vals.decode(rv[j * BS + i]), xv[i], acc[j]);
        }
#pragma unroll 2
        for (int k = part + PRE * SPLIT; k < w; k += SPLIT) {
            const int64_t slot = base + (int64_t)k * 64;
            ACC xv[BS];
            gx((int64_t)ld_stream<NT>(scol + slot + lane), xv);
#pragma unroll
            for (int j = 0; j < BS; ++j)
#pragma unroll
                for (int i = 0; i < BS; ++i)
                    acc[j] = fmaT<ACC>((ACC)vals.template get<NT>(slot * B2 + lane + (j * BS + i) * 64), xv[i], acc[j]);
        }
    }
};

// The block columns part, part + SPLIT, ... of this lane's block row in FP64
// (SPLIT wavefronts share a slice; their sums are added by sell_combine), and
// aout[j] = sum |M_ji x_i|.  gx(c, x) gathers block row c of the vector.
template <int BS, int SPLIT, typename Gather>
__device__ __forceinline__ void sell_row_abs_part(const int64_t* __restrict__ sl_ptr, const int32_t* __restrict__ sl_w,
                                                  const int32_t* __restrict__ scol, const double* __restrict__ sval,
                                                  int64_t sl, int lane, int part, Gather gx, double out[BS],
                                                  double aout[BS]) {
    constexpr int B2 = BS * BS;
    const int64_t base = glb(sl_ptr)[sl];
    const int w = glb(sl_w)[sl];
#pragma unroll
    for (int j = 0; j < BS; ++j) out[j] = aout[j] = 0.0;
    auto add = [&](const double (&m)[B2], const double (&xv)[BS]) {
#pragma unroll
        for (int j = 0; j < BS; ++j)
#pragma unroll
            for (int i = 0; i < BS; ++i) {
                out[j] = fma(m[j * BS + i], xv[i], out[j]);
                aout[j] = fma(fabs(m[j * BS + i]), fabs(xv[i]), aout[j]);
            }
    };
    // two block columns at a time: both columns' ids and values are in flight
    // before either gather
    int k = part;
#pragma unroll 1
    for (; k + SPLIT < w; k += 2 * SPLIT) {
        const int64_t s0 = base + (int64_t)k * 64, s1 = s0 + SPLIT * 64;
        const int64_t c0 = ld_stream<true>(scol + s0 + lane), c1 = ld_stream<true>(scol + s1 + lane);
        double m0[B2], m1[B2], x0[BS], x1[BS];
#pragma unroll
        for (int i = 0; i < B2; ++i) m0[i] = ld_stream<true>(sval + s0 * B2 + lane + i * 64);
#pragma unroll
        for (int i = 0; i < B2; ++i) m1[i] = ld_stream<true>(sval + s1 * B2 + lane + i * 64);
        gx(c0, x0);
        gx(c1, x1);
        add(m0, x0);
        add(m1, x1);
    }
    if (k < w) {
        const int64_t s0 = base + (int64_t)k * 64;
        const int64_t c0 = ld_stream<true>(scol + s0 + lane);
        double m0[B2], x0[BS];
#pragma unroll
        for (int i = 0; i < B2; ++i) m0[i] = ld_stream<true>(sval + s0 * B2 + lane + i * 64);
        gx(c0, x0);
        add(m0, x0);
    }
}

// Sums the W values each lane of SPLIT wavefronts holds for its row into the
// slice's first wavefront (parts in ascending order).  buf: one W x 64 array
// per wavefront of the block.  Every thread of the block must call it; the
// caller's buf is free again after its next barrier.
template <int W, int SPLIT, typename ACC>
__device__ __forceinline__ void sell_combine(ACC (&v)[W], ACC (*buf)[W][64]) {
    if constexpr (SPLIT > 1) {
        const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
        if (wv % SPLIT)
#pragma unroll
            for (int j = 0; j < W; ++j) buf[wv][j][lane] = v[j];
        __syncthreads();
        if (wv % SPLIT == 0)
#pragma unroll
            for (int h = 1; h < SPLIT; ++h)
#pragma unroll
                for (int j = 0; j < W; ++j) v[j] += buf[wv + h][j][lane];
    }
}

// sell_row in FP64 plus aout[j] = sum |M_ji x_i| over the row's blocks.  Per
// pair of block columns the ids and all values are loaded before any of them
// is used, then the gathers (scheduling barriers keep that order); the
// arithmetic order per row is k, then j, then i.
template <int BS, typename Gather>
__device__ __forceinline__ void sell_row_abs(const int64_t* __restrict__ sl_ptr, const int32_t* __restrict__ sl_w,
                                             const int32_t* __restrict__ scol, const double* __restrict__ sval,
                                             int64_t sl, int lane, Gather gx, double out[BS], double aout[BS]) {
    constexpr int B2 = BS * BS;
    const int64_t base = glb(sl_ptr)[sl];
    const int w = glb(sl_w)[sl];
#pragma unroll
    for (int j = 0; j < BS; ++j) out[j] = aout[j] = 0.0;
    auto step = [&](const double (&m)[B2], const double (&xv)[BS]) {
#pragma unroll
        for (int j = 0; j < BS; ++j)
#pragma unroll
            for (int i = 0; i < BS; ++i) {
                out[j] = fma(m[j * BS + i], xv[i], out[j]);
                aout[j] = fma(fabs(m[j * BS + i]), fabs(xv[i]), aout[j]);
            }
    };
    int k = 0;
    for (; k + 2 <= w; k += 2) {
        const int64_t s0 = base + (int64_t)k * 64, s1 = s0 + 64;
        const int64_t c0 = ld_stream<true>(scol + s0 + lane), c1 = ld_stream<true>(scol + s1 + lane);
        double m0[B2], m1[B2];
#pragma unroll
        for (int m = 0; m < B2; ++m) m0[m] = ld_stream<true>(sval + s0 * B2 + lane + m * 64);
#pragma unroll
        for (int m = 0; m < B2; ++m) m1[m] = ld_stream<true>(sval + s1 * B2 + lane + m * 64);
        __builtin_amdgcn_sched_barrier(0);
        double x0[BS], x1[BS];
#pragma unroll
        for (int i = 0; i < BS; ++i) x0[i] = gx(c0 * BS + i);
#pragma unroll
        for (int i = 0; i < BS; ++i) x1[i] = gx(c1 * BS + i);
        __builtin_amdgcn_sched_barrier(0);
        step(m0, x0);
        step(m1, x1);
    }
    if (k < w) {
        const int64_t s0 = base + (int64_t)k * 64;
        const int64_t c0 = ld_stream<true>(scol + s0 + lane);
        double m0[B2], x0[BS];
#pragma unroll
        for (int m = 0; m < B2; ++m) m0[m] = ld_stream<true>(sval + s0 * B2 + lane + m * 64);
#pragma unroll
        for (int i = 0; i < BS; ++i) x0[i] = gx(c0 * BS + i);
        step(m0, x0);
    }
}

// Wavefronts per slice of a sliced operator in the multigrid solve: 1, or 4 (a
// block per slice; in the outer CG p is then formed in the operator's
// gathers).  A wavefront per slice leaves a small system with fewer wavefronts
// than the device holds, each with up to 27 block columns of loads one after
// the other.  Distorted 3D grids, FP64, us per iteration with 1 / 4 wavefronts
// for the outer operator and the FP16 smoother alike: 276 slices 133 / 109,
// 1,089 174 / 149, 2,102 264 / 246, 3,752 329 / 360, 4,802 407 / 430, 8,450
// 743 / 756; with this rule (the smoother's 22 bytes a block still shared) 326,
// 389 and 717 at the last three.  2D (9 block columns): 190 slices 93 / 84,
// 1,177 130 / 126, 2,468 160 / 159, 8,452 279 / 307.  8 wavefronts gain nothing
// over 4.
constexpr double kSharedBytes = 400e6;    // 3D: operator bytes
constexpr int64_t kSharedSlices2 = 1536;  // 2D: slices
inline int slice_split(const sfem_ctx* ctx, int64_t nslices, int bs, double operator_bytes) {
    if (ctx->tune_split > 0) return ctx->tune_split >= 4 ? 4 : 1;
    return (bs == 3 ? operator_bytes <= kSharedBytes : nslices <= kSharedSlices2) ? 4 : 1;
}

// Non-temporal operator loads in the multigrid solve: once the operator no
// longer stays in the memory-side cache between iterations.
inline bool stream_loads(const sfem_ctx* ctx, double operator_bytes) {
    return ctx->tune_nt && operator_bytes > kSharedBytes;
}

}  // namespace
}  // namespace sfem
