// pcg.hip -- Jacobi-preconditioned CG on K_ff for gfx950.
//
// Replaces the reference's dense inverse (smearFEM examples/vector3D.jl:318,
// inv(Matrix(K_free)) * C' * (-K q_d)) with an iterative solve that keeps K_ff
// sparse and resident in HBM.  Three precisions share one driver:
//
//   FP64        : operator, vectors and reductions in FP64.
//   MIXED       : FP32 operator values and FP32 CG vectors; the solution
//                 increment is folded into an FP64 solution.
//   FP32_MATRIX : FP32 operator values, FP64 CG vectors.
// In every mode the true residual rhs - K_ff x is recomputed with the FP64
// operator whenever the recurrence residual has dropped by `reliable_delta`
// since the last replacement, or claims convergence ("reliable updates"), and
// the search direction is re-orthogonalised against the new residual.  In the
// low-precision modes this is what carries the solve to FP64 accuracy; in
// FP64 it costs one extra SpMV per 10x drop and keeps the recurrence honest.
// Every mode stops only on that FP64 residual.
//
// Per iteration two kernels run, with no host round trip:
//   operator pass : beta from the last update's sums; p = zcoef z + beta p
//             (formed where a row gathers it, and written once: p is double
//             buffered), q = K_ff p, per-block p.q.  When a replacement is
//             due the pass forms the FP64 residual instead, with z = D^-1 r.
//             On large systems p is a pass of its own (direction_kernel).
//   update pass   : alpha from the pass's p.q; x += alpha p, r -= alpha q,
//             z = D^-1 r, per-block r.z and r.r; after a residual it only
//             takes the residual's sums (beta, the stopping tests;
//             replacements that stop making progress end the solve:
//             "stagnation", the tolerance is below what FP64 can reach).
// The scalars are formed by the kernel that needs them: every block sums the
// previous kernel's per-block partials, in one fixed order, and block 0
// writes the state copy the next kernel reads.  Below ~100k dofs a launch is
// bound by its chain of dependent latencies (about 1 us for each of: the
// state, a last-block arrival, its partials), not by bytes: at 64x16x16 Hex8
// (18.5k nodes, FP64) four kernels with last-block reductions took 41 us an
// iteration.
// The host reads the state every `check_every` steps (an iteration or an FP64
// residual each).
//
// Reductions are deterministic: wave64 butterfly shuffles, a fixed combine
// of a block's wavefronts, per-block partials summed in a fixed order.  The
// grid is a fixed function of the problem size, so results are bitwise
// reproducible run to run.
#include <chrono>
#include <cmath>
#include <string>
#include <vector>

#include "sfem_objects.hpp"
#include "solver_common.hpp"

namespace sfem {

namespace {

// ------------------------------------------------------ state logic ----
// After an update: beta, the replacement triggers and the stopping backstops
// from r.z and r.r.
__device__ __forceinline__ void cg_after_update(CgState& s, double trz, double trr) {
    s.rz_prev = s.rz;
    s.rz = trz;
    s.beta = trz / s.rz_prev;
    s.rr = trr;
    s.iters += 1;
    s.fold_pending = 0;
    s.zcoef = 1.0;
    // replacement when the recurrence converged, dropped by delta, or
    // made no such drop for max(256, iteration of the best true residual)
    const long long since = s.iters - s.last_upd;
    const long long every = s.best_true_it > 256 ? s.best_true_it : 256;
    if (trr <= s.tol2bb || trr < s.delta2 * s.maxrr || since >= every) s.need_update = 1;
    // backstop for a recurrence that stops decreasing: no 2x drop of |r|
    // within max(10000, 4x the iterations it took to reach the best)
    if (trr < 0.25 * s.best_rr) {
        s.best_rr = trr;
        s.best_it = s.iters;
    } else if (s.iters - s.best_it > (4 * s.best_it > 10000 ? 4 * s.best_it : 10000)) {
        s.done = 3;
    }
    if (!std::isfinite(trr)) s.done = 2;
}

// After an FP64 residual: sums are r.r, r.z, r.p and the floor scale.  The
// search direction is made orthogonal to the new residual (p <- p - gamma z,
// gamma = r.p/r.z), folded into zcoef of the next operator pass.
template <bool FOLD>
__device__ __forceinline__ void cg_after_resid(CgState& s, const double (&sums)[4]) {
    const double trr = sums[0], trz = sums[1], trp = sums[2];
    // 16x the attainable |r|^2, (eps * || |rhs| + |K||x| ||)^2
    const double floor_rr = 16.0 * kEps64 * kEps64 * sums[3];
    const double rec = s.rr;  // recurrence |r|^2 that triggered this replacement
    s.rr_true = trr;
    s.floor_rr = floor_rr;
    s.rr = trr;
    s.last_upd = s.iters;
    s.updates += 1;
    s.need_update = 0;
    s.fold_pending = FOLD ? 1 : 0;
    if (trr <= s.tol2bb) {
        s.done = 1;
    } else {
        const double beta = trz / s.rz_prev;
        s.beta = beta;
        s.zcoef = 1.0 - beta * (trp / trz);
        s.rz = trz;
        s.maxrr = trr;
        // Attainable-floor test.  A replacement whose true residual does
        // not beat the best by 10% ends the solve when it is within 4x of
        // the rounding floor eps*|| |rhs| + |K||x| ||, and counts once
        // when the recurrence ran 5x below it (the residual gap of finite
        // precision; twice in a row ends the solve).  Slow progress away
        // from the floor never stops it: the CG residual norm can plateau
        // for thousands of iterations.
        const bool gap = s.iters > 0 && 25.0 * rec < trr;
        if (trr <= 0.81 * s.best_true) {
            s.stall = 0;
            s.best_true_it = s.iters;
        } else if (trr <= floor_rr) {
            s.stall += 2;
        } else if (gap) {
            s.stall += 1;
        }
        if (s.stall >= 2) s.done = 3;
    }
    if (trr < s.best_true) s.best_true = trr;
    if (!std::isfinite(trr)) s.done = 2;
    if (s.capped && !s.done) s.done = 4;
}

// What a pass tells its threads.
struct PassGo {
    double beta, zcoef;  // operator pass: p = zcoef z + beta p
    int done, resid;
};

// What a timed pass was (the host leaves residuals out of the times).
enum PassKind : int { kPassNone = 0, kPassIteration = 1, kPassResidual = 2 };

// Start of an operator pass, by every block: the last update's sums (upd:
// r.z, r.r per block), the state after it, and what this pass has to do.
// kind: where a timed pass records it, else NULL.
template <int NW>
__device__ __forceinline__ PassGo pass_begin(const CgState* __restrict__ in, CgState* __restrict__ out,
                                             const double* __restrict__ upd, int nupd, double* sh, PassGo* shgo,
                                             int* kind) {
    double t[2] = {0.0, 0.0};
    if (in->fresh) sum_parts_all<2, NW>(upd, nupd, t, sh);
    if (threadIdx.x == 0) {
        CgState s = *in;
        if (!s.done) {
            if (s.fresh) cg_after_update(s, t[0], t[1]);
            if (!s.done && !s.need_update && s.iters >= s.max_iter) s.need_update = s.capped = 1;
        }
        s.fresh = 0;
        s.resid = s.need_update;
        if (kind && blockIdx.x == 0) *kind = s.done ? kPassNone : s.resid ? kPassResidual : kPassIteration;
        *shgo = PassGo{s.beta, s.zcoef, s.done, s.resid};
        if (blockIdx.x == 0) *out = s;
    }
    __syncthreads();
    return *shgo;
}

// Per-block partials of an operator pass: p.q (stride 1), or the residual's
// four sums (stride 4).
template <int NW>
__device__ __forceinline__ void put_parts4(double rr, double rz, double rp, double ff, double* __restrict__ parts,
                                           double* sh) {
    const double b0 = block_sum_waves<NW>(rr, sh), b1 = block_sum_waves<NW>(rz, sh);
    const double b2 = block_sum_waves<NW>(rp, sh), b3 = block_sum_waves<NW>(ff, sh);
    if (threadIdx.x == 0) {
        parts[4 * (int64_t)blockIdx.x] = b0;
        parts[4 * (int64_t)blockIdx.x + 1] = b1;
        parts[4 * (int64_t)blockIdx.x + 2] = b2;
        parts[4 * (int64_t)blockIdx.x + 3] = b3;
    }
}

// ---------------------------------------------------- operator pass ----
// Vectors of a pass.  Where p is formed in the gathers (FLY), p and z lie side
// by side, a record of BS values of p then BS of z per block row: a gathered
// row is one record, in 16-byte loads (a mesh in no particular numbering
// gathers a cache line per row and vector).  There are two arrays of records:
// a pass reads the one (p, z) and writes the other's p, and the update that
// follows writes its z.  Else p and z are plain vectors, updated in place.
template <typename T>
struct PassVecs {
    const T* p;
    const T* z;
    T* pnew;
    T* znew;
    T* q;
    T* r;
    const double* x64;
    const T* xs;  // FP32 solution increment (FOLD)
    const double* rhs;
    const T* dinv;
    const T* binv;  // node-block Jacobi: planar inverse blocks, stride nrows
    int* kind;      // a timed pass records what it was here, else NULL
};

// Elements between block rows of p and z.
template <int BS, bool FLY>
constexpr int kRowStride = FLY ? 2 * BS : BS;

template <int BS, typename T>
struct alignas(2 * BS * sizeof(T) % 16 == 0 ? 16 : 8) PzRecord {
    T p[BS], z[BS];
};

// p = zcoef z + beta p in place, and the pass's state: the first half of an
// operator pass on a large system (FLY false below).  There a row's second
// gathered vector costs more than this stream (256x64x64 Hex8, FP64 Jacobi:
// 508 us an iteration with p formed in the gathers, 478 us so).
template <typename T>
__global__ __launch_bounds__(kThreads) void direction_kernel(T* __restrict__ p, const T* __restrict__ z, int64_t n,
                                                             int64_t per_block, const CgState* in, CgState* out,
                                                             const double* __restrict__ upd, int nupd, int* kind) {
    constexpr int NW = kThreads / 64;
    __shared__ double sh[NW];
    __shared__ PassGo shgo;
    const PassGo go = pass_begin<NW>(in, out, upd, nupd, sh, &shgo, kind);
    if (go.done || go.resid) return;
    const T beta = (T)go.beta, zc = (T)go.zcoef;
    const int64_t i0 = (int64_t)blockIdx.x * per_block;
    const int64_t i1 = min(n, i0 + per_block);
#pragma unroll 4  // four strides of loads in flight; the same order of operations
    for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) p[i] = fmaT<T>(beta, p[i], zc * z[i]);
}

// Scalar CSR, G lanes per row.
template <int G, typename TV, typename T, bool FLY, bool FOLD>
__global__ __launch_bounds__(kThreads) void csr_pass_kernel(const int32_t* __restrict__ rowptr,
                                                            const int32_t* __restrict__ col,
                                                            const TV* __restrict__ val,
                                                            const double* __restrict__ val64, int64_t nrows,
                                                            int64_t rows_per_block, PassVecs<T> v, const CgState* in,
                                                            CgState* out, const double* __restrict__ upd, int nupd,
                                                            double* __restrict__ parts) {
    constexpr int NW = kThreads / 64;
    __shared__ double sh[NW];
    __shared__ PassGo shgo;
    PassGo go;
    if constexpr (FLY) go = pass_begin<NW>(in, out, upd, nupd, sh, &shgo, v.kind);
    else go = PassGo{0.0, 0.0, in->done, in->resid};  // direction_kernel has begun the pass
    if (go.done) return;
    const int64_t r0 = logical_block() * rows_per_block;
    const int64_t r1 = min(nrows, r0 + rows_per_block);
    const int g = threadIdx.x / G, lane = threadIdx.x % G;
    if (!go.resid) {
        const T beta = (T)go.beta, zc = (T)go.zcoef;
        const T* __restrict__ p = v.p;
        auto gx = [=](int64_t c) {
            if constexpr (FLY) {
                const PzRecord<1, T> w = ((const PzRecord<1, T>*)p)[c];
                return fmaT<T>(beta, w.p[0], zc * w.z[0]);
            } else {
                return p[c];
            }
        };
        double dot = 0.0;
        for (int64_t row = r0 + g; row < r1; row += kThreads / G) {
            const T s = csr_row<G, TV, T>(rowptr, col, val, row, lane, gx);
            if (lane == 0) {
                const T pr = gx(row);
                if (FLY) v.pnew[row * 2] = pr;
                v.q[row] = s;
                dot += (double)pr * (double)s;
            }
        }
        dot = block_sum_waves<NW>(dot, sh);
        if (threadIdx.x == 0) parts[blockIdx.x] = dot;
        return;
    }
    double rr = 0.0, rz = 0.0, rp = 0.0, ff = 0.0;
    const double* __restrict__ x64 = v.x64;
    const T* __restrict__ xs = v.xs;
    auto gx = [=](int64_t c) { return FOLD ? x64[c] + (double)xs[c] : x64[c]; };
    for (int64_t row = r0 + g; row < r1; row += kThreads / G) {
        double a;
        const double s = csr_row_abs<G>(rowptr, col, val64, row, lane, gx, &a);
        if (lane == 0) {
            const double res = v.rhs[row] - s;
            const double sc = fabs(v.rhs[row]) + a;
            ff += sc * sc;
            const T rt = (T)res;
            const T zt = v.dinv[row] * rt;
            constexpr int RS = kRowStride<1, FLY>;
            const T pr = v.p[row * RS];
            v.r[row] = rt;
            v.znew[row * RS] = zt;
            if (FLY) v.pnew[row * RS] = pr;
            rr += res * res;
            rz += (double)rt * (double)zt;
            rp += (double)rt * (double)pr;
        }
    }
    put_parts4<NW>(rr, rz, rp, ff, parts, sh);
}

// Node-block sliced rows.  SPLIT wavefronts share a slice (64 block rows),
// each taking every SPLIT-th block column: 1 (4 or more slices per block), or
// 4, the whole block (slices_per_block is 1).  BPC: z = B^-1 r with the
// node's inverse diagonal block instead of the point Jacobi dinv.
// With a shared slice p is formed in the gathers, and the slice's column ids
// and first values are loaded before the pass's scalars are known, so the
// two chains of loads overlap (64x16x16 Hex8, FP64 Jacobi: 17.9 -> 15.8 us
// an iteration; 41 us with four kernels per iteration and a wavefront per
// slice, 0.92 TB/s of operator then, 2.4 TB/s now).
template <int BS, typename TV, typename T, bool NT, int SPLIT, bool FOLD, bool BPC>
__global__ __launch_bounds__(kThreads) void sell_pass_kernel(
    const int64_t* __restrict__ sl_ptr, const int32_t* __restrict__ sl_w, const int32_t* __restrict__ scol,
    Vals<TV> sval, const double* __restrict__ sval64, int64_t nslices, int64_t nrows, int64_t slices_per_block,
    PassVecs<T> v, const CgState* in, CgState* out, const double* __restrict__ upd, int nupd,
    double* __restrict__ parts) {
    constexpr int NW = kThreads / 64, B2 = BS * BS;
    static_assert(SPLIT == 1 || SPLIT == NW, "a slice belongs to a wavefront or to the block");
    constexpr bool FLY = SPLIT > 1;
    __shared__ double sh[NW];
    __shared__ PassGo shgo;
    __shared__ double buf[SPLIT > 1 ? NW : 1][2 * BS][64];
    const int64_t s0 = logical_block() * slices_per_block;
    const int64_t s1 = min(nslices, s0 + slices_per_block);
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int part = wv % SPLIT;
    if constexpr (FLY) {
        const int64_t sl = s0;
        const bool live = sl < s1;
        SharedSlice<BS, TV, NT> row_cols(scol, sval);
        if (live) row_cols.load(sl_ptr, sl_w, sl);
        const PassGo go = pass_begin<NW>(in, out, upd, nupd, sh, &shgo, v.kind);
        if (go.done) return;
        if (!go.resid) {
            const T beta = (T)go.beta, zc = (T)go.zcoef;
            const PzRecord<BS, T>* __restrict__ pz = (const PzRecord<BS, T>*)v.p;
            auto gx = [=](int64_t c, T(&x)[BS]) {
                const PzRecord<BS, T> w = pz[c];
#pragma unroll
                for (int i = 0; i < BS; ++i) x[i] = fmaT<T>(beta, w.p[i], zc * w.z[i]);
            };
            T acc[BS] = {};
            row_cols.apply(gx, acc);
            sell_combine<BS, SPLIT>(acc, reinterpret_cast<T(*)[BS][64]>(&buf[0][0][0]));
            double dot = 0.0;
            const int64_t row = sl * 64 + lane;
            if (part == 0 && live && row < nrows) {
                T pr[BS];
                gx(row, pr);
#pragma unroll
                for (int j = 0; j < BS; ++j) {
                    v.pnew[row * 2 * BS + j] = pr[j];
                    v.q[row * BS + j] = acc[j];
                    dot += (double)pr[j] * (double)acc[j];
                }
            }
            dot = block_sum_waves<NW>(dot, sh);
            if (threadIdx.x == 0) parts[blockIdx.x] = dot;
            return;
        }
    } else {
        if (in->done) return;  // direction_kernel has begun the pass
        if (!in->resid) {
            const T* __restrict__ p = v.p;
            auto gx = [=](int64_t c) { return p[c]; };
            double dot = 0.0;
            for (int64_t sl = s0 + wv; sl < s1; sl += NW) {
                T acc[BS];
                sell_row<BS, TV, T, NT>(sl_ptr, sl_w, scol, sval, sl, lane, gx, acc);
                const int64_t row = sl * 64 + lane;
                if (row < nrows) {
                    T pr[BS];  // loaded before the stores, which may alias for all the compiler knows
#pragma unroll
                    for (int j = 0; j < BS; ++j) pr[j] = p[row * BS + j];
#pragma unroll
                    for (int j = 0; j < BS; ++j) {
                        v.q[row * BS + j] = acc[j];
                        dot += (double)pr[j] * (double)acc[j];
                    }
                }
            }
            dot = block_sum_waves<NW>(dot, sh);
            if (threadIdx.x == 0) parts[blockIdx.x] = dot;
            return;
        }
    }
    double rr = 0.0, rz = 0.0, rp = 0.0, ff = 0.0;
    const double* __restrict__ x64 = v.x64;
    const T* __restrict__ xs = v.xs;
    auto gx = [=](int64_t c, double(&x)[BS]) {
#pragma unroll
        for (int i = 0; i < BS; ++i) x[i] = FOLD ? x64[c * BS + i] + (double)xs[c * BS + i] : x64[c * BS + i];
    };
    auto slice = [&](int64_t sl, bool live) {
        double acc[2 * BS] = {};
        if (live) {
            double o[BS], a[BS];
            sell_row_abs_part<BS, SPLIT>(sl_ptr, sl_w, scol, sval64, sl, lane, part, gx, o, a);
#pragma unroll
            for (int j = 0; j < BS; ++j) {
                acc[j] = o[j];
                acc[BS + j] = a[j];
            }
        }
        sell_combine<2 * BS, SPLIT>(acc, buf);
        const int64_t row = sl * 64 + lane;
        if (part == 0 && live && row < nrows) {
            T rt[BS];
#pragma unroll
            for (int j = 0; j < BS; ++j) {
                const int64_t d = row * BS + j;
                const double res = v.rhs[d] - acc[j];
                const double sc = fabs(v.rhs[d]) + acc[BS + j];
                ff += sc * sc;
                rt[j] = (T)res;
                const int64_t e = row * kRowStride<BS, FLY> + j;
                const T pr = v.p[e];
                v.r[d] = rt[j];
                if (FLY) v.pnew[e] = pr;
                rr += res * res;
                rp += (double)rt[j] * (double)pr;
            }
#pragma unroll
            for (int j = 0; j < BS; ++j) {
                const int64_t d = row * BS + j;
                T zt;
                if constexpr (BPC) {
                    zt = 0;
#pragma unroll
                    for (int i = 0; i < BS; ++i) zt = fmaT<T>(v.binv[(j * BS + i) * nrows + row], rt[i], zt);
                } else {
                    zt = v.dinv[d] * rt[j];
                }
                v.znew[row * kRowStride<BS, FLY> + j] = zt;
                rz += (double)rt[j] * (double)zt;
            }
        }
    };
    if constexpr (SPLIT == 1) {
        for (int64_t sl = s0 + wv; sl < s1; sl += NW) slice(sl, true);
    } else {
        slice(s0, s0 < s1);
    }
    put_parts4<NW>(rr, rz, rp, ff, parts, sh);
}

// ------------------------------------------------------ update pass ----
// Start of an update pass: false when there is nothing to update (the solve
// has stopped, or the operator pass was a residual, whose sums block 0
// takes).  np: blocks of the operator pass.
template <bool FOLD>
__device__ __forceinline__ bool update_begin(const CgState* __restrict__ in, CgState* __restrict__ out,
                                             const double* __restrict__ parts, int np, double* sh, double* shalpha,
                                             double& alpha, bool& fold) {
    constexpr int NW = kThreads / 64;
    if (in->done || in->resid) {
        if (blockIdx.x != 0) return false;
        double t[4] = {0.0, 0.0, 0.0, 0.0};
        if (!in->done) sum_parts_all<4, NW>(parts, np, t, sh);
        if (threadIdx.x == 0) {
            CgState s = *in;
            if (!s.done) cg_after_resid<FOLD>(s, t);
            *out = s;
        }
        return false;
    }
    double pq[1];
    sum_parts_all<1, NW>(parts, np, pq, sh);
    if (threadIdx.x == 0) {
        const double a = in->rz / pq[0];
        const bool ok = pq[0] > 0.0 && std::isfinite(a);
        *shalpha = ok ? a : NAN;
        if (blockIdx.x == 0) {
            CgState s = *in;
            s.alpha = a;
            if (!ok) s.done = 2;  // breakdown
            s.fresh = ok ? 1 : 0;
            *out = s;
        }
    }
    __syncthreads();
    alpha = *shalpha;
    fold = FOLD && in->fold_pending;
    return alpha == alpha;
}

// x += alpha p, r -= alpha q, z = D^-1 r, partial r.z and r.r.  With FOLD
// (FP32 solution increment xs) a pending fold moves xs into x64 first.
// BS: values of p (and of z) per record (FLY), 0 for plain vectors.
template <int BS, typename T, bool FOLD>
__global__ __launch_bounds__(kThreads) void cg_update_kernel(T* __restrict__ x, double* __restrict__ x64,
                                                             T* __restrict__ r, T* __restrict__ z,
                                                             const T* __restrict__ p, const T* __restrict__ q,
                                                             const T* __restrict__ dinv, int64_t n,
                                                             int64_t per_block, const CgState* in, CgState* out,
                                                             const double* __restrict__ parts, int np,
                                                             double* __restrict__ upd) {
    constexpr int NW = kThreads / 64;
    __shared__ double sh[NW], shalpha;
    const int64_t i0 = (int64_t)blockIdx.x * per_block;
    const int64_t i1 = min(n, i0 + per_block);
    // the first stride's operands are loaded before alpha is known
    const int64_t f0 = i0 + threadIdx.x;
    const bool first = f0 < i1;
    T fx = 0, fp = 0, fq = 0, fr = 0, fd = 0;
    auto pz = [](int64_t i) {
        if constexpr (BS == 0) return i;
        else return (int64_t)((uint32_t)i + (uint32_t)i / (BS ? BS : 1) * BS);  // (i / BS) 2 BS + i % BS
    };
    if (first) fx = x[f0], fp = p[pz(f0)], fq = q[f0], fr = r[f0], fd = dinv[f0];
    double alpha;
    bool fold;
    if (!update_begin<FOLD>(in, out, parts, np, sh, &shalpha, alpha, fold)) return;
    const T a = (T)alpha;
    double rz = 0.0, rr = 0.0;
    auto step = [&](int64_t i, T xi, T pi, T qi, T ri0, T di) {
        if (fold) {
            x64[i] += (double)xi;
            xi = 0;
        }
        const T ri = fmaT<T>(-a, qi, ri0);
        const T zi = di * ri;
        x[i] = fmaT<T>(a, pi, xi);
        r[i] = ri;
        z[pz(i)] = zi;
        rz += (double)ri * (double)zi;
        rr += (double)ri * (double)ri;
    };
    if (first) step(f0, fx, fp, fq, fr, fd);
#pragma unroll 4  // four strides of loads in flight; the same order of operations
    for (int64_t i = f0 + kThreads; i < i1; i += kThreads) step(i, x[i], p[pz(i)], q[i], r[i], dinv[i]);
    const double b0 = block_sum_waves<NW>(rz, sh);
    const double b1 = block_sum_waves<NW>(rr, sh);
    if (threadIdx.x == 0) {
        upd[2 * (int64_t)blockIdx.x] = b0;
        upd[2 * (int64_t)blockIdx.x + 1] = b1;
    }
}

// Node-block Jacobi form: one thread per node; z = B^-1 r with B^-1 the
// node's inverse diagonal block (planar: binv[(j*BS+i)*nnodes + n]).
template <int BS, bool FLY, typename T, bool FOLD>
__global__ __launch_bounds__(kThreads) void cg_update_block_kernel(T* __restrict__ x, double* __restrict__ x64,
                                                                   T* __restrict__ r, T* __restrict__ z,
                                                                   const T* __restrict__ p, const T* __restrict__ q,
                                                                   const T* __restrict__ binv, int64_t nnodes,
                                                                   int64_t per_block, const CgState* in, CgState* out,
                                                                   const double* __restrict__ parts, int np,
                                                                   double* __restrict__ upd) {
    constexpr int NW = kThreads / 64;
    __shared__ double sh[NW], shalpha;
    const int64_t n0 = (int64_t)blockIdx.x * per_block;
    const int64_t n1 = min(nnodes, n0 + per_block);
    struct In {
        T x[BS], p[BS], q[BS], r[BS], b[BS * BS];
    };
    auto load = [&](int64_t n, In& o) {
#pragma unroll
        for (int j = 0; j < BS; ++j) {
            const int64_t i = n * BS + j;
            o.x[j] = x[i], o.p[j] = p[n * kRowStride<BS, FLY> + j], o.q[j] = q[i], o.r[j] = r[i];
        }
#pragma unroll
        for (int m = 0; m < BS * BS; ++m) o.b[m] = binv[m * nnodes + n];
    };
    // the first node's operands are loaded before alpha is known
    const int64_t f0 = n0 + threadIdx.x;
    const bool first = f0 < n1;
    In f{};
    if (first) load(f0, f);
    double alpha;
    bool fold;
    if (!update_begin<FOLD>(in, out, parts, np, sh, &shalpha, alpha, fold)) return;
    const T a = (T)alpha;
    double rz = 0.0, rr = 0.0;
    auto step = [&](int64_t n, const In& o) {
        T rv[BS];
#pragma unroll
        for (int j = 0; j < BS; ++j) {
            const int64_t i = n * BS + j;
            T xi = o.x[j];
            if (fold) {
                x64[i] += (double)xi;
                xi = 0;
            }
            x[i] = fmaT<T>(a, o.p[j], xi);
            rv[j] = fmaT<T>(-a, o.q[j], o.r[j]);
            r[i] = rv[j];
            rr += (double)rv[j] * (double)rv[j];
        }
#pragma unroll
        for (int j = 0; j < BS; ++j) {
            T zj = 0;
#pragma unroll
            for (int i = 0; i < BS; ++i) zj = fmaT<T>(o.b[j * BS + i], rv[i], zj);
            z[n * kRowStride<BS, FLY> + j] = zj;
            rz += (double)rv[j] * (double)zj;
        }
    };
    if (first) step(f0, f);
    for (int64_t n = f0 + kThreads; n < n1; n += kThreads) {
        In o;
        load(n, o);
        step(n, o);
    }
    const double b0 = block_sum_waves<NW>(rz, sh);
    const double b1 = block_sum_waves<NW>(rr, sh);
    if (threadIdx.x == 0) {
        upd[2 * (int64_t)blockIdx.x] = b0;
        upd[2 * (int64_t)blockIdx.x + 1] = b1;
    }
}

// x64 += xs, xs = 0: the FP32 increment folded at the end of a solve.
__global__ __launch_bounds__(kThreads) void fold_kernel(double* __restrict__ x64, float* __restrict__ xs, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        x64[i] += (double)xs[i];
        xs[i] = 0.0f;
    }
}

// bb = rhs.rhs (FP64), once per solve
__global__ __launch_bounds__(kThreads) void norm2_kernel(const double* __restrict__ v, int64_t n, int64_t per_block,
                                                         CgStates* sts, double* __restrict__ partials, double rtol,
                                                         double delta) {
    __shared__ double sh[8];
    CgState* st = &sts->s[0];
    const int64_t i0 = (int64_t)blockIdx.x * per_block;
    const int64_t i1 = min(n, i0 + per_block);
    double s = 0.0;
#pragma unroll 4  // four strides of loads in flight; the same order of operations
    for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) s += v[i] * v[i];
    const double b = block_sum_256(s, sh);
    if (threadIdx.x == 0) {
        st_coherent(partials + 3 * blockIdx.x, b);
        st_coherent(partials + 3 * blockIdx.x + 1, 0.0);
        st_coherent(partials + 3 * blockIdx.x + 2, 0.0);
    }
    if (last_block_arrive(&sts->arrive)) {
        double bb, u1, u2;
        sum_partials3(partials, gridDim.x, &bb, &u1, &u2, sh);
        if (threadIdx.x == 0) {
            st->bb = bb;
            st->tol2bb = rtol * rtol * bb;
            st->delta2 = delta * delta;
            st->maxrr = bb;
        }
    }
}

// --------------------------------------------------- plain y = A x -----
template <int G, typename TV, typename T>
__global__ __launch_bounds__(kThreads) void csr_spmv_kernel(const int32_t* __restrict__ rowptr,
                                                            const int32_t* __restrict__ col,
                                                            const TV* __restrict__ val, int64_t nrows,
                                                            int64_t rows_per_block, const T* __restrict__ x,
                                                            T* __restrict__ y) {
    const int64_t r0 = logical_block() * rows_per_block;
    const int64_t r1 = min(nrows, r0 + rows_per_block);
    const int g = threadIdx.x / G, lane = threadIdx.x % G;
    auto gx = [=](int64_t c) { return x[c]; };
    for (int64_t row = r0 + g; row < r1; row += kThreads / G) {
        const T s = csr_row<G, TV, T>(rowptr, col, val, row, lane, gx);
        if (lane == 0) y[row] = s;
    }
}

template <int BS, typename TV, typename T, bool NT>
__global__ __launch_bounds__(kThreads) void sell_spmv_kernel(const int64_t* __restrict__ sl_ptr,
                                                             const int32_t* __restrict__ sl_w,
                                                             const int32_t* __restrict__ scol, Vals<TV> sval,
                                                             int64_t nslices,
                                                             int64_t nrows, int64_t slices_per_block,
                                                             const T* __restrict__ x, T* __restrict__ y) {
    const int64_t s0 = logical_block() * slices_per_block;
    const int64_t s1 = min(nslices, s0 + slices_per_block);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    auto gx = [=](int64_t c) { return x[c]; };
    for (int64_t sl = s0 + w; sl < s1; sl += kThreads / 64) {
        T out[BS];
        sell_row<BS, TV, T, NT>(sl_ptr, sl_w, scol, sval, sl, lane, gx, out);
        const int64_t row = sl * 64 + lane;
        if (row < nrows)
#pragma unroll
            for (int j = 0; j < BS; ++j) y[row * BS + j] = out[j];
    }
}

__global__ void f64_to_f32_kernel(const double* __restrict__ a, float* __restrict__ b, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        b[i] = (float)a[i];
}

// Streaming copy used as the measured HBM ceiling: UNROLL 16-byte loads in
// flight per thread before the stores, optionally non-temporal.
typedef float v4f __attribute__((ext_vector_type(4)));

template <int UNROLL, bool NT>
__global__ __launch_bounds__(kThreads) void copy_kernel(const v4f* __restrict__ a, v4f* __restrict__ b, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * kThreads * UNROLL;
    for (int64_t base = (int64_t)blockIdx.x * kThreads * UNROLL + threadIdx.x; base < n; base += stride) {
        v4f v[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int64_t i = base + (int64_t)u * kThreads;
            if (i < n) v[u] = ld_stream<NT>(a + i);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int64_t i = base + (int64_t)u * kThreads;
            if (i < n) {
                if constexpr (NT) __builtin_nontemporal_store(v[u], b + i);
                else b[i] = v[u];
            }
        }
    }
}

// --------------------------------------------------------- host side ---
// Slices up to which a block's four wavefronts share a slice and form p in the
// gathers; above, a wavefront takes a slice and direction_kernel forms p.  A
// small system else has fewer wavefronts than the device holds, each with up
// to 27 block columns of loads one after the other; on a larger one the second
// gathered vector costs more, most of all where the nodes are numbered in no
// particular order.  Node-block Jacobi, us an iteration, one wavefront / four:
//   grid numbering  FP64 276 slices 28.8 / 19.1, 625 30.7 / 26.2, 1,225 49.6 /
//     42.2, 1,541 51.6 / 51.3, 3,038 99.6 / 107.7; FP32 values (fp32_matrix)
//     1,225 36.1 / 33.8, 1,541 38.4 / 40.0, 4,802 98.5 / 117.5
//   shuffled  FP64 1,225 61.6 / 56.9, 1,369 62.2 / 66.2, 1,712 75.6 / 83.2;
//     split 1,225 59.0 / 51.4, 1,541 60.1 / 68.3; fp32_matrix 1,225 49.3 / 49.3,
//     1,369 48.8 / 56.3, 4,802 155.6 / 224.3; mixed 1,369 44.1 / 43.7, 1,712
//     46.7 / 52.1, 4,802 128.3 / 174.4
//   2D, shuffled  FP64 1,177 26.4 / 25.2, 1,449 27.7 / 28.2; split 1,177 24.4 /
//     24.8, 1,355 25.9 / 28.8
constexpr int64_t kSharedSlices = 1280;

// Operator bytes from which its loads are non-temporal (a wavefront per slice):
// where it no longer stays in the 256 MB memory-side cache between iterations.
// us an iteration without / with: 211 MB (split) 60.7 / 67.2, 259 MB (mixed)
// 64.8 / 66.7, 276 MB (FP64) 77.7 / 79.3, 305 MB (split) 78.6 / 76.3, 332 MB
// (mixed) 91.8 / 84.2, 376 MB (split) 104.8 / 94.6, 399 MB (FP64) 99.6 / 91.7.
constexpr double kStreamBytes = 290e6;

// Scalar CSR: p formed in the gathers up to this many dofs.  us an iteration
// with p in the gathers / by direction_kernel, FP64 Jacobi: 3D, 1,944 dofs 12.1
// / 15.1, 20,808 16.2 / 18.7, 60,000 29.2 / 26.9, 90,000 36.8 / 33.1, 322,752
// 128 / 100; 2D, 7,320 dofs 13.3 / 15.0, 45,300 21.5 / 19.0, 97,240 25.8 /
// 21.7; mixed precision turns at the same sizes.
constexpr int64_t kFlyDofs = 30000;
constexpr int kCsrLanes = 16;  // lanes per CSR row (rows of K_ff hold up to 81 entries)

struct Launch {
    unsigned grid;
    int64_t per_block;  // rows / slices / elements per block
};

// grid: a multiple of 8 (XCD mapping), at most `cap` blocks, each block a
// contiguous range that is a multiple of `quantum` items
Launch plan(int64_t items, int quantum, unsigned cap) {
    int64_t need = (items + quantum - 1) / quantum;
    int64_t grid = std::min<int64_t>(need, cap);
    grid = std::max<int64_t>(8, (grid + 7) / 8 * 8);
    int64_t per = (items + grid - 1) / grid;
    per = (per + quantum - 1) / quantum * quantum;
    if (per == 0) per = quantum;
    return {(unsigned)grid, per};
}

// Sliced-operator launches: `wave_slices` > 0 gives every wavefront that
// many slices (grid = slices / (4 * wave_slices)); 0 spreads them over the cap.
Launch plan_sell(int64_t nslices, unsigned cap, int wave_slices) {
    if (wave_slices <= 0) return plan(nslices, kThreads / 64, cap);
    const int64_t per = (int64_t)wave_slices * (kThreads / 64);
    int64_t grid = (nslices + per - 1) / per;
    grid = std::max<int64_t>(8, (grid + 7) / 8 * 8);
    return {(unsigned)grid, per};
}

struct Ops {
    sfem_ctx* ctx;
    sfem_system* S;
    int fmt;  // SFEM_FMT_CSR / SFEM_FMT_BSR
    unsigned cap;
    Launch csr, sell, vec;
    int split;      // wavefronts per slice
    bool fly;       // p formed in the operator pass (double buffered)
    bool nt;        // non-temporal matrix loads in the sliced SpMV
    bool block_pc;  // node-block Jacobi preconditioner
    Launch node;    // one thread per node (block update)
    // vectors of the solve: the free dofs, or the padded block rows when
    // the node-block format carries partially fixed nodes
    double* x64;
    const double* rhs;
    int64_t n;
    unsigned pass_grid() const { return fmt == SFEM_FMT_BSR ? sell.grid : csr.grid; }
    unsigned update_grid() const { return block_pc ? node.grid : vec.grid; }
};

template <typename TV>
const TV* csr_vals(const sfem_system* S);
template <>
const double* csr_vals<double>(const sfem_system* S) { return S->val64.get(); }
template <>
const float* csr_vals<float>(const sfem_system* S) { return S->val32.get(); }
template <typename TV>
Vals<TV> sell_vals(const sfem_system* S);
template <>
Vals<double> sell_vals<double>(const sfem_system* S) { return {S->sval64.get()}; }
template <>
Vals<float> sell_vals<float>(const sfem_system* S) { return {S->sval32.get()}; }
template <>
Vals<SplitVal> sell_vals<SplitVal>(const sfem_system* S) { return {S->sval32.get(), S->sval16.get()}; }

// bytes per stored operator value
template <typename TV>
constexpr double val_bytes() { return std::is_same<TV, SplitVal>::value ? 6.0 : (double)sizeof(TV); }

// One operator pass: state st->s[0] -> st->s[1].  begin: an event recorded in
// front of the operator's own kernel, or NULL.
template <typename TV, typename T>
void launch_pass(const Ops& o, const PassVecs<T>& v, CgStates* st, const double* upd, double* parts,
                 hipEvent_t begin) {
    constexpr bool FOLD = std::is_same<T, float>::value;
    sfem_system* S = o.S;
    hipStream_t s = o.ctx->stream;
    const int nupd = (int)o.update_grid();
    const CgState* in = &st->s[0];
    CgState* out = &st->s[1];
    if (!o.fly) {
        hipLaunchKernelGGL(direction_kernel<T>, dim3(o.vec.grid), dim3(kThreads), 0, s, v.pnew, (const T*)v.z, o.n,
                           o.vec.per_block, in, out, upd, nupd, v.kind);
        SFEM_LAUNCH_CHECK();
        in = out;
    }
    if (begin) SFEM_HIP(hipEventRecord(begin, s));
    if (o.fmt == SFEM_FMT_BSR) {
        auto run = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(o.sell.grid), dim3(kThreads), 0, s, S->sl_ptr.get(), S->sl_w.get(),
                               S->scol.get(), sell_vals<TV>(S), S->sval64.get(), S->nslices, S->nfb, o.sell.per_block,
                               v, in, out, upd, nupd, parts);
        };
        auto pick = [&](auto bs, auto bpc) {
            constexpr int BS = decltype(bs)::value;
            constexpr bool BPC = decltype(bpc)::value;
            if (o.split == 4) run(sell_pass_kernel<BS, TV, T, false, 4, FOLD, BPC>);
            else if (o.nt) run(sell_pass_kernel<BS, TV, T, true, 1, FOLD, BPC>);
            else run(sell_pass_kernel<BS, TV, T, false, 1, FOLD, BPC>);
        };
        if (S->bs == 3) {
            if (o.block_pc) pick(std::integral_constant<int, 3>(), std::true_type());
            else pick(std::integral_constant<int, 3>(), std::false_type());
        } else {
            if (o.block_pc) pick(std::integral_constant<int, 2>(), std::true_type());
            else pick(std::integral_constant<int, 2>(), std::false_type());
        }
    } else if constexpr (!std::is_same<TV, SplitVal>::value) {
        auto run = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(o.csr.grid), dim3(kThreads), 0, s, S->rowptr.get(), S->col.get(),
                               csr_vals<TV>(S), S->val64.get(), S->nf, o.csr.per_block, v, in, out, upd, nupd, parts);
        };
        if (o.fly) run(csr_pass_kernel<kCsrLanes, TV, T, true, FOLD>);
        else run(csr_pass_kernel<kCsrLanes, TV, T, false, FOLD>);
    } else {
        fail(SFEM_ERR_UNSUPPORTED, "split precision needs the node-block format");
    }
    SFEM_LAUNCH_CHECK();
}

// One update pass: state st->s[1] -> st->s[0].
template <typename T>
void launch_update(const Ops& o, const PassVecs<T>& v, T* x, double* x64, CgStates* st, const double* parts,
                   double* upd) {
    constexpr bool FOLD = std::is_same<T, float>::value;
    hipStream_t s = o.ctx->stream;
    const CgState* in = &st->s[1];
    CgState* out = &st->s[0];
    const int np = (int)o.pass_grid();
    auto point = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(o.vec.grid), dim3(kThreads), 0, s, x, x64, v.r, v.znew, (const T*)v.pnew,
                           (const T*)v.q, v.dinv, o.n, o.vec.per_block, in, out, parts, np, upd);
    };
    auto block = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(o.node.grid), dim3(kThreads), 0, s, x, x64, v.r, v.znew, (const T*)v.pnew,
                           (const T*)v.q, v.binv, o.S->nfb, o.node.per_block, in, out, parts, np, upd);
    };
    const bool bs3 = o.S->bs == 3;
    if (!o.block_pc) {
        if (!o.fly) point(cg_update_kernel<0, T, FOLD>);
        else if (o.fmt != SFEM_FMT_BSR) point(cg_update_kernel<1, T, FOLD>);
        else if (bs3) point(cg_update_kernel<3, T, FOLD>);
        else point(cg_update_kernel<2, T, FOLD>);
    } else if (o.fly) {
        if (bs3) block(cg_update_block_kernel<3, true, T, FOLD>);
        else block(cg_update_block_kernel<2, true, T, FOLD>);
    } else {
        if (bs3) block(cg_update_block_kernel<3, false, T, FOLD>);
        else block(cg_update_block_kernel<2, false, T, FOLD>);
    }
    SFEM_LAUNCH_CHECK();
}

double spmv_bytes_for(const sfem_system* S, int fmt, double sv, double sx, int nvec) {
    const int64_t nv = (fmt == SFEM_FMT_BSR && S->partial) ? S->nfb * S->bs : S->nf;
    const double vec = (double)nvec * (double)nv * sx;
    if (fmt == SFEM_FMT_BSR)
        return (double)S->nnzb * (S->bs * S->bs * sv + 4.0) + (double)(S->nslices + 1) * 8.0 +
               (double)S->nslices * 4.0 + vec;
    return (double)S->nnz * (sv + 4.0) + (double)(S->nf + 1) * 4.0 + vec;
}

void ensure_val32(sfem_ctx* ctx, sfem_system* S) {
    ensure_csr(ctx, S);
    if (S->val32.size() == (size_t)S->nnz || S->nnz == 0) return;
    S->val32.reset(ctx, (size_t)S->nnz);
    hipLaunchKernelGGL(f64_to_f32_kernel, dim3(2048), dim3(256), 0, ctx->stream, S->val64.get(), S->val32.get(),
                       S->nnz);
    SFEM_LAUNCH_CHECK();
}

int resolve_format(const sfem_system* S, int fmt) {
    if (fmt == SFEM_FMT_BSR && !S->has_block) return SFEM_FMT_CSR;
    if (fmt == SFEM_FMT_AUTO) return S->has_block ? SFEM_FMT_BSR : SFEM_FMT_CSR;
    return fmt;
}

// Device workspace of one solve when the caller provides it (the solve that
// allocates nothing): the CG vectors r and q, the direction and z (pz: two
// arrays of records, or p and z in the first), the FP32 solution increment,
// the per-block partial sums and the state.
struct CgWork {
    void *r, *q, *pz[2], *xs;
    double* partials;
    size_t max_partials;  // doubles
    CgStates* st;
};

// Zeroes n elements of a vector (a kernel, not hipMemsetAsync, so that the
// solve that allocates nothing issues kernels only).
template <typename T>
__global__ __launch_bounds__(kThreads) void zero_kernel(T* __restrict__ v, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
        v[i] = T(0);
}

__global__ __launch_bounds__(64) void cg_state_init_kernel(CgStates* st, long long max_iter) {
    for (int k = (int)threadIdx.x; k < (int)(sizeof(st->arrive.c) / sizeof(st->arrive.c[0])); k += 64)
        st->arrive.c[k] = 0;
    if (threadIdx.x != 0) return;
    CgState init{};
    init.rr = HUGE_VAL;
    init.rz_prev = HUGE_VAL;
    init.zcoef = 1.0;
    init.best_rr = HUGE_VAL;
    init.best_true = HUGE_VAL;
    init.need_update = 1;
    init.max_iter = max_iter;
    st->s[0] = init;
}

template <typename T>
void zero_dev(sfem_ctx* ctx, T* v, int64_t n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(zero_kernel<T>, dim3(std::min<unsigned>(grid_for(n, kThreads), 2048)), dim3(kThreads), 0,
                       ctx->stream, v, n);
    SFEM_LAUNCH_CHECK();
}

// TV: operator value type, T: CG vector type.  FOLD (T == float): the
// solution increment lives in FP32 and is folded into the FP64 solution at
// every residual replacement.  ws: the caller's workspace (no device
// allocation, no events, no host-to-device copies), or NULL.
template <typename TV, typename T>
void run_pcg(sfem_ctx* ctx, sfem_system* S, const sfem_solve_opts* o, sfem_solve_stats* stats, int fmt,
             const CgWork* ws = nullptr) {
    constexpr bool FOLD = std::is_same<T, float>::value;
    const bool padded = fmt == SFEM_FMT_BSR && S->partial;
    const int64_t nf = padded ? S->nfb * S->bs : S->nf;  // length of the solve's vectors
    const bool block_pc = o->preconditioner == SFEM_PC_BLOCK_JACOBI;
    if (block_pc && fmt != SFEM_FMT_BSR)
        fail(SFEM_ERR_UNSUPPORTED, "block-Jacobi preconditioning needs the node-block format");
    if (o->preconditioner != SFEM_PC_JACOBI && !block_pc) fail(SFEM_ERR_ARGUMENT, "solve: unknown preconditioner");
    double* x64 = padded ? S->px.get() : S->x.get();
    Ops ops{ctx, S, fmt, (unsigned)std::max(8, ctx->n_cu * 8), {}, {}, {}, 1, false, false, block_pc, {},
            x64, padded ? S->prhs.get() : S->rhs.get(), nf};
    if (block_pc) ops.node = plan(S->nfb, kThreads, std::max(8, ctx->n_cu * 4));
    ops.csr = plan(S->nf, kThreads / kCsrLanes, ops.cap);
    ops.fly = nf <= kFlyDofs;
    if (fmt == SFEM_FMT_BSR) {
        const double op_bytes = spmv_bytes_for(S, fmt, val_bytes<TV>(), 0, 0);
        const bool share = ctx->tune_split > 0 ? ctx->tune_split >= 4 : S->nslices <= kSharedSlices;
        ops.split = share ? 4 : 1;
        ops.fly = ops.split > 1;
        ops.nt = ctx->tune_nt && op_bytes > kStreamBytes;
        if (ops.split > 1) {  // a block per slice
            ops.sell = {(unsigned)std::max<int64_t>(8, (S->nslices + 7) / 8 * 8), 1};
        } else {
            ops.sell = plan_sell(S->nslices, ops.cap, ctx->tune_wave_slices);
        }
    }
    ops.vec = plan(nf, kThreads, std::max(8, ctx->n_cu * 4));
    // the operator pass's sums (4 per block), then the update's (2 per block;
    // the rhs norm's first: 3 per block)
    const size_t nparts = 4 * (size_t)ops.pass_grid();
    const size_t nupd = std::max(2 * (size_t)ops.update_grid(), 3 * (size_t)ops.vec.grid);

    DevBuf<T> rb, qb, pzb[2], xsb;
    DevBuf<double> partb;
    DevBuf<CgStates> dst;
    T *r, *q, *pz[2], *xsv = nullptr;
    double* parts;
    CgStates* st;
    if (ws) {
        if (nparts + nupd > ws->max_partials) fail(SFEM_ERR_UNSUPPORTED, "solve: workspace too small");
        r = (T*)ws->r, q = (T*)ws->q, pz[0] = (T*)ws->pz[0], pz[1] = (T*)ws->pz[1];
        if (FOLD) xsv = (T*)ws->xs;
        parts = ws->partials;
        st = ws->st;
    } else {
        rb.reset(ctx, nf), qb.reset(ctx, nf), pzb[0].reset(ctx, 2 * nf);
        if (ops.fly) pzb[1].reset(ctx, 2 * nf);
        r = rb.get(), q = qb.get(), pz[0] = pzb[0].get(), pz[1] = pzb[1].get();
        if (FOLD) {
            xsb.reset(ctx, nf);
            xsv = xsb.get();
        }
        partb.reset(ctx, nparts + nupd);
        parts = partb.get();
        dst.reset(ctx, 1);
        st = dst.get();
    }
    // z: BS values after a record's p, or the second half of the first array
    const int64_t zoff = !ops.fly ? nf : fmt == SFEM_FMT_BSR ? S->bs : 1;
    double* upd = parts + nparts;
    const T* dinv = padded ? (FOLD ? (const T*)S->pdinv32.get() : (const T*)S->pdinv64.get())
                           : (FOLD ? (const T*)S->dinv32.get() : (const T*)S->dinv64.get());
    const T* binv = FOLD ? (const T*)S->binv32.get() : (const T*)S->binv64.get();
    T* x = (T*)x64;  // FP64 paths update the FP64 solution directly
    if (FOLD) {
        zero_dev(ctx, xsv, nf);
        x = xsv;
    }
    const T* xs = FOLD ? xsv : nullptr;
    if (o->x0_zero) zero_dev(ctx, S->x.get(), S->nf);
    if (padded) pad_gather(ctx, S, S->x.get(), x64);  // start from the current solution
    zero_dev(ctx, pz[0], 2 * nf);
    hipLaunchKernelGGL(cg_state_init_kernel, dim3(1), dim3(64), 0, ctx->stream, st, (long long)o->max_iter);
    SFEM_LAUNCH_CHECK();

    const bool timed_run = ws == nullptr;  // events are runtime objects: none in the no-allocation solve
    hipEvent_t t0 = nullptr, t1 = nullptr;
    if (timed_run) {
        SFEM_HIP(hipEventCreate(&t0));
        SFEM_HIP(hipEventCreate(&t1));
    }
    const auto w0 = std::chrono::steady_clock::now();
    const bool time_passes = o->time_kernels && timed_run;
    const int check = std::max(1, time_passes ? std::min(o->check_every, 64) : o->check_every);
    std::vector<hipEvent_t> ev;
    DevBuf<int> dkinds;
    std::vector<int> kinds;
    if (time_passes) {
        dkinds.reset(ctx, (size_t)check);
        kinds.resize((size_t)check);
        ev.resize(2 * (size_t)check);
        for (auto& e : ev) SFEM_HIP(hipEventCreate(&e));
    }
    if (timed_run) SFEM_HIP(hipEventRecord(t0, ctx->stream));
    hipLaunchKernelGGL(norm2_kernel, dim3(ops.vec.grid), dim3(kThreads), 0, ctx->stream, ops.rhs, nf,
                       ops.vec.per_block, st, upd, o->rtol, o->reliable_delta);
    SFEM_LAUNCH_CHECK();
    T* const pz1 = ops.fly ? pz[1] : pz[0];
    PassVecs<T> v{pz[0], pz[0] + zoff, pz1, pz1 + zoff, q, r, x64, xs, ops.rhs, dinv, binv, nullptr};

    CgState host{};
    int64_t timed = 0;
    double spmv_ms = 0.0;
    // the first step is the residual of the start; a step is an iteration or
    // a residual replacement, and the device stops at the iteration cap
    for (int64_t chunk = 1; !host.done; chunk = check) {
        for (int64_t k = 0; k < chunk; ++k) {
            if (time_passes) v.kind = dkinds.get() + k;
            launch_pass<TV, T>(ops, v, st, upd, parts, time_passes ? ev[2 * k] : nullptr);
            if (time_passes) SFEM_HIP(hipEventRecord(ev[2 * k + 1], ctx->stream));
            launch_update<T>(ops, v, x, x64, st, parts, upd);
            T *const po = v.pnew, *const zo = v.znew;  // in place: the same arrays
            v.pnew = const_cast<T*>(v.p), v.znew = const_cast<T*>(v.z);
            v.p = po, v.z = zo;
        }
        d2h(ctx, &host, &st->s[0], sizeof(host));
        if (time_passes) {
            // launches after the stop exit at once, and residuals are another operator
            d2h(ctx, kinds.data(), dkinds.get(), sizeof(int) * (size_t)chunk);
            for (int64_t k = 0; k < chunk; ++k) {
                if (kinds[(size_t)k] != kPassIteration) continue;
                float ms = 0;
                SFEM_HIP(hipEventElapsedTime(&ms, ev[2 * k], ev[2 * k + 1]));
                spmv_ms += ms;
                ++timed;
            }
        }
    }
    if (FOLD) {  // x = x64 + xs
        hipLaunchKernelGGL(fold_kernel, dim3(ops.vec.grid), dim3(kThreads), 0, ctx->stream, x64, (float*)xsv, nf);
        SFEM_LAUNCH_CHECK();
    }
    if (padded) pad_scatter(ctx, S, x64, S->x.get());
    float total = 0;
    if (timed_run) {
        SFEM_HIP(hipEventRecord(t1, ctx->stream));
        sync(ctx);
        SFEM_HIP(hipEventElapsedTime(&total, t0, t1));
        for (auto& e : ev) (void)hipEventDestroy(e);
        (void)hipEventDestroy(t0);
        (void)hipEventDestroy(t1);
    } else {
        sync(ctx);
        total = (float)std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - w0).count();
    }

    stats->iterations = host.iters;
    stats->fp64_updates = host.updates;
    stats->spmv_launches = host.iters;
    stats->spmv64_launches = host.updates;
    stats->rel_residual = host.bb > 0 ? std::sqrt(host.rr_true / host.bb) : 0.0;
    stats->solve_ms = total;
    stats->spmv_ms = spmv_ms;
    stats->spmv_timed = timed;
    // the operator pass: matrix once, p read once, q written; where it also
    // forms p, z read and the new p written
    stats->spmv_bytes = spmv_bytes_for(S, fmt, val_bytes<TV>(), sizeof(T), ops.fly ? 4 : 2);
    stats->converged = host.done == 1 ? 1 : 0;
    stats->format = fmt;
    stats->stop_reason = host.done;
    stats->floor_residual = host.bb > 0 ? std::sqrt(host.floor_rr / 16.0 / host.bb) : 0.0;
}

}  // namespace

// ---------------------------------------------- the no-allocation solve --
// Workspace of sfem_system_solve_noalloc: a file-scope device array, one copy
// per GPU, held until the process ends.  Layout: six CG vectors of
// kNoAllocMaxDofs doubles (r, q, and p with z twice; the FP32 vectors are half
// as long, and the increment lies behind r), the per-block partial sums, the
// CG state.  Host code reaches it only through the address
// hipGetSymbolAddress returns for the current device (sfem_ctx::scratch).
namespace {
constexpr size_t kNoAllocVec = sizeof(double) * (size_t)kNoAllocMaxDofs;
constexpr size_t kNoAllocPartials = 4 * 16384;  // doubles: 4 per block of the largest plan
constexpr size_t kNoAllocBytes = 6 * kNoAllocVec + sizeof(double) * kNoAllocPartials + (sizeof(CgStates) + 255) / 256 * 256;
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];
}  // namespace

void* noalloc_scratch_address() {
    void* ptr = nullptr;
    SFEM_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    return ptr;
}

size_t noalloc_scratch_bytes() { return kNoAllocBytes; }

void system_solve_noalloc(sfem_ctx* ctx, sfem_system* S, const sfem_solve_opts* o, sfem_solve_stats* st) {
    *st = sfem_solve_stats{};
    if (!ctx->scratch) fail(SFEM_ERR_STATE, "solve_noalloc: no workspace address for this device");
    if (!(o->rtol >= 0.0) || o->max_iter < 0) fail(SFEM_ERR_ARGUMENT, "solve: bad rtol or max_iter");
    if (o->preconditioner == SFEM_PC_MULTIGRID)
        fail(SFEM_ERR_UNSUPPORTED, "solve_noalloc: point or block Jacobi only (the multigrid V-cycle allocates)");
    const int fmt = resolve_format(S, o->format);
    const int64_t nv = (fmt == SFEM_FMT_BSR && S->partial) ? S->nfb * S->bs : S->nf;
    if (nv > kNoAllocMaxDofs)
        fail(SFEM_ERR_UNSUPPORTED, "solve_noalloc: " + std::to_string(nv) + " solver dofs, at most " +
                                       std::to_string(kNoAllocMaxDofs));
    if (S->nf == 0) {
        st->converged = 1;
        st->stop_reason = 1;
        return;
    }
    // the operator formats are built by the first allocating solve; this one
    // only reads them
    const bool f32 = o->precision == SFEM_PREC_MIXED || o->precision == SFEM_PREC_FP32_MATRIX;
    const bool ready = S->dinv64.size() &&
                       (fmt == SFEM_FMT_BSR ? S->sell_ready
                                            : (S->col.size() == (size_t)S->nnz && (!f32 || S->val32.size())));
    if (!ready)
        fail(SFEM_ERR_STATE, "solve_noalloc: the operator format these options read is not built yet; one "
                             "sfem_system_solve with the same precision and format builds it");
    unsigned char* base = static_cast<unsigned char*>(ctx->scratch);
    unsigned char* end = base + 6 * kNoAllocVec;
    CgWork ws{base, base + kNoAllocVec, {base + 2 * kNoAllocVec, base + 4 * kNoAllocVec}, base + kNoAllocVec / 2,
              reinterpret_cast<double*>(end), kNoAllocPartials,
              reinterpret_cast<CgStates*>(end + sizeof(double) * kNoAllocPartials)};
    sfem_solve_opts oo = *o;
    oo.time_kernels = 0;
    switch (o->precision) {
        case SFEM_PREC_FP64: run_pcg<double, double>(ctx, S, &oo, st, fmt, &ws); break;
        case SFEM_PREC_MIXED: run_pcg<float, float>(ctx, S, &oo, st, fmt, &ws); break;
        case SFEM_PREC_FP32_MATRIX: run_pcg<float, double>(ctx, S, &oo, st, fmt, &ws); break;
        case SFEM_PREC_SPLIT:
            if (fmt != SFEM_FMT_BSR) fail(SFEM_ERR_UNSUPPORTED, "split precision needs the node-block format");
            run_pcg<SplitVal, double>(ctx, S, &oo, st, fmt, &ws);
            break;
        default: fail(SFEM_ERR_ARGUMENT, "solve: unknown precision");
    }
    if (!st->converged) {
        static const char* why[] = {"", "", "breakdown", "stagnation", "iteration cap reached"};
        char buf[200];
        std::snprintf(buf, sizeof buf, "solve: %s after %lld iterations (relative residual %.3e)",
                      why[st->stop_reason], (long long)st->iterations, st->rel_residual);
        fail(SFEM_ERR_NOT_CONVERGED, buf);
    }
}

void system_solve(sfem_ctx* ctx, sfem_system* S, const sfem_solve_opts* o, sfem_solve_stats* st) {
    *st = sfem_solve_stats{};
    if (S->nf == 0) {
        st->converged = 1;
        st->stop_reason = 1;
        return;
    }
    if (!(o->rtol >= 0.0) || o->max_iter < 0) fail(SFEM_ERR_ARGUMENT, "solve: bad rtol or max_iter");
    const int fmt = resolve_format(S, o->format);
    if (fmt == SFEM_FMT_CSR) ensure_csr(ctx, S);
    if (o->preconditioner != SFEM_PC_MULTIGRID) {  // multigrid builds what its levels read
        if (fmt == SFEM_FMT_BSR) ensure_sell(ctx, S);
        ensure_dinv(ctx, S);
    }
    if (o->preconditioner == SFEM_PC_MULTIGRID) {
        if (fmt != SFEM_FMT_BSR) fail(SFEM_ERR_UNSUPPORTED, "multigrid: needs the node-block format");
        mg_solve(ctx, S, o, st);
    } else switch (o->precision) {
        case SFEM_PREC_FP64: run_pcg<double, double>(ctx, S, o, st, fmt); break;
        case SFEM_PREC_MIXED:
            if (fmt == SFEM_FMT_CSR) ensure_val32(ctx, S);
            run_pcg<float, float>(ctx, S, o, st, fmt);
            break;
        case SFEM_PREC_FP32_MATRIX:
            if (fmt == SFEM_FMT_CSR) ensure_val32(ctx, S);
            run_pcg<float, double>(ctx, S, o, st, fmt);
            break;
        case SFEM_PREC_SPLIT:
            if (fmt != SFEM_FMT_BSR) fail(SFEM_ERR_UNSUPPORTED, "split precision needs the node-block format");
            run_pcg<SplitVal, double>(ctx, S, o, st, fmt);
            break;
        default: fail(SFEM_ERR_ARGUMENT, "solve: unknown precision");
    }
    if (!st->converged) {
        static const char* why[] = {"", "", "breakdown", "stagnation", "iteration cap reached"};
        char buf[200];
        std::snprintf(buf, sizeof buf, "solve: %s after %lld iterations (relative residual %.3e)",
                      why[st->stop_reason], (long long)st->iterations, st->rel_residual);
        fail(SFEM_ERR_NOT_CONVERGED, buf);
    }
}

namespace {
template <typename TV, typename T>
double spmv_bench_impl(sfem_ctx* ctx, sfem_system* S, int fmt, int reps, bool nt) {
    const bool padded = fmt == SFEM_FMT_BSR && S->partial;
    const int64_t nf = padded ? S->nfb * S->bs : S->nf;
    const unsigned cap = (unsigned)std::max(8, ctx->n_cu * 8);
    const Launch lc = plan(nf, kThreads / kCsrLanes, cap);
    const Launch ls = S->has_block ? plan_sell(S->nslices, cap, ctx->tune_wave_slices) : Launch{8, 1};
    DevBuf<double> x64(ctx, nf);
    DevBuf<T> x(ctx, nf), y(ctx, nf);
    SFEM_HIP(hipMemcpyAsync(x64.get(), padded ? S->prhs.get() : S->rhs.get(), sizeof(double) * nf,
                            hipMemcpyDeviceToDevice, ctx->stream));
    if (std::is_same<T, float>::value)
        hipLaunchKernelGGL(f64_to_f32_kernel, dim3(1024), dim3(256), 0, ctx->stream, x64.get(), (float*)x.get(), nf);
    else
        SFEM_HIP(hipMemcpyAsync(x.get(), x64.get(), sizeof(double) * nf, hipMemcpyDeviceToDevice, ctx->stream));
    auto launch = [&]() {
        hipStream_t s = ctx->stream;
        if (fmt == SFEM_FMT_BSR) {
            auto go = [&](auto kern) {
                hipLaunchKernelGGL(kern, dim3(ls.grid), dim3(kThreads), 0, s, S->sl_ptr.get(), S->sl_w.get(),
                                   S->scol.get(), sell_vals<TV>(S), S->nslices, S->nfb, ls.per_block, x.get(), y.get());
            };
            if (S->bs == 3) {
                if (nt) go(sell_spmv_kernel<3, TV, T, true>);
                else go(sell_spmv_kernel<3, TV, T, false>);
            } else {
                if (nt) go(sell_spmv_kernel<2, TV, T, true>);
                else go(sell_spmv_kernel<2, TV, T, false>);
            }
        } else if constexpr (!std::is_same<TV, SplitVal>::value) {
            hipLaunchKernelGGL((csr_spmv_kernel<kCsrLanes, TV, T>), dim3(lc.grid), dim3(kThreads), 0, s,
                               S->rowptr.get(), S->col.get(), csr_vals<TV>(S), nf, lc.per_block, x.get(), y.get());
        }
        SFEM_LAUNCH_CHECK();
    };
    launch();  // warm
    hipEvent_t a, b;
    SFEM_HIP(hipEventCreate(&a));
    SFEM_HIP(hipEventCreate(&b));
    SFEM_HIP(hipEventRecord(a, ctx->stream));
    for (int i = 0; i < reps; ++i) launch();
    SFEM_HIP(hipEventRecord(b, ctx->stream));
    sync(ctx);
    float ms = 0;
    SFEM_HIP(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return reps > 0 ? ms / reps : 0.0;
}
}  // namespace

void system_spmv_bench(sfem_ctx* ctx, sfem_system* S, int precision, int format, int reps, double* avg_ms,
                       double* bytes) {
    const int fmt = resolve_format(S, format);
    if (fmt == SFEM_FMT_CSR) ensure_csr(ctx, S);
    if (fmt == SFEM_FMT_BSR) ensure_sell(ctx, S);
    if (precision != SFEM_PREC_FP64 && fmt == SFEM_FMT_CSR) ensure_val32(ctx, S);
    switch (precision) {
        case SFEM_PREC_FP64:
            *avg_ms = spmv_bench_impl<double, double>(ctx, S, fmt, reps, ctx->tune_nt);
            *bytes = spmv_bytes_for(S, fmt, 8, 8, 2);
            break;
        case SFEM_PREC_MIXED:
            *avg_ms = spmv_bench_impl<float, float>(ctx, S, fmt, reps, ctx->tune_nt);
            *bytes = spmv_bytes_for(S, fmt, 4, 4, 2);
            break;
        case SFEM_PREC_FP32_MATRIX:
            *avg_ms = spmv_bench_impl<float, double>(ctx, S, fmt, reps, ctx->tune_nt);
            *bytes = spmv_bytes_for(S, fmt, 4, 8, 2);
            break;
        case SFEM_PREC_SPLIT:
            if (fmt != SFEM_FMT_BSR) fail(SFEM_ERR_UNSUPPORTED, "split precision needs the node-block format");
            *avg_ms = spmv_bench_impl<SplitVal, double>(ctx, S, fmt, reps, ctx->tune_nt);
            *bytes = spmv_bytes_for(S, fmt, 6, 8, 2);
            break;
        default: fail(SFEM_ERR_ARGUMENT, "spmv bench: unknown precision");
    }
}

void stream_copy_bench(sfem_ctx* ctx, int64_t bytes, int reps, double* avg_ms) {
    const int64_t n4 = bytes / 16;
    if (n4 <= 0) fail(SFEM_ERR_ARGUMENT, "copy bench: size too small");
    DevBuf<v4f> a(ctx, n4), b(ctx, n4);
    memset_d(ctx, a.get(), 0, sizeof(v4f) * n4);
    hipEvent_t e0, e1;
    SFEM_HIP(hipEventCreate(&e0));
    SFEM_HIP(hipEventCreate(&e1));
    double best = 1e30;
    // best of a few launch shapes and of plain vs non-temporal access
    auto trial = [&](auto kern, unsigned grid) {
        hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads), 0, ctx->stream, a.get(), b.get(), n4);
        SFEM_LAUNCH_CHECK();
        SFEM_HIP(hipEventRecord(e0, ctx->stream));
        for (int i = 0; i < reps; ++i)
            hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads), 0, ctx->stream, a.get(), b.get(), n4);
        SFEM_LAUNCH_CHECK();
        SFEM_HIP(hipEventRecord(e1, ctx->stream));
        sync(ctx);
        float ms = 0;
        SFEM_HIP(hipEventElapsedTime(&ms, e0, e1));
        best = std::min(best, (double)ms / std::max(1, reps));
    };
    for (unsigned mult : {4u, 8u, 16u}) {
        const unsigned grid = (unsigned)std::max(8, ctx->n_cu * (int)mult);
        trial(copy_kernel<1, false>, grid);
        trial(copy_kernel<4, false>, grid);
        trial(copy_kernel<4, true>, grid);
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *avg_ms = best;
}

}  // namespace sfem
