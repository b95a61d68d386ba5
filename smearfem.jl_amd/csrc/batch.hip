// batch.hip -- many independent meshes assembled together and solved by
// persistent (cooperative) kernel launches; the same engine runs the request
// table of the serving loop (serve.hip).
//
// A batch is a block-diagonal system: the meshes are concatenated (node ids
// offset per problem) and assembled by the single-mesh sort-by-key pipeline
// (duplicates never cross problems, so each problem's K is bitwise the one it
// gets alone), then Dirichlet-eliminated into one node-block sliced operator
// in which every problem starts on a fresh 64-row slice ("padded layout":
// padding rows have zero matrix rows, zero rhs and unit diagonal, so they
// stay exactly zero through the iteration).
//
// The solver keeps one CG state per problem.  Every per-problem dot product is
// formed from that problem's slice partials in a fixed order, whichever blocks
// made them.  A problem's arithmetic therefore depends only on its own data:
// it is bitwise the same alone, in this batch, in any other batch, for any
// grid size, for any item_slices and for any split of its iterations over
// launches.
//
// Reference: the per-problem maths is smearFEM's assemble_system
// (src/fem.jl:135-256) and the example's elimination and solve
// (examples/vector3D.jl:314-322); batching has no reference counterpart.

#include <algorithm>
#include <cmath>
#include <memory>
#include <string>
#include <type_traits>
#include <vector>

#include "batch.hpp"
#include "block_ops.hpp"
#include "grid_barrier.hpp"
#include "solver_common.hpp"


using namespace sfem;

sfem_batch::~sfem_batch() {
    if (K) sfem_csr_destroy(K);
    if (bc) sfem_bc_destroy(bc);
    if (mesh) sfem_mesh_destroy(mesh);
}

namespace sfem {
namespace {

// ------------------------------------------------ padded elimination ---
// A node with any free dof is a block row; its fixed dofs (a partially fixed
// node) get a zero row / column and a unit diagonal, zero rhs and zero start,
// so they stay exactly 0.
__global__ void unit_free_kernel(const uint8_t* __restrict__ fixed, int64_t nunits, int bs,
                                 uint32_t* __restrict__ ufree) {
    const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= nunits) return;
    int c = 0;
    for (int i = 0; i < bs; ++i) c += fixed[u * bs + i] ? 1 : 0;
    ufree[u] = c < bs ? 1u : 0u;
}

// out[i] = upos[idx[i]] (idx[i] == nunits gives the total)
__global__ void gather_pos_kernel(const uint32_t* __restrict__ upos, const int64_t* __restrict__ idx, int64_t n,
                                  int64_t nunits, const uint32_t* __restrict__ total, uint32_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = idx[i] < nunits ? upos[idx[i]] : *total;
}

__global__ void pad_map_kernel(const uint32_t* __restrict__ ufree, const uint32_t* __restrict__ upos,
                               const int64_t* __restrict__ node_off, const uint32_t* __restrict__ first_free,
                               const int64_t* __restrict__ pad_base, int64_t nprob, int64_t nunits,
                               int32_t* __restrict__ pad_of) {
    const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= nunits) return;
    if (!ufree[u]) { pad_of[u] = -1; return; }
    int64_t lo = 0, hi = nprob - 1;  // last problem whose first node is <= u
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) / 2;
        if (node_off[mid] <= u) lo = mid;
        else hi = mid - 1;
    }
    pad_of[u] = (int32_t)(pad_base[lo] + (int64_t)(upos[u] - first_free[lo]));
}

__global__ void pad_blen_kernel(const int64_t* __restrict__ bcolptr, const int32_t* __restrict__ browidx,
                                const int32_t* __restrict__ pad_of, int64_t nunits, int32_t* __restrict__ blen) {
    const int64_t cu = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (cu >= nunits) return;
    const int32_t row = pad_of[cu];
    if (row < 0) return;
    int cnt = 0;
    for (int64_t u = bcolptr[cu]; u < bcolptr[cu + 1]; ++u) cnt += pad_of[browidx[u]] >= 0 ? 1 : 0;
    blen[row] = cnt;
}

__global__ void slice_w_kernel(const int32_t* __restrict__ blen, int64_t nslices, int32_t* __restrict__ sl_w,
                               int64_t* __restrict__ cnt) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nslices) return;
    int w = 0;
    for (int l = 0; l < 64; ++l) w = max(w, blen[s * 64 + l]);
    sl_w[s] = w;
    cnt[s] = (int64_t)w * 64;
}

// Row `row` of the sliced operator from column unit cu of K (K symmetric):
// its free blocks in ascending order, then padding slots (own column, zeros).
template <int BS>
__global__ void sell_fill_pad_kernel(const int64_t* __restrict__ bcolptr, const int32_t* __restrict__ browidx,
                                     const double* __restrict__ bval, const int32_t* __restrict__ pad_of,
                                     int64_t nunits, const int64_t* __restrict__ sl_ptr,
                                     const int32_t* __restrict__ sl_w, int32_t* __restrict__ scol,
                                     double* __restrict__ sval64, float* __restrict__ sval32,
                                     int16_t* __restrict__ sval16, int64_t nrows, double* __restrict__ binv64,
                                     float* __restrict__ binv32, const uint8_t* __restrict__ fixed) {
    constexpr int B2 = BS * BS;
    const int64_t cu = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (cu >= nunits) return;
    const int32_t row = pad_of[cu];
    if (row < 0) return;
    const int64_t s = row / 64;
    const int lane = row % 64;
    int k = 0;
    for (int64_t u = bcolptr[cu]; u < bcolptr[cu + 1]; ++u) {
        const int64_t ru = browidx[u];
        const int32_t c = pad_of[ru];
        if (c < 0) continue;
        const int64_t slot = sl_ptr[s] + (int64_t)k * 64;
        scol[slot + lane] = c;
        // plane j*BS+i holds M[j][i] = K[(row,j),(c,i)] = K[(c,i),(row,j)];
        // fixed dofs of a partially fixed node: zero row / column, unit diagonal
        double m[B2];
#pragma unroll
        for (int j = 0; j < BS; ++j)
#pragma unroll
            for (int i = 0; i < BS; ++i) {
                const bool masked = fixed[cu * BS + j] || fixed[ru * BS + i];
                m[j * BS + i] = masked ? ((ru == cu && i == j) ? 1.0 : 0.0) : bval[u * B2 + i * BS + j];
            }
#pragma unroll
        for (int v = 0; v < B2; ++v) {
            sval64[slot * B2 + v * 64 + lane] = m[v];
            sval32[slot * B2 + v * 64 + lane] = (float)m[v];
            sval16[slot * B2 + v * 64 + lane] = split_correction(m[v]);
        }
        if (c == row) {  // diagonal block: its inverse for block-Jacobi preconditioning
            double inv[B2];
            invert_block<BS>(m, inv);
#pragma unroll
            for (int v = 0; v < B2; ++v) {
                binv64[v * nrows + row] = inv[v];
                binv32[v * nrows + row] = (float)inv[v];
            }
        }
        ++k;
    }
    for (; k < sl_w[s]; ++k) {
        const int64_t slot = sl_ptr[s] + (int64_t)k * 64;
        scol[slot + lane] = row;
        for (int v = 0; v < B2; ++v) {
            sval64[slot * B2 + v * 64 + lane] = 0.0;
            sval32[slot * B2 + v * 64 + lane] = 0.0f;
            sval16[slot * B2 + v * 64 + lane] = 0;
        }
    }
}

// identity blocks for every row (padding rows keep them)
__global__ void binv_identity_kernel(double* __restrict__ binv64, float* __restrict__ binv32, int64_t nrows,
                                     int bs) {
    const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= nrows) return;
    for (int j = 0; j < bs; ++j)
        for (int i = 0; i < bs; ++i) {
            binv64[(j * bs + i) * nrows + row] = i == j ? 1.0 : 0.0;
            binv32[(j * bs + i) * nrows + row] = i == j ? 1.0f : 0.0f;
        }
}

// padding rows (no source column unit, blen < 0): every slot is padding
template <int BS>
__global__ void sell_pad_gap_kernel(const int32_t* __restrict__ blen, int64_t nrows,
                                    const int64_t* __restrict__ sl_ptr, const int32_t* __restrict__ sl_w,
                                    int32_t* __restrict__ scol, double* __restrict__ sval64,
                                    float* __restrict__ sval32, int16_t* __restrict__ sval16) {
    constexpr int B2 = BS * BS;
    const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= nrows || blen[row] >= 0) return;
    const int64_t s = row / 64;
    const int lane = (int)(row % 64);
    for (int k = 0; k < sl_w[s]; ++k) {
        const int64_t slot = sl_ptr[s] + (int64_t)k * 64;
        scol[slot + lane] = (int32_t)row;
        for (int v = 0; v < B2; ++v) {
            sval64[slot * B2 + v * 64 + lane] = 0.0;
            sval32[slot * B2 + v * 64 + lane] = 0.0f;
            sval16[slot * B2 + v * 64 + lane] = 0;
        }
    }
}

__global__ void fill_pad_vectors_kernel(double* __restrict__ rhs, double* __restrict__ dinv64,
                                        float* __restrict__ dinv32, double* __restrict__ x, int64_t npad) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npad) return;
    rhs[i] = 0.0;
    dinv64[i] = 1.0;
    dinv32[i] = 1.0f;
    x[i] = 0.0;
}

// rhs = f - K q_d and 1/diag for every free dof, in padded numbering
__global__ void pad_rhs_kernel(const int64_t* __restrict__ bcolptr, const int32_t* __restrict__ browidx,
                               const double* __restrict__ bval, const int32_t* __restrict__ pad_of,
                               const uint8_t* __restrict__ fixed, const double* __restrict__ qd,
                               const double* __restrict__ f, int64_t n, int bs, double* __restrict__ rhs,
                               double* __restrict__ dinv64, float* __restrict__ dinv32) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int64_t cu = s / bs;
    const int j = (int)(s - cu * bs);
    const int32_t prow = pad_of[cu];
    if (prow < 0) return;
    if (fixed[s]) {  // fixed dof of a partially fixed node: stays 0
        const int64_t pd = (int64_t)prow * bs + j;
        rhs[pd] = 0.0;
        dinv64[pd] = 1.0;
        dinv32[pd] = 1.0f;
        return;
    }
    double lift = 0.0, diag = 0.0;
    for (int64_t u = bcolptr[cu]; u < bcolptr[cu + 1]; ++u) {
        const int64_t r = browidx[u];
        for (int i = 0; i < bs; ++i) {
            const int64_t d = r * bs + i;
            const double v = bval[u * bs * bs + i * bs + j];
            if (fixed[d]) lift = fma(v, qd[d], lift);
            else if (d == s) diag = v;
        }
    }
    const int64_t pd = (int64_t)prow * bs + j;
    rhs[pd] = f[s] - lift;
    dinv64[pd] = diag != 0.0 ? 1.0 / diag : 1.0;
    dinv32[pd] = (float)dinv64[pd];
}

__global__ void batch_recombine_kernel(const int32_t* __restrict__ pad_of, const uint8_t* __restrict__ fixed,
                                       const double* __restrict__ x, const double* __restrict__ qd, int64_t n, int bs,
                                       double* __restrict__ q) {
    const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= n) return;
    const int32_t pr = pad_of[d / bs];
    q[d] = (pr >= 0 && !fixed[d]) ? x[(int64_t)pr * bs + d % bs] : qd[d];
}

__global__ void fold_all_kernel(double* __restrict__ x64, float* __restrict__ xs, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        x64[i] += (double)xs[i];
        xs[i] = 0.0f;
    }
}

// ----------------------------------------------------- persistent PCG ---
// One launch iterates every problem of a table; between the passes of an
// iteration the grid meets at a barrier, and a problem's scalars are formed by
// the blocks that need them.  Per iteration:
//
//   A  per run of slices of one problem: the sums the last pass left (r.z and
//      r.r of an update, or the sums of an FP64 residual) give beta, the
//      stopping tests and what comes next; then either the FP64 residual of
//      the run's rows, if it is due, or q = K p with p = zcoef z + beta p
//      formed in the gathers (p has two buffers), and the slice partials of p.q
//   U  alpha from the partials of p.q, whose sum is left for the next A;
//      x += alpha p; r -= alpha q; z = M^-1 r; slice partials of r.z and r.r
//
// The block that holds a problem's first slice writes its new state to the
// other of two state slots, so no block reads what another one writes.  What
// bounds a small table is the chain barrier - partials - operator - barrier,
// not bytes: the form before this one had four barriers an iteration (six
// with a residual due), a wavefront per slice and skipped finished problems
// item by item.  24 Hex8 problems of 180 to 20,000 nodes, mixed precision,
// 1,229 iterations: 95.5 ms before, 48.3 now; 256 problems up to 31,700
// nodes, split precision, 808 iterations: 314 ms before, 259 now.
//
// A table with more than item_slices active slices per block is bound by HBM
// instead: there p is formed by a pass of its own (a third barrier; the
// gathers then read one vector, not two) and each wavefront takes a whole
// slice with non-temporal operator loads, the residuals that are due spread
// over all blocks (in one block's run they kept the rest waiting: 399 ms).
// Both forms add the same numbers in the same order, so the active problems
// may move from one to the other as others finish.  The line at 8 slices a
// block, 24 / 256 problems as above: always the second form 56.5 / 260 ms, at
// 8 slices 48.3 / 259, at 64 48.3 / 338.  For 3D slices of 64-bit values it
// lies lower (kShareSlices64).

enum TableFlags : int32_t { kFlagDone = 1, kFlagResid = 2, kFlagBuf = 4 };  // what a pass needs of a state

// Slices per block up to which the first form is taken where an operator value
// takes more than 32 bits (FP64, split) in 3D, at most.  One problem, us an
// iteration with the first / the second form on 512 blocks: FP64 1,369 slices
// 66 / 89, 1,839 102 / 70, 3,602 197 / 119; split 63 / 85, 77 / 60, 185 / 100;
// FP32 values 2,532 slices 57 / 65, 3,602 89 / 82, mixed 70 / 77, 5,585 slices
// 125 / 106.  In 2D (9 block columns) FP64 4,697 slices 57 / 59, 11,265 129 /
// 106: item_slices alone decides.
constexpr int kShareSlices64 = 3;

// Work of a 3D slice in the operator pass, a 2D slice being 1: 27 block columns
// of 9 values against 9 of 4.  A server's table holds both; equal counts of
// slices per XCD left those with 2D slices waiting (48 requests of 1e3 to 1e6
// dofs at once, FP64: 2.34 s, 2.13 with the parts cut by work).
constexpr int kWork3 = 6;

constexpr int kMaxGroups = 2048;  // problems, or groups of them, whose activity a block tracks

// The slices still iterated, in table order: groups of `gs` problems, their
// slice counts (0 once all problems of the group are done) and the prefix
// sums; w3, pre3 the same for the slices of 3D problems alone.
struct ActiveSet {
    int pre[kMaxGroups + 1], pre3[kMaxGroups + 1];
    int w[kMaxGroups], w3[kMaxGroups];
};

// Descriptors do not change during a launch: read as constants, so that what
// they hold (the same in every lane) stays in scalar registers.
using DescPtr = const ProbDesc __attribute__((address_space(4)))*;

// A value that is the same in every lane of the wavefront, in scalar registers.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uniform(double v) {
    const int2 u = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(double, make_int2(uniform(u.x), uniform(u.y)));
}

// Prefix sums of w[0..ng); returns the total.  Every thread of the block calls.
__device__ __forceinline__ int active_prefix(const int* w, int* pre, int ng) {
    constexpr int PER = kMaxGroups / kThreads;
    __shared__ int tot[kThreads / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int s = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int g = threadIdx.x * PER + i;
        s += g < ng ? w[g] : 0;
    }
    int inc = s;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(inc, off, 64);
        if (lane >= off) inc += v;
    }
    if (lane == 63) tot[wv] = inc;
    __syncthreads();
    int base = inc - s;
    for (int i = 0; i < wv; ++i) base += tot[i];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int g = threadIdx.x * PER + i;
        if (g < ng) {
            pre[g] = base;
            base += w[g];
            if (g == ng - 1) pre[ng] = base;
        }
    }
    __syncthreads();
    return uniform(pre[ng]);
}

// The operator values of a descriptor as the launch's value source.
template <typename TV>
__device__ __forceinline__ Vals<TV> desc_vals(DescPtr D) {
    if constexpr (std::is_same<TV, SplitVal>::value) return Vals<SplitVal>{(const float*)D->sval, D->sval16};
    else return Vals<TV>{(const TV*)D->sval};
}

// z = preconditioner(r) for the BS dofs of node row `row`
template <int BS, typename T>
__device__ __forceinline__ void apply_pc(DescPtr D, int64_t row, const T (&rv)[BS], T (&zv)[BS]) {
    if (D->block_pc) {
        const SFEM_GLOBAL T* binv = glb((const T*)D->binv);
        T m[BS * BS];
#pragma unroll
        for (int v = 0; v < BS * BS; ++v) m[v] = binv[v * D->binv_stride + row];
#pragma unroll
        for (int j = 0; j < BS; ++j) {
            T acc = 0;
#pragma unroll
            for (int i = 0; i < BS; ++i) acc = fmaT<T>(m[j * BS + i], rv[i], acc);
            zv[j] = acc;
        }
    } else {
        const SFEM_GLOBAL T* dinv = glb((const T*)D->dinv);
#pragma unroll
        for (int j = 0; j < BS; ++j) zv[j] = dinv[row * BS + j] * rv[j];
    }
}

// Update of one node row: x += al p, r -= al q, z = M^-1 r; returns its r.z
// and r.r.
template <int BS, typename T, bool FOLD>
__device__ __forceinline__ void update_row(DescPtr D, int64_t n, const T* p_, T al, bool fold, double& rz,
                                           double& rr) {
    SFEM_GLOBAL double* x64 = glb(D->x64);
    SFEM_GLOBAL T* xs = glb((T*)D->xs);
    SFEM_GLOBAL T* r = glb((T*)D->r);
    SFEM_GLOBAL T* z = glb((T*)D->z);
    const SFEM_GLOBAL T* p = glb(p_);
    const SFEM_GLOBAL T* q = glb((const T*)D->q);
    T pv[BS], qv[BS], rv[BS], zv[BS];
#pragma unroll
    for (int j = 0; j < BS; ++j) {
        pv[j] = p[n * BS + j];
        qv[j] = q[n * BS + j];
        rv[j] = r[n * BS + j];
    }
#pragma unroll
    for (int j = 0; j < BS; ++j) {
        const int64_t i = n * BS + j;
        if constexpr (FOLD) {
            T xi = xs[i];
            if (fold) {
                x64[i] += (double)xi;
                xi = 0;
            }
            xs[i] = fmaT<T>(al, pv[j], xi);
        } else {
            x64[i] = fma((double)al, (double)pv[j], x64[i]);
        }
        rv[j] = fmaT<T>(-al, qv[j], rv[j]);
        r[i] = rv[j];
        rr += (double)rv[j] * (double)rv[j];
    }
    apply_pc<BS, T>(D, n, rv, zv);
#pragma unroll
    for (int j = 0; j < BS; ++j) {
        z[n * BS + j] = zv[j];
        rz += (double)rv[j] * (double)zv[j];
    }
}

// The scalars of a problem from the sums its last pass left: `v` holds p.q,
// r.z, r.r of an update, r.r, r.z, r.p and the rounding-floor scale of an
// FP64 residual, or |rhs|^2 on the first visit.
template <bool FOLD>
__device__ void consume(ProbState& S, const double* v) {
    if (S.init_pending) {
        S.bb = v[0];
        S.tol2bb = S.rtol * S.rtol * S.bb;
        S.delta2 = S.delta * S.delta;
        S.maxrr = S.bb;
        S.rz = 0.0;
        S.rz_prev = HUGE_VAL;
        S.beta = 0.0;
        S.zcoef = 1.0;
        S.best_rr = HUGE_VAL;
        S.best_true = HUGE_VAL;
        S.rr_true = S.bb;
        S.need_update = 1;
        S.capped = S.max_iter <= 0 ? 1 : 0;
        S.init_pending = 0;
    } else if (S.pending == kUpdateSums) {
        const double pq = v[0], trz = v[1], trr = v[2];
        S.rz_prev = S.rz;
        S.rz = trz;
        S.beta = trz / S.rz_prev;
        S.iters += 1;
        S.fold_pending = 0;
        S.zcoef = 1.0;
        S.rr_rec = trr;
        const int64_t since = S.iters - S.last_upd;
        if (trr <= S.tol2bb || trr < S.delta2 * S.maxrr || since >= (S.best_true_it > 256 ? S.best_true_it : 256))
            S.need_update = 1;
        // backstop for a recurrence that stops decreasing: no 2x drop of |r|
        // within max(10000, 4x the iterations it took to reach the best)
        if (trr < 0.25 * S.best_rr) {
            S.best_rr = trr;
            S.best_it = S.iters;
        } else if (S.iters - S.best_it > (4 * S.best_it > 10000 ? 4 * S.best_it : 10000)) {
            S.done = 3;
        }
        if (S.iters >= S.max_iter && !S.done) {  // final FP64 residual, then stop
            S.need_update = 1;
            S.capped = 1;
        }
        if (!(pq > 0.0) || !isfinite(trr)) S.done = 2;
    } else if (S.pending == kResidSums) {
        const double trr = v[0], trz = v[1], trp = v[2];
        // 16x the attainable |r|^2, (eps * || |rhs| + |K||x| ||)^2
        const double floor_rr = 16.0 * kEps64 * kEps64 * v[3];
        S.rr_true = trr;
        S.floor_rr = floor_rr;
        S.updates += 1;
        S.last_upd = S.iters;
        S.need_update = 0;
        S.fold_pending = FOLD ? 1 : 0;
        if (trr <= S.tol2bb) {
            S.done = 1;
        } else if (S.capped) {
            S.done = 4;
        } else {
            S.beta = trz / S.rz_prev;
            S.zcoef = 1.0 - S.beta * (trp / trz);
            S.rz = trz;
            S.maxrr = trr;
            // attainable floor: no 10% gain on the best true residual
            // within 4x of the rounding floor, or twice in a row while
            // the recurrence ran 5x below it
            const bool gap = S.iters > 0 && 25.0 * S.rr_rec < trr;
            if (trr <= 0.81 * S.best_true) {
                S.stall = 0;
                S.best_true_it = S.iters;
            } else if (trr <= floor_rr) {
                S.stall += 2;
            } else if (gap) {
                S.stall += 1;
            }
            if (S.stall >= 2) S.done = 3;
        }
        if (trr < S.best_true) S.best_true = trr;
        if (!isfinite(trr)) S.done = 2;
    }
    S.pending = kNoSums;
}

// This lane's block row of slice `sl` by one wavefront, with the sums of a
// slice shared by four (SharedSlice, sell_combine): one accumulator per
// residue of the block column modulo 4, added in ascending order.  Per pair of
// block columns the column ids and all value loads are issued before any of
// them is used, then the gathers, then the arithmetic; scheduling barriers
// keep the compiler from interleaving loads with their uses, which would leave
// one load in flight per wavefront.
template <int BS, typename TV, typename ACC, bool NT, typename Gather>
__device__ __forceinline__ void sell_row_quads(const int64_t* __restrict__ sl_ptr, const int32_t* __restrict__ sl_w,
                                               const int32_t* __restrict__ scol, Vals<TV> vals, int64_t sl, int lane,
                                               Gather gx, ACC out[BS]) {
    constexpr int B2 = BS * BS;
    using Raw = typename Vals<TV>::Raw;
    const int64_t base = glb(sl_ptr)[sl];
    const int w = glb(sl_w)[sl];
    ACC acc[4][BS];
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int j = 0; j < BS; ++j) acc[h][j] = 0;
    auto add = [&](const Raw (&rv)[B2], const ACC (&xv)[BS], ACC (&s)[BS]) {
#pragma unroll
        for (int j = 0; j < BS; ++j)
#pragma unroll
            for (int i = 0; i < BS; ++i) s[j] = fmaT<ACC>((ACC)vals.decode(rv[j * BS + i]), xv[i], s[j]);
    };
    auto pair = [&](int k, ACC (&sa)[BS], ACC (&sb)[BS]) {
        const int64_t s0 = base + (int64_t)k * 64, s1 = s0 + 64;
        const int64_t c0 = ld_stream<NT>(scol + s0 + lane), c1 = ld_stream<NT>(scol + s1 + lane);
        Raw r0[B2], r1[B2];
#pragma unroll
        for (int m = 0; m < B2; ++m) r0[m] = vals.template raw<NT>(s0 * B2 + lane + m * 64);
#pragma unroll
        for (int m = 0; m < B2; ++m) r1[m] = vals.template raw<NT>(s1 * B2 + lane + m * 64);
        __builtin_amdgcn_sched_barrier(0);
        ACC x0[BS], x1[BS];
        gx(c0, x0);
        gx(c1, x1);
        __builtin_amdgcn_sched_barrier(0);
        add(r0, x0, sa);
        add(r1, x1, sb);
    };
    auto single = [&](int k, ACC (&s)[BS]) {
        const int64_t s0 = base + (int64_t)k * 64;
        const int64_t c0 = ld_stream<NT>(scol + s0 + lane);
        Raw r0[B2];
#pragma unroll
        for (int m = 0; m < B2; ++m) r0[m] = vals.template raw<NT>(s0 * B2 + lane + m * 64);
        ACC x0[BS];
        gx(c0, x0);
        add(r0, x0, s);
    };
    int k = 0;
    for (; k + 4 <= w; k += 4) {
        pair(k, acc[0], acc[1]);
        pair(k + 2, acc[2], acc[3]);
    }
    if (k + 2 <= w) {
        pair(k, acc[0], acc[1]);
        if (k + 3 <= w) single(k + 2, acc[2]);
    } else if (k < w) {
        single(k, acc[0]);
    }
#pragma unroll
    for (int j = 0; j < BS; ++j) out[j] = ((acc[0][j] + acc[1][j]) + acc[2][j]) + acc[3][j];
}

// FP64 residual of one slice: r = rhs - K x, z = M^-1 r; slice partials of
// |r|^2, r.z, r.p and the rounding-floor scale (stride `ps`).  SHARED: by the
// block, each wavefront a quarter of the block columns; otherwise by one
// wavefront, the quarters one after the other and added in the same order.
template <int BS, typename T, bool FOLD, bool SHARED>
__device__ __forceinline__ void resid_slice(DescPtr D, int64_t s, const T* p_, double* part, int64_t ps,
                                            double (*buf)[6][64]) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const SFEM_GLOBAL double* x64 = glb((const double*)D->x64);
    const SFEM_GLOBAL T* xs = glb((const T*)D->xs);
    const SFEM_GLOBAL T* p = glb(p_);
    const SFEM_GLOBAL double* rhs = glb(D->rhs);
    SFEM_GLOBAL T* r = glb((T*)D->r);
    SFEM_GLOBAL T* z = glb((T*)D->z);
    auto gx = [&](int64_t c, double (&x)[BS]) {
#pragma unroll
        for (int i = 0; i < BS; ++i) x[i] = FOLD ? x64[c * BS + i] + (double)xs[c * BS + i] : x64[c * BS + i];
    };
    const int64_t sl = D->slice0 + s;
    double v[2 * BS] = {};
#pragma unroll 1
    for (int h = 0; h < (SHARED ? 1 : 4); ++h) {
        double out[BS], aout[BS];
        sell_row_abs_part<BS, 4>(D->sl_ptr, D->sl_w, D->scol, D->sval64, sl, lane, SHARED ? wv : h, gx, out, aout);
#pragma unroll
        for (int j = 0; j < BS; ++j) {
            v[j] = h ? v[j] + out[j] : out[j];
            v[BS + j] = h ? v[BS + j] + aout[j] : aout[j];
        }
    }
    if constexpr (SHARED) sell_combine<2 * BS, 4>(v, reinterpret_cast<double (*)[2 * BS][64]>(buf));
    if (!SHARED || wv == 0) {
        const int64_t row = sl * 64 + lane;
        double rr = 0.0, rz = 0.0, rp = 0.0, ff = 0.0;
        T rt[BS], zt[BS];
#pragma unroll
        for (int j = 0; j < BS; ++j) {
            const int64_t d = row * BS + j;
            const double res = rhs[d] - v[j];
            const double sc = fabs(rhs[d]) + v[BS + j];
            ff += sc * sc;
            rt[j] = (T)res;
            r[d] = rt[j];
            rr += res * res;
            rp += (double)rt[j] * (double)p[d];
        }
        apply_pc<BS, T>(D, row, rt, zt);
#pragma unroll
        for (int j = 0; j < BS; ++j) {
            z[row * BS + j] = zt[j];
            rz += (double)rt[j] * (double)zt[j];
        }
        const double b0 = wave_sum(rr), b1 = wave_sum(rz), b2 = wave_sum(rp), b3 = wave_sum(ff);
        if (lane == 0) {
            const int64_t t = D->t0 + s;
            glb(part)[t] = b0;
            glb(part)[ps + t] = b1;
            glb(part)[2 * ps + t] = b2;
            glb(part)[3 * ps + t] = b3;
        }
    }
    if constexpr (SHARED) __syncthreads();
}

// q = K p of slices [s0, s1), each shared by the block, and the slice
// partials of p.q.  FLY: p = zc z + beta pold, written to pnew; otherwise
// pold is p.  `sl` holds the first slice's early loads.
template <int BS, typename TV, typename T, bool FLY>
__device__ __forceinline__ void shared_run(SharedSlice<BS, TV, !FLY>& sl, DescPtr D, int64_t s0, int64_t s1,
                                           T beta, T zc, const T* pold_, T* pnew_, double* part,
                                           double (*buf)[6][64]) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const SFEM_GLOBAL T* z = glb((const T*)D->z);
    const SFEM_GLOBAL T* pold = glb(pold_);
    SFEM_GLOBAL T* pnew = glb(pnew_);
    SFEM_GLOBAL T* q = glb((T*)D->q);
    auto gx = [&](int64_t c, T (&x)[BS]) {
#pragma unroll
        for (int i = 0; i < BS; ++i)
            x[i] = FLY ? fmaT<T>(beta, pold[c * BS + i], zc * z[c * BS + i]) : pold[c * BS + i];
    };
    for (int64_t s = s0; s < s1; ++s) {
        const int64_t row = (D->slice0 + s) * 64 + lane;
        T own[BS] = {};
        if (wv == 0) gx(row, own);
        T acc[BS] = {};
        sl.apply(gx, acc);
        if (s + 1 < s1) sl.load(D->sl_ptr, D->sl_w, D->slice0 + s + 1);
        sell_combine<BS, 4>(acc, reinterpret_cast<T (*)[BS][64]>(buf));
        if (wv == 0) {
            double dot = 0.0;
#pragma unroll
            for (int j = 0; j < BS; ++j) {
                if (FLY) pnew[row * BS + j] = own[j];
                q[row * BS + j] = acc[j];
                dot += (double)own[j] * (double)acc[j];
            }
            dot = wave_sum(dot);
            if (lane == 0) glb(part)[D->t0 + s] = dot;
        }
        __syncthreads();
    }
}

// This thread's part of the sums of W arrays of n partials, `stride` apart:
// entries threadIdx.x, + 256, ... in ascending order.  U strides are loaded
// before the first is added: every block of a large problem sums all of its
// slices' partials, and one stride after the other was a chain of up to 66
// loads in front of a pass (16,900 slices, FP64: 557 us an iteration, 505 so).
template <int W, int U>
__device__ __forceinline__ void sum_slices(const double* src, int64_t stride, int n, double* v) {
    const SFEM_GLOBAL double* g = glb(src);
    if (n <= kThreads) {
        if ((int)threadIdx.x < n)
#pragma unroll
            for (int m = 0; m < W; ++m) v[m] += g[m * stride + threadIdx.x];
        return;
    }
    for (int b = 0; b < n; b += U * kThreads) {
        double t[U][W];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = min(b + u * kThreads + (int)threadIdx.x, n - 1);
#pragma unroll
            for (int m = 0; m < W; ++m) t[u][m] = g[m * stride + i];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < W; ++m) v[m] += b + u * kThreads + (int)threadIdx.x < n ? t[u][m] : 0.0;
    }
}

// A run of slices of one problem inside a block's part of the active slices.
struct RunCursor {
    int g, pos, left;  // group, slices of it passed, slices of the part left
    int prob, off;     // problem of the group reached, slices of it passed
};

template <typename TV, typename T, bool FOLD>
__global__ __launch_bounds__(kThreads, 2) void table_pcg_kernel(TableLaunch a) {
    GridBarrier grid{a.bar_ws, a.bar_timeout, 0u, false};
    if (!grid.start(a.bar_grouped != 0)) return;
    __shared__ ActiveSet set;
    __shared__ ProbState S;  // the state of the problem at hand
    __shared__ double sh[16];
    __shared__ double buf[kThreads / 64][6][64];
    const int G = gridDim.x, w = uniform((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const DescPtr probs = (DescPtr)a.probs;
    DescPtr D = probs;
    const int64_t ps = a.nslices;
    double* const partu = a.part + 8 * ps;  // r.z, r.r of the update
    const int gs = (a.nprob + kMaxGroups - 1) / kMaxGroups, ng = (a.nprob + gs - 1) / gs;

    // ---- the active problems ----
    int init = 0;
    for (int g = threadIdx.x; g < ng; g += kThreads) {
        int n = 0, n3 = 0;
        bool any = false;
        for (int p = g * gs; p < min(a.nprob, (g + 1) * gs); ++p) {
            ProbState* st = probs[p].st;
            const bool open = !st->done && probs[p].nslices > 0;
            n += probs[p].nslices;
            n3 += probs[p].bs == 3 ? probs[p].nslices : 0;
            any |= open;
            init |= open && st->init_pending ? 1 : 0;
        }
        set.w[g] = any ? n : 0;
        set.w3[g] = any ? n3 : 0;
    }
    init = __syncthreads_or(init);

    // this block's part of the active slices; consecutive parts share an XCD,
    // and the XCD's part [x0, x0 + xs) by the work of the slices
    const int xn = G % 8 ? 1 : 8, xb = G / xn, bx = blockIdx.x / xn;
    int total = 0, first = 0, count = 0, g0 = 0, x0 = 0, xs = 0;
    bool shared = false;  // the first form
    auto work_before = [&](int g) {
        return (int64_t)uniform(set.pre[g]) + (int64_t)(kWork3 - 1) * uniform(set.pre3[g]);
    };
    auto share = [&](int x, bool mixed) {  // active position at which x of xn equal shares of the work end
        if (x == 0 || x == xn || !mixed) return (int)((int64_t)total * x / xn);
        const int64_t W = work_before(ng) * x / xn;
        int lo = 0, hi = ng;  // the last group that begins at or before W: it has slices
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (work_before(mid) <= W) lo = mid;
            else hi = mid;
        }
        const int64_t w0 = work_before(lo);
        return uniform(set.pre[lo]) + (int)((W - w0) * uniform(set.w[lo]) / (work_before(lo + 1) - w0));
    };
    auto cut = [&] {
        total = active_prefix(set.w, set.pre, ng);
        const int total3 = active_prefix(set.w3, set.pre3, ng);
        shared = (int64_t)a.item_slices * total3 + (int64_t)a.item_slices3 * (total - total3) <=
                 (int64_t)a.item_slices * a.item_slices3 * G;
        const int64_t lb = logical_block();
        first = (int)(lb * total / G);
        count = (int)((lb + 1) * total / G) - first;
        int lo = 0, hi = ng;  // the last group whose prefix is <= first
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (uniform(set.pre[mid]) <= first) lo = mid;
            else hi = mid;
        }
        g0 = lo;
        if (!shared) {
            const bool mixed = total3 > 0 && total3 < total;
            x0 = share(blockIdx.x % xn, mixed);
            xs = share(blockIdx.x % xn + 1, mixed) - x0;
        }
    };
    cut();
    auto runs = [&] {
        const int off = first - uniform(set.pre[g0]);
        return RunCursor{g0, off, count, g0 * gs, off};
    };
    auto next = [&](RunCursor& c, int& p, int& s0, int& s1) {
        while (c.left > 0) {
            const int gw = uniform(set.w[c.g]);
            if (c.pos >= gw) {  // next group that has slices
                ++c.g;
                c.pos = c.off = 0;
                c.prob = c.g * gs;
                continue;
            }
            const int ns = gs == 1 ? gw : probs[c.prob].nslices;
            if (c.off >= ns) {
                c.off -= ns;
                ++c.prob;
                continue;
            }
            const int len = min(ns - c.off, c.left);
            p = c.prob;
            s0 = c.off;
            s1 = c.off + len;
            c.pos += len;
            c.off += len;
            c.left -= len;
            return true;
        }
        return false;
    };

    // ---- the problem at hand: descriptor and state (slot i & 1), the
    // state kept in LDS while a block stays with one problem ----
    int have = -1;
    int64_t have_slot = -1;
    auto copy_words = [&](void* dst, const void* src, int words) {
        for (int i = threadIdx.x; i < words; i += kThreads) ((uint32_t*)dst)[i] = glb((const uint32_t*)src)[i];
    };
    auto take_desc = [&](int p) {
        if (have != p) have_slot = -1;
        have = p;
        D = probs + p;
    };
    auto take_state = [&](int p, int64_t slot) {
        if (have_slot == slot) return;
        __syncthreads();
        copy_words(&S, (slot & 1) ? a.alt + p : D->st, sizeof(ProbState) / 4);
        __syncthreads();
        have_slot = slot;
    };
    // pass A of iteration k reaches a run: state, sums, scalars; the run with
    // the problem's first slice records the new state
    auto advance = [&](int p, int s0, int64_t k, bool fly) __attribute__((always_inline)) {
        take_state(p, k);
        const double* pa = a.part + ((k + 1) & 1) * 4 * ps + D->t0;
        const double* pu = partu + D->t0;
        const int ns = D->nslices;
        double pq = 0.0;  // thread 0
        if (!S.done && (S.init_pending || S.pending != kNoSums)) {
            if (threadIdx.x == 0) pq = glb(a.pq)[p];
            double v[4] = {};
            if (S.init_pending) sum_slices<1, 8>(pa, 0, ns, v);
            else if (S.pending == kUpdateSums) sum_slices<2, 4>(pu, ps, ns, v + 1);
            else sum_slices<4, 2>(pa, ps, ns, v);
#pragma unroll
            for (int m = 0; m < 4; ++m) v[m] = wave_sum(v[m]);
            if (lane == 0)
#pragma unroll
                for (int m = 0; m < 4; ++m) sh[w * 4 + m] = v[m];
        }
        __syncthreads();
        if (threadIdx.x == 0 && !S.done) {
            if (S.init_pending || S.pending != kNoSums) {
                double v[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) v[m] = (sh[m] + sh[4 + m]) + (sh[8 + m] + sh[12 + m]);
                if (!S.init_pending && S.pending == kUpdateSums) v[0] = pq;
                consume<FOLD>(S, v);
            }
            if (!S.done) {
                S.pending = S.need_update ? kResidSums : kUpdateSums;
                if (!S.need_update && fly) S.pbuf ^= 1;
            }
        }
        __syncthreads();
        have_slot = k + 1;
        if (s0 == 0) {
            uint32_t* dst = (uint32_t*)(((k + 1) & 1) ? a.alt + p : D->st);
            for (int i = threadIdx.x; i < (int)(sizeof(ProbState) / 4); i += kThreads)
                glb(dst)[i] = ((const uint32_t*)&S)[i];
            if (threadIdx.x == 0)
                glb(a.flags)[((k + 1) & 1) * a.nprob + p] =
                    (S.done ? kFlagDone : 0) | (S.need_update ? kFlagResid : 0) | (S.pbuf ? kFlagBuf : 0);
        }
    };

    // ---- first launch of a problem: slice partials of |rhs|^2 ----
    if (init) {
        RunCursor c = runs();
        for (int p, s0, s1; next(c, p, s0, s1);) {
            take_desc(p);
            take_state(p, 0);
            if (!S.init_pending) continue;
            const SFEM_GLOBAL double* rhs = glb(D->rhs);
            const int n = 64 * D->bs;
            for (int64_t s = s0 + w; s < s1; s += kThreads / 64) {
                double v = 0.0;
                for (int i = lane; i < n; i += 64) {
                    const double b = rhs[(D->slice0 + s) * n + i];
                    v = fma(b, b, v);
                }
                v = wave_sum(v);
                if (lane == 0) glb(a.part)[4 * ps + D->t0 + s] = v;
            }
        }
        if (!grid.sync()) return;
    }

    int64_t k = 0;
    for (; k < a.iters && total > 0; ++k) {
        double* pa = a.part + (k & 1) * 4 * ps;
        if (shared) {
            // ---- A, slices shared by the block ----
            auto run = [&](auto bs, int p, int s0, int s1) {
                constexpr int BS = decltype(bs)::value;
                SharedSlice<BS, TV> sl(D->scol, desc_vals<TV>(D));
                sl.load(D->sl_ptr, D->sl_w, D->slice0 + s0);
                advance(p, s0, k, true);
                if (uniform(S.done)) return;
                const int pb = uniform(S.pbuf);
                if (uniform(S.need_update)) {
                    for (int s = s0; s < s1; ++s)
                        resid_slice<BS, T, FOLD, true>(D, s, (const T*)D->p[pb], pa, ps, buf);
                } else {
                    shared_run<BS, TV, T, true>(sl, D, s0, s1, (T)uniform(S.beta), (T)uniform(S.zcoef), (const T*)D->p[pb ^ 1],
                                                (T*)D->p[pb], pa, buf);
                }
            };
            RunCursor c = runs();
            for (int p, s0, s1; next(c, p, s0, s1);) {
                take_desc(p);
                if (D->bs == 3) run(std::integral_constant<int, 3>{}, p, s0, s1);
                else run(std::integral_constant<int, 2>{}, p, s0, s1);
            }
        } else {
            // ---- A, p by a pass of its own ----
            RunCursor c = runs();
            for (int p, s0, s1; next(c, p, s0, s1);) {
                take_desc(p);
                advance(p, s0, k, false);
                if (uniform(S.done)) continue;
                const int pb = uniform(S.pbuf);
                if (uniform(S.need_update)) continue;
                const T beta = (T)uniform(S.beta), zc = (T)uniform(S.zcoef);
                SFEM_GLOBAL T* pv = glb((T*)D->p[pb]);
                const SFEM_GLOBAL T* z = glb((const T*)D->z);
                const int64_t n = 64 * D->bs;
                for (int64_t i = (D->slice0 + s0) * n + threadIdx.x; i < (D->slice0 + s1) * n; i += kThreads)
                    pv[i] = fmaT<T>(beta, pv[i], zc * z[i]);
            }
            if (!grid.sync()) return;
            // ---- q = K p or the residual: the blocks of an XCD go through
            // its part of the active slices together, a slice per wavefront (a
            // residual pass, twice the bytes, so meets all blocks alike); what
            // is left after the last whole round is shared slice by slice ----
            const int rest = xs % (4 * xb);
            const int whole = rest > 3 * xb ? xs : xs - rest;
            auto spmv = [&](auto bs, DescPtr P, int64_t s, int buf_of) {
                constexpr int BS = decltype(bs)::value;
                const SFEM_GLOBAL T* pv = glb((const T*)P->p[buf_of]);
                SFEM_GLOBAL T* q = glb((T*)P->q);
                auto gx = [&](int64_t col, T (&x)[BS]) {
#pragma unroll
                    for (int i = 0; i < BS; ++i) x[i] = pv[col * BS + i];
                };
                const int64_t row = (P->slice0 + s) * 64 + lane;
                T out[BS];
                sell_row_quads<BS, TV, T, true>(P->sl_ptr, P->sl_w, P->scol, desc_vals<TV>(P), P->slice0 + s, lane, gx,
                                                out);
                double dot = 0.0;
#pragma unroll
                for (int j = 0; j < BS; ++j) {
                    q[row * BS + j] = out[j];
                    dot += (double)pv[row * BS + j] * (double)out[j];
                }
                dot = wave_sum(dot);
                if (lane == 0) glb(pa)[P->t0 + s] = dot;
            };
            auto find = [&](int at, int& off) {  // problem and slice of an active position
                int lo = 0, hi = ng;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) / 2;
                    if (uniform(set.pre[mid]) <= at) lo = mid;
                    else hi = mid;
                }
                off = at - uniform(set.pre[lo]);
                int q = lo * gs;
                if (gs > 1)
                    while (off >= probs[q].nslices) off -= probs[q++].nslices;
                return q;
            };
            const SFEM_GLOBAL int32_t* fl = glb(a.flags) + ((k + 1) & 1) * a.nprob;
            for (int i = 4 * bx + w; i < whole; i += 4 * xb) {
                int off;
                const int q = find(x0 + i, off);
                const int f = uniform(fl[q]);
                if (f & kFlagDone) continue;
                const DescPtr P = probs + q;
                if (f & kFlagResid) {
                    const T* pv = (const T*)P->p[f & kFlagBuf ? 1 : 0];
                    if (P->bs == 3) resid_slice<3, T, FOLD, false>(P, off, pv, pa, ps, buf);
                    else resid_slice<2, T, FOLD, false>(P, off, pv, pa, ps, buf);
                } else if (P->bs == 3) spmv(std::integral_constant<int, 3>{}, P, off, f & kFlagBuf ? 1 : 0);
                else spmv(std::integral_constant<int, 2>{}, P, off, f & kFlagBuf ? 1 : 0);
            }
            for (int i = whole + bx; i < xs; i += xb) {
                int off;
                const int q = find(x0 + i, off);
                const int f = uniform(fl[q]);
                if (f & kFlagDone) continue;
                const DescPtr P = probs + q;
                auto run = [&](auto bs) {
                    constexpr int BS = decltype(bs)::value;
                    if (f & kFlagResid) {
                        resid_slice<BS, T, FOLD, true>(P, off, (const T*)P->p[f & kFlagBuf ? 1 : 0], pa, ps, buf);
                        return;
                    }
                    SharedSlice<BS, TV, true> sl(P->scol, desc_vals<TV>(P));
                    sl.load(P->sl_ptr, P->sl_w, P->slice0 + off);
                    shared_run<BS, TV, T, false>(sl, P, off, off + 1, T(0), T(0), (const T*)P->p[f & kFlagBuf ? 1 : 0],
                                                 nullptr, pa, buf);
                };
                if (P->bs == 3) run(std::integral_constant<int, 3>{});
                else run(std::integral_constant<int, 2>{});
            }
        }
        if (!grid.sync()) return;

        // ---- U, a wavefront per slice ----
        // problems that were done before this iteration leave the active set:
        // both state slots hold their final state (one group per thread and
        // iteration in turn)
        const int gd = (int)(k % ((ng + kThreads - 1) / kThreads)) * kThreads + threadIdx.x;
        int gone = 0;
        if (k > 0 && gd < ng && set.w[gd] > 0) {
            gone = 1;
            for (int p = gd * gs; p < min(a.nprob, (gd + 1) * gs); ++p)
                gone &= (gs > 1 && probs[p].nslices == 0) || (glb(a.flags)[(k & 1) * a.nprob + p] & kFlagDone) ? 1 : 0;
        }
        RunCursor c = runs();
        for (int p, s0, s1; next(c, p, s0, s1);) {
            take_desc(p);
            take_state(p, k + 1);
            if (uniform(S.done | S.need_update)) continue;
            const int pb = uniform(S.pbuf);
            double v = 0.0;
            sum_slices<1, 8>(pa + D->t0, 0, D->nslices, &v);
            const double pq = block_sum_256(v, sh);
            if (s0 == 0 && threadIdx.x == 0) glb(a.pq)[p] = pq;
            const T al = (T)uniform(S.rz / pq);
            const bool fold = FOLD && uniform(S.fold_pending);
            const T* pv = (const T*)D->p[pb];
            for (int64_t s = s0 + w; s < s1; s += kThreads / 64) {
                const int64_t row = (D->slice0 + s) * 64 + lane;
                double rz = 0.0, rr = 0.0;
                if (D->bs == 3) update_row<3, T, FOLD>(D, row, pv, al, fold, rz, rr);
                else update_row<2, T, FOLD>(D, row, pv, al, fold, rz, rr);
                rz = wave_sum(rz);
                rr = wave_sum(rr);
                if (lane == 0) {
                    glb(partu)[D->t0 + s] = rz;
                    glb(partu)[ps + D->t0 + s] = rr;
                }
            }
        }
        if (!grid.sync()) return;
        if (__syncthreads_or(gone)) {
            if (gone) set.w[gd] = set.w3[gd] = 0;
            __syncthreads();
            cut();
        }
    }

    // ---- the sums the last pass left, and the state back to the host's slot ----
    for (int p = blockIdx.x; p < a.nprob; p += G) {
        take_desc(p);
        have_slot = -1;
        take_state(p, 0);
        if (S.done) continue;
        if (D->nslices == 0) {  // no rows: solved
            if (threadIdx.x == 0) {
                D->st->init_pending = D->st->need_update = 0;
                D->st->updates = 1;
                D->st->done = 1;
            }
            continue;
        }
        have_slot = -1;
        take_state(p, k);
        const double* pa = a.part + ((k + 1) & 1) * 4 * ps + D->t0;
        double v[4] = {};
        if (S.pending == kUpdateSums) sum_slices<2, 4>(partu + D->t0, ps, D->nslices, v + 1);
        else if (S.pending != kNoSums) sum_slices<4, 2>(pa, ps, D->nslices, v);
        for (int m = 0; m < 4; ++m) v[m] = block_sum_256(v[m], sh);
        if (S.pending == kUpdateSums) v[0] = glb(a.pq)[p];
        if (threadIdx.x == 0) {
            if (!S.done && !S.init_pending && S.pending != kNoSums) consume<FOLD>(S, v);
            *D->st = S;
        }
    }
}

template <typename TV, typename T, bool FOLD>
void launch_table(sfem_ctx* ctx, const TableLaunch& a, int grid) {
    TableLaunch arg = a;
    void* args[] = {&arg};
    SFEM_HIP(hipLaunchCooperativeKernel((const void*)table_pcg_kernel<TV, T, FOLD>, dim3(grid), dim3(kThreads), args,
                                        0, ctx->stream));
}

template <typename TV, typename T, bool FOLD>
int resident_blocks() {
    int per_cu = 0;
    SFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, table_pcg_kernel<TV, T, FOLD>, kThreads, 0));
    return per_cu;
}

}  // namespace

size_t prec_vec_bytes(int precision) { return precision == SFEM_PREC_MIXED ? sizeof(float) : sizeof(double); }

int table_max_blocks_per_cu(int precision) {
    switch (precision) {
        case SFEM_PREC_FP64: return resident_blocks<double, double, false>();
        case SFEM_PREC_MIXED: return resident_blocks<float, float, true>();
        case SFEM_PREC_FP32_MATRIX: return resident_blocks<float, double, false>();
        case SFEM_PREC_SPLIT: return resident_blocks<SplitVal, double, false>();
        default: fail(SFEM_ERR_ARGUMENT, "unknown precision");
    }
}

void table_launch(sfem_ctx* ctx, int precision, const TableLaunch& a0, int grid) {
    if (a0.nprob <= 0) return;
    if (!ctx->bar_ws) ctx->bar_ws = static_cast<unsigned*>(ctx->alloc->alloc(sizeof(unsigned) * kBarWords));
    TableLaunch a = a0;
    a.bar_ws = ctx->bar_ws;
    a.bar_timeout = ctx->bar_timeout_ticks;
    a.bar_grouped = ctx->bar_grouped ? 1 : 0;
    a.item_slices = std::min(a.item_slices, 1 << 20);  // more than any grid has to share
    const bool wide = precision == SFEM_PREC_FP64 || precision == SFEM_PREC_SPLIT;
    a.item_slices3 = wide ? std::min(a.item_slices, kShareSlices64) : a.item_slices;
    SFEM_HIP(hipMemsetAsync(a.bar_ws, 0, sizeof(unsigned) * kBarWords, ctx->stream));
    switch (precision) {
        case SFEM_PREC_FP64: launch_table<double, double, false>(ctx, a, grid); break;
        case SFEM_PREC_MIXED: launch_table<float, float, true>(ctx, a, grid); break;
        case SFEM_PREC_FP32_MATRIX: launch_table<float, double, false>(ctx, a, grid); break;
        case SFEM_PREC_SPLIT: launch_table<SplitVal, double, false>(ctx, a, grid); break;
        default: fail(SFEM_ERR_ARGUMENT, "unknown precision");
    }
    unsigned flags[2] = {0u, 0u};
    d2h(ctx, flags, a.bar_ws + kBarFlags, sizeof(flags));
    ctx->bar_last_grouped = a.bar_grouped && flags[0] == 0u;
    if (flags[1]) fail(SFEM_ERR_DEVICE, "persistent solver: a grid barrier wait exceeded its time limit");
}

TableLaunch table_prepare(sfem_ctx* ctx, TableWork& W, std::vector<ProbDesc>& descs, int item_slices) {
    const size_t np = descs.size();
    int64_t t0 = 0;
    for (ProbDesc& D : descs) {
        D.t0 = t0;
        t0 += D.nslices;
    }
    if (W.descs.size() < np) {
        W.descs.reset(ctx, np * 2);
        W.alt.reset(ctx, np * 2);
        W.pq.reset(ctx, np * 2);
        W.flags.reset(ctx, np * 4);
    }
    if (W.part.size() < (size_t)t0 * kTableSums) W.part.reset(ctx, (size_t)t0 * kTableSums * 2);
    h2d(ctx, W.descs.get(), descs.data(), sizeof(ProbDesc) * np);
    TableLaunch a{};
    a.probs = W.descs.get();
    a.nprob = (int)np;
    a.item_slices = item_slices;
    a.nslices = t0;
    a.part = W.part.get();
    a.alt = W.alt.get();
    a.pq = W.pq.get();
    a.flags = W.flags.get();
    return a;
}

void table_fold(sfem_ctx* ctx, double* x64, void* xs, int64_t n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(fold_all_kernel, dim3(std::min<unsigned>(grid_for(n, 256), 4096)), dim3(256), 0, ctx->stream,
                       x64, (float*)xs, n);
    SFEM_LAUNCH_CHECK();
}

int table_grid(sfem_ctx* ctx, int precision, int blocks_per_cu) {
    const int maxb = table_max_blocks_per_cu(precision);
    if (maxb < 1) fail(SFEM_ERR_DEVICE, "persistent solver kernel cannot be resident");
    const int b = blocks_per_cu > 0 ? std::min(blocks_per_cu, maxb) : std::min(maxb, 2);
    return b * ctx->n_cu;
}

void batch_build(sfem_ctx* ctx, sfem_batch* B) {
    const sfem_csr* K = B->K;
    const sfem_bc* bc = B->bc;
    const int bs = K->bs;
    if (bs != B->ndof || bs < 2 || bs > 3) fail(SFEM_ERR_UNSUPPORTED, "batch: needs node-blocked 2D or 3D dofs");
    const int64_t nunits = K->nunits;
    B->bs = bs;
    B->n = K->n;
    hipEvent_t e0, e1;
    SFEM_HIP(hipEventCreate(&e0));
    SFEM_HIP(hipEventCreate(&e1));
    SFEM_HIP(hipEventRecord(e0, ctx->stream));
    DevBuf<uint32_t> ufree(ctx, (size_t)nunits), upos(ctx, (size_t)nunits), utot(ctx, 1);
    const dim3 gu(grid_for(nunits, 256));
    hipLaunchKernelGGL(unit_free_kernel, gu, dim3(256), 0, ctx->stream, bc->fixed.get(), nunits, bs, ufree.get());
    SFEM_LAUNCH_CHECK();
    exclusive_scan_u32_dev(ctx, ufree.get(), upos.get(), nunits, utot.get());
    const int64_t np = B->nprob;
    DevBuf<int64_t> doff(ctx, (size_t)np + 1);
    h2d(ctx, doff.get(), B->node_off.data(), sizeof(int64_t) * (np + 1));
    DevBuf<uint32_t> dfirst(ctx, (size_t)np + 1);
    hipLaunchKernelGGL(gather_pos_kernel, dim3(grid_for(np + 1, 256)), dim3(256), 0, ctx->stream, upos.get(),
                       doff.get(), np + 1, nunits, utot.get(), dfirst.get());
    SFEM_LAUNCH_CHECK();
    std::vector<uint32_t> first((size_t)np + 1);
    d2h(ctx, first.data(), dfirst.get(), sizeof(uint32_t) * (np + 1));
    // padded layout: each problem starts on a new slice
    std::vector<int64_t> pad_base((size_t)np + 1);
    B->hprobs.resize((size_t)np);
    int64_t base = 0;
    for (int64_t p = 0; p < np; ++p) {
        const int64_t nfu = (int64_t)first[p + 1] - (int64_t)first[p];
        const int64_t ns = (nfu + 63) / 64;
        pad_base[p] = base;
        BatchProb& P = B->hprobs[(size_t)p];
        P.slice0 = base / 64;
        P.slice1 = P.slice0 + ns;
        P.n_free = nfu * bs;
        base += ns * 64;
    }
    pad_base[(size_t)np] = base;
    if (base * bs >= (int64_t(1) << 31)) fail(SFEM_ERR_UNSUPPORTED, "batch: 2^31 or more padded dofs");
    if (base == 0) fail(SFEM_ERR_ARGUMENT, "batch: no free dofs");
    B->npad = base * bs;
    B->nslices = base / 64;
    DevBuf<int64_t> dpb(ctx, (size_t)np + 1);
    h2d(ctx, dpb.get(), pad_base.data(), sizeof(int64_t) * (np + 1));
    B->pad_of.reset(ctx, (size_t)nunits);
    hipLaunchKernelGGL(pad_map_kernel, gu, dim3(256), 0, ctx->stream, ufree.get(), upos.get(), doff.get(),
                       dfirst.get(), dpb.get(), np, nunits, B->pad_of.get());
    SFEM_LAUNCH_CHECK();
    // slice widths; blen < 0 marks padding rows
    DevBuf<int32_t> blen(ctx, (size_t)base);
    memset_d(ctx, blen.get(), 0xFF, sizeof(int32_t) * base);
    hipLaunchKernelGGL(pad_blen_kernel, gu, dim3(256), 0, ctx->stream, K->bcolptr.get(), K->browidx.get(),
                       B->pad_of.get(), nunits, blen.get());
    SFEM_LAUNCH_CHECK();
    B->sl_w.reset(ctx, (size_t)B->nslices);
    B->sl_ptr.reset(ctx, (size_t)B->nslices + 1);
    DevBuf<int64_t> cnt(ctx, (size_t)B->nslices + 1);
    memset_d(ctx, cnt.get(), 0, sizeof(int64_t) * (B->nslices + 1));
    hipLaunchKernelGGL(slice_w_kernel, dim3(grid_for(B->nslices, 256)), dim3(256), 0, ctx->stream, blen.get(),
                       B->nslices, B->sl_w.get(), cnt.get());
    SFEM_LAUNCH_CHECK();
    const int64_t slots = exclusive_scan_i64(ctx, cnt.get(), B->sl_ptr.get(), B->nslices + 1);
    B->sell_blocks = slots;
    B->scol.reset(ctx, (size_t)slots);
    B->sval64.reset(ctx, (size_t)slots * bs * bs);
    B->sval32.reset(ctx, (size_t)slots * bs * bs);
    B->sval16.reset(ctx, (size_t)slots * bs * bs);
    B->binv64.reset(ctx, (size_t)base * bs * bs);
    B->binv32.reset(ctx, (size_t)base * bs * bs);
    const dim3 gr(grid_for(base, 256));
    hipLaunchKernelGGL(binv_identity_kernel, gr, dim3(256), 0, ctx->stream, B->binv64.get(), B->binv32.get(), base,
                       bs);
    SFEM_LAUNCH_CHECK();
    if (bs == 3) {
        hipLaunchKernelGGL(sell_fill_pad_kernel<3>, gu, dim3(256), 0, ctx->stream, K->bcolptr.get(), K->browidx.get(),
                           K->bval.get(), B->pad_of.get(), nunits, B->sl_ptr.get(), B->sl_w.get(), B->scol.get(),
                           B->sval64.get(), B->sval32.get(), B->sval16.get(), base, B->binv64.get(),
                           B->binv32.get(), bc->fixed.get());
        SFEM_LAUNCH_CHECK();
        hipLaunchKernelGGL(sell_pad_gap_kernel<3>, gr, dim3(256), 0, ctx->stream, blen.get(), base, B->sl_ptr.get(),
                           B->sl_w.get(), B->scol.get(), B->sval64.get(), B->sval32.get(), B->sval16.get());
    } else {
        hipLaunchKernelGGL(sell_fill_pad_kernel<2>, gu, dim3(256), 0, ctx->stream, K->bcolptr.get(), K->browidx.get(),
                           K->bval.get(), B->pad_of.get(), nunits, B->sl_ptr.get(), B->sl_w.get(), B->scol.get(),
                           B->sval64.get(), B->sval32.get(), B->sval16.get(), base, B->binv64.get(),
                           B->binv32.get(), bc->fixed.get());
        SFEM_LAUNCH_CHECK();
        hipLaunchKernelGGL(sell_pad_gap_kernel<2>, gr, dim3(256), 0, ctx->stream, blen.get(), base, B->sl_ptr.get(),
                           B->sl_w.get(), B->scol.get(), B->sval64.get(), B->sval32.get(), B->sval16.get());
    }
    SFEM_LAUNCH_CHECK();
    B->rhs.reset(ctx, (size_t)B->npad);
    B->x.reset(ctx, (size_t)B->npad);
    B->dinv64.reset(ctx, (size_t)B->npad);
    B->dinv32.reset(ctx, (size_t)B->npad);
    hipLaunchKernelGGL(fill_pad_vectors_kernel, dim3(grid_for(B->npad, 256)), dim3(256), 0, ctx->stream,
                       B->rhs.get(), B->dinv64.get(), B->dinv32.get(), B->x.get(), B->npad);
    SFEM_LAUNCH_CHECK();
    hipLaunchKernelGGL(pad_rhs_kernel, dim3(grid_for(B->n, 256)), dim3(256), 0, ctx->stream, K->bcolptr.get(),
                       K->browidx.get(), K->bval.get(), B->pad_of.get(), bc->fixed.get(), bc->qd.get(), bc->f.get(),
                       B->n, bs, B->rhs.get(), B->dinv64.get(), B->dinv32.get());
    SFEM_LAUNCH_CHECK();
    SFEM_HIP(hipEventRecord(e1, ctx->stream));
    sync(ctx);
    float ms = 0;
    SFEM_HIP(hipEventElapsedTime(&ms, e0, e1));
    B->t_eliminate_ms = ms;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
}

void batch_ensure_work(sfem_ctx* ctx, sfem_batch* B, int precision) {
    const size_t vb = prec_vec_bytes(precision);
    if (B->work_vb != vb) {
        B->wr.reset(ctx, vb * B->npad);
        B->wz.reset(ctx, vb * B->npad);
        B->wp.reset(ctx, vb * B->npad);
        B->wp2.reset(ctx, vb * B->npad);
        B->wq.reset(ctx, vb * B->npad);
        B->work_vb = vb;
    }
    if (precision == SFEM_PREC_MIXED && B->wxs.size() != sizeof(float) * B->npad)
        B->wxs.reset(ctx, sizeof(float) * B->npad);
}

ProbDesc batch_desc(sfem_batch* B, int precision, int preconditioner, ProbState* st, const BatchProb& P) {
    ProbDesc D{};
    D.sl_ptr = B->sl_ptr.get();
    D.sl_w = B->sl_w.get();
    D.scol = B->scol.get();
    D.sval = precision == SFEM_PREC_FP64 ? (const void*)B->sval64.get() : (const void*)B->sval32.get();
    D.sval16 = B->sval16.get();
    D.sval64 = B->sval64.get();
    D.rhs = B->rhs.get();
    D.x64 = B->x.get();
    D.xs = precision == SFEM_PREC_MIXED ? (void*)B->wxs.get() : nullptr;
    D.r = B->wr.get();
    D.z = B->wz.get();
    D.p[0] = B->wp.get();
    D.p[1] = B->wp2.get();
    D.q = B->wq.get();
    D.dinv = precision == SFEM_PREC_MIXED ? (const void*)B->dinv32.get() : (const void*)B->dinv64.get();
    D.binv = precision == SFEM_PREC_MIXED ? (const void*)B->binv32.get() : (const void*)B->binv64.get();
    D.binv_stride = B->nslices * 64;
    D.block_pc = preconditioner == SFEM_PC_BLOCK_JACOBI ? 1 : 0;
    D.st = st;
    D.bs = B->bs;
    D.slice0 = P.slice0;
    D.nslices = (int32_t)(P.slice1 - P.slice0);
    return D;
}

ProbState initial_state(const sfem_solve_opts& o) {
    ProbState S{};
    S.rtol = o.rtol;
    S.delta = o.reliable_delta;
    S.max_iter = o.max_iter;
    S.init_pending = 1;
    return S;
}

void batch_reset(sfem_ctx* ctx, sfem_batch* B, int precision, const sfem_solve_opts& o, ProbState* d_st) {
    batch_ensure_work(ctx, B, precision);
    const size_t vb = prec_vec_bytes(precision);
    memset_d(ctx, B->wp.get(), 0, vb * B->npad);
    if (precision == SFEM_PREC_MIXED) memset_d(ctx, B->wxs.get(), 0, sizeof(float) * B->npad);
    if (o.x0_zero) memset_d(ctx, B->x.get(), 0, sizeof(double) * B->npad);
    if (d_st) {
        std::vector<ProbState> hst((size_t)B->nprob, initial_state(o));
        h2d(ctx, d_st, hst.data(), sizeof(ProbState) * B->nprob);
    }
}

double batch_run(sfem_ctx* ctx, sfem_batch* B, const sfem_solve_opts& o, int item_slices, int blocks_per_cu,
                 int64_t* launches) {
    const int prec = o.precision;
    if (prec != SFEM_PREC_FP64 && prec != SFEM_PREC_MIXED && prec != SFEM_PREC_FP32_MATRIX && prec != SFEM_PREC_SPLIT)
        fail(SFEM_ERR_ARGUMENT, "batch solve: unknown precision");
    if (o.preconditioner != SFEM_PC_JACOBI && o.preconditioner != SFEM_PC_BLOCK_JACOBI)
        fail(SFEM_ERR_ARGUMENT, "batch solve: unknown preconditioner");
    if (item_slices < 1) fail(SFEM_ERR_ARGUMENT, "batch solve: item_slices must be >= 1");
    if (o.max_iter < 0) fail(SFEM_ERR_ARGUMENT, "batch solve: max_iter must be >= 0");
    if (B->st.size() != (size_t)B->nprob) B->st.reset(ctx, (size_t)B->nprob);
    batch_reset(ctx, B, prec, o, B->st.get());
    std::vector<ProbDesc> descs((size_t)B->nprob);
    for (int64_t p = 0; p < B->nprob; ++p)
        descs[(size_t)p] = batch_desc(B, prec, o.preconditioner, B->st.get() + p, B->hprobs[(size_t)p]);
    TableWork work;
    TableLaunch a = table_prepare(ctx, work, descs, item_slices);
    const int grid = table_grid(ctx, prec, blocks_per_cu);
    // One launch holds the whole solve unless a per-launch iteration budget
    // (check_every > 0) splits it; the state lives in memory either way.  A
    // problem needs at most 2 max_iter + 2 loop passes: an FP64 residual at the
    // start and after every iteration; the last sums are taken as a launch ends.
    const int64_t need = 2 * std::min<int64_t>(o.max_iter, INT64_MAX / 4) + 3;
    const int64_t budget = o.check_every > 0 ? std::min<int64_t>(o.check_every, need) : need;
    hipEvent_t e0, e1;
    SFEM_HIP(hipEventCreate(&e0));
    SFEM_HIP(hipEventCreate(&e1));
    SFEM_HIP(hipEventRecord(e0, ctx->stream));
    std::vector<ProbState> hst((size_t)B->nprob);
    int64_t nl = 0, run = 0;
    while (true) {
        a.iters = budget;
        table_launch(ctx, prec, a, grid);
        ++nl;
        run += budget;
        d2h(ctx, hst.data(), B->st.get(), sizeof(ProbState) * B->nprob);
        const bool all = std::all_of(hst.begin(), hst.end(), [](const ProbState& s) { return s.done != 0; });
        if (all || run >= need) break;
    }
    if (prec == SFEM_PREC_MIXED) table_fold(ctx, B->x.get(), B->wxs.get(), B->npad);
    SFEM_HIP(hipEventRecord(e1, ctx->stream));
    sync(ctx);
    float ms = 0;
    SFEM_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (launches) *launches = nl;
    return ms;
}

void batch_solution(sfem_ctx* ctx, const sfem_batch* B, double* q) {
    DevBuf<double> dq(ctx, (size_t)B->n);
    hipLaunchKernelGGL(batch_recombine_kernel, dim3(grid_for(B->n, 256)), dim3(256), 0, ctx->stream,
                       B->pad_of.get(), B->fixed.get(), B->x.get(), B->qd.get(), B->n, B->bs, dq.get());
    SFEM_LAUNCH_CHECK();
    d2h(ctx, q, dq.get(), sizeof(double) * B->n);
}

// The padded operator of problems already on the device as one
// concatenated mesh (node ids offset per problem) with its loads and
// constraints.  Takes ownership of mesh and bc (both are destroyed once the
// operator exists, or on failure).  nfree: free dofs per problem.
sfem_batch* batch_from_device(sfem_ctx* ctx, int64_t nprob, sfem_mesh* mesh, sfem_bc* bc,
                              const std::vector<int64_t>& node_offsets, const std::vector<int64_t>& nfree) {
    std::unique_ptr<sfem_batch> B(new sfem_batch());
    B->ctx = ctx;
    B->mesh = mesh;
    B->bc = bc;
    B->nprob = nprob;
    B->ndim = mesh->ndim;
    B->ndof = mesh->ndof;
    B->node_off = node_offsets;
    const int64_t N = mesh->n_nodes;
    const int n_dof = mesh->ndof;
    sfem_csr* K = nullptr;
    int s = sfem_assemble_mesh(ctx, mesh, SFEM_ASM_DEFAULT, &K);
    if (s) fail(s, ctx->last_error);
    B->K = K;
    B->t_assemble_ms = K->t_total;
    if (K->n != N * n_dof || K->bs != n_dof)
        fail(SFEM_ERR_ARGUMENT, "batch_create: every node must belong to an element");
    if (bc->n != K->n) fail(SFEM_ERR_ARGUMENT, "batch_create: loads do not match the mesh");
    batch_build(ctx, B.get());
    B->qd.reset(ctx, (size_t)B->n);
    SFEM_HIP(hipMemcpyAsync(B->qd.get(), bc->qd.get(), sizeof(double) * B->n, hipMemcpyDeviceToDevice, ctx->stream));
    B->fixed.reset(ctx, (size_t)B->n);
    SFEM_HIP(hipMemcpyAsync(B->fixed.get(), bc->fixed.get(), (size_t)B->n, hipMemcpyDeviceToDevice, ctx->stream));
    // free dofs per problem (a partially fixed node keeps only its free dofs)
    for (int64_t p = 0; p < nprob; ++p) B->hprobs[(size_t)p].n_free = nfree[(size_t)p];
    sync(ctx);
    sfem_csr_destroy(B->K);
    B->K = nullptr;
    sfem_bc_destroy(B->bc);
    B->bc = nullptr;
    sfem_mesh_destroy(B->mesh);
    B->mesh = nullptr;
    return B.release();
}

sfem_batch* batch_create(sfem_ctx* ctx, int64_t nprob, int ndim, int n_dof, const double* node_list,
                         const int64_t* node_offsets, const int64_t* ien, int nen, const int64_t* elem_offsets,
                         const double* young, const double* nu, const double* f, const uint8_t* fixed,
                         const double* q_d) {
    if (nprob <= 0 || !node_list || !node_offsets || !ien || !elem_offsets || !young || !nu || !fixed)
        fail(SFEM_ERR_ARGUMENT, "batch_create: NULL array or empty batch");
    if (n_dof != ndim || (ndim != 2 && ndim != 3) || nen != (1 << ndim))
        fail(SFEM_ERR_UNSUPPORTED, "batch_create: Q4 (2D) or Hex8 (3D) vector problems only");
    if (node_offsets[0] != 0 || elem_offsets[0] != 0)
        fail(SFEM_ERR_ARGUMENT, "batch_create: offsets must start at 0");
    for (int64_t p = 0; p < nprob; ++p)
        if (node_offsets[p + 1] <= node_offsets[p] || elem_offsets[p + 1] <= elem_offsets[p])
            fail(SFEM_ERR_ARGUMENT, "batch_create: every problem needs nodes and elements (problem " +
                                        std::to_string(p) + ")");
    const int64_t N = node_offsets[nprob], E = elem_offsets[nprob];
    std::vector<int64_t> gien((size_t)(E * nen)), gid((size_t)(N * n_dof));
    for (int64_t p = 0; p < nprob; ++p)
        for (int64_t e = elem_offsets[p]; e < elem_offsets[p + 1]; ++e)
            for (int a = 0; a < nen; ++a) {
                const int64_t v = ien[(int64_t)a * E + e];
                if (v < 1 || v > node_offsets[p + 1] - node_offsets[p])
                    fail(SFEM_ERR_BOUNDS, "batch_create: IEN entry outside its problem's nodes (problem " +
                                              std::to_string(p) + ")");
                gien[(size_t)((int64_t)a * E + e)] = v + node_offsets[p];
            }
    for (int64_t m = 0; m < N; ++m)
        for (int l = 0; l < n_dof; ++l) gid[(size_t)((int64_t)l * N + m)] = (int64_t)n_dof * m + l + 1;
    sfem_mesh* mesh = nullptr;
    int s = sfem_mesh_create(ctx, ndim, SFEM_Q1, n_dof, node_list, N, gien.data(), E, nen, E, gid.data(), N, young, E,
                             0.3, &mesh);
    if (s) fail(s, ctx->last_error);
    try {
        mesh->nu_e.reset(ctx, (size_t)E);
        h2d(ctx, mesh->nu_e.get(), nu, sizeof(double) * E);
    } catch (...) {
        sfem_mesh_destroy(mesh);
        throw;
    }
    sfem_bc* bc = nullptr;
    s = sfem_bc_create(ctx, N * n_dof, f, fixed, q_d, &bc);
    if (s) {
        sfem_mesh_destroy(mesh);
        fail(s, ctx->last_error);
    }
    std::vector<int64_t> noff(node_offsets, node_offsets + nprob + 1), nfree((size_t)nprob, 0);
    for (int64_t p = 0; p < nprob; ++p)
        for (int64_t d = node_offsets[p] * n_dof; d < node_offsets[p + 1] * n_dof; ++d)
            nfree[(size_t)p] += fixed[d] ? 0 : 1;
    return batch_from_device(ctx, nprob, mesh, bc, noff, nfree);
}

int64_t batch_device_bytes(const sfem_batch* B, int precision) {
    const int64_t b2 = (int64_t)B->bs * B->bs;
    const int64_t vb = (int64_t)prec_vec_bytes(precision);
    return B->sell_blocks * (4 + b2 * 14) + B->nslices * 12 + B->npad * (8 * 3 + 4 + 5 * vb + (vb == 4 ? 4 : 0)) +
           B->nslices * 64 * b2 * 12 + (int64_t)B->pad_of.size() * 4 + B->n * 9;
}

}  // namespace sfem

extern "C" {

int sfem_batch_create(sfem_ctx* ctx, int64_t nprob, int ndim, int n_dof, const double* node_list,
                      const int64_t* node_offsets, const int64_t* ien, int nen, const int64_t* elem_offsets,
                      const double* young, const double* nu, const double* f, const uint8_t* fixed,
                      const double* q_d, sfem_batch** out) {
    if (!ctx) return SFEM_ERR_ARGUMENT;
    if (!out) { ctx->last_error = "batch_create: NULL out"; return SFEM_ERR_ARGUMENT; }
    *out = nullptr;
    sfem_batch* B = nullptr;
    const int st = guard(ctx, [&] {
        B = batch_create(ctx, nprob, ndim, n_dof, node_list, node_offsets, ien, nen, elem_offsets, young, nu, f,
                         fixed, q_d);
    });
    if (st) return st;
    ctx_retain(ctx);
    *out = B;
    return SFEM_OK;
}

int sfem_batch_info(const sfem_batch* B, int64_t* n_total, int64_t* n_padded, int64_t* slices, double* assemble_ms,
                    double* eliminate_ms) {
    if (!B) return SFEM_ERR_ARGUMENT;
    if (n_total) *n_total = B->n;
    if (n_padded) *n_padded = B->npad;
    if (slices) *slices = B->nslices;
    if (assemble_ms) *assemble_ms = B->t_assemble_ms;
    if (eliminate_ms) *eliminate_ms = B->t_eliminate_ms;
    return SFEM_OK;
}

int sfem_batch_solve(sfem_ctx* ctx, sfem_batch* B, const sfem_solve_opts* opts, int item_slices,
                     int blocks_per_cu, sfem_batch_problem_stats* per, sfem_batch_stats* stats) {
    if (!ctx) return SFEM_ERR_ARGUMENT;
    if (!B) { ctx->last_error = "batch_solve: NULL batch"; return SFEM_ERR_ARGUMENT; }
    sfem_solve_opts o;
    sfem_solve_opts_default(&o);
    if (opts) o = *opts;
    return guard(ctx, [&] {
        int64_t nl = 0;
        const double ms = batch_run(ctx, B, o, item_slices, blocks_per_cu, &nl);
        std::vector<ProbState> hst((size_t)B->nprob);
        d2h(ctx, hst.data(), B->st.get(), sizeof(ProbState) * B->nprob);
        int64_t bad = 0, max_it = 0, sum_it = 0;
        for (int64_t p = 0; p < B->nprob; ++p) {
            const ProbState& S = hst[(size_t)p];
            if (per) {
                per[p].iterations = S.iters;
                per[p].fp64_updates = S.updates;
                per[p].rel_residual = S.bb > 0 ? std::sqrt(S.rr_true / S.bb) : 0.0;
                per[p].n_free = B->hprobs[(size_t)p].n_free;
                per[p].stop_reason = S.done == 0 ? 4 : S.done;
                per[p].floor_residual = S.bb > 0 ? std::sqrt(S.floor_rr / 16.0 / S.bb) : 0.0;
            }
            max_it = std::max<int64_t>(max_it, S.iters);
            sum_it += S.iters;
            if (S.done != 1) ++bad;
        }
        if (stats) {
            stats->solve_ms = ms;
            stats->launches = nl;
            stats->max_iterations = max_it;
            stats->sum_iterations = sum_it;
            stats->not_converged = bad;
            stats->grid = table_grid(ctx, o.precision, blocks_per_cu);
            stats->device_bytes = batch_device_bytes(B, o.precision);
            stats->barrier_grouped = ctx->bar_last_grouped ? 1 : 0;
        }
        if (bad) fail(SFEM_ERR_NOT_CONVERGED, "batch_solve: " + std::to_string(bad) + " problems did not converge");
    });
}

int sfem_batch_solution(sfem_ctx* ctx, const sfem_batch* B, double* q) {
    if (!ctx) return SFEM_ERR_ARGUMENT;
    if (!B || !q) { ctx->last_error = "batch_solution: NULL argument"; return SFEM_ERR_ARGUMENT; }
    return guard(ctx, [&] { batch_solution(ctx, B, q); });
}

int sfem_batch_max_blocks_per_cu(sfem_ctx* ctx, int precision, int* blocks) {
    if (!ctx) return SFEM_ERR_ARGUMENT;
    if (!blocks) { ctx->last_error = "NULL blocks"; return SFEM_ERR_ARGUMENT; }
    return guard(ctx, [&] { *blocks = table_max_blocks_per_cu(precision); });
}

void sfem_batch_destroy(sfem_batch* B) {
    if (!B) return;
    sfem_ctx* ctx = B->ctx;
    delete B;
    ctx_release(ctx);
}

}  // extern "C"
