// Device side of the smoothed-aggregation preconditioner (amg.hpp): the
// hierarchy's arrays in HBM, the numeric phase that follows the matrix
// values (fine values from the 2x2-block matrix, diagonal inverses, a power
// iteration for lambda_max(D^-1 A), the smoothed prolongator, W = A P and
// A_c = P^T W, the coarsest inverse), and the FP32 V-cycle.
//
// Every kernel sums in the pattern's order, so runs are reproducible.  The
// V-cycle kernels return at once when the solve has stopped (st->done), like
// the flexible CG's own kernels.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <new>
#include <type_traits>
#include <vector>

#include "amg.hpp"
#include "fem.hpp"
#include "rows.hpp"

namespace nbx {

// Block sliced ELL for the V-cycle's FP32 products: block rows of R
// scalar rows (one node or aggregate), blocks of R x C values, 64 block
// rows per slice; block k of block row I at slot slice_ptr[I/64] + 64 k +
// I%64, its value (r, c) in plane r C + c (val[(r C + c) slots + slot]), so
// a wavefront's loads of one block position are coalesced.  The levels'
// operators (3 x 3 blocks below the finest level), P (2 x 3 on the finest
// level, 3 x 3 below) and P^T (3 x 2, 3 x 3) take this form: all R rows of
// a block row share one pattern of C-column groups.
struct BellDev {
    uint32_t rows = 0;
    int lanes = 1;             // lanes per block row in the V-cycle's products
    uint32_t wmax = 0;         // blocks of the longest row
    uint32_t width = 0;        // the width of every slice where they are alike, or 0
    size_t slots = 0;
    uint32_t* slice_ptr = nullptr;
    uint16_t* len = nullptr;
    uint32_t* bcol = nullptr;
    float* val = nullptr;
};

struct AmgDevLevel {
    uint32_t n = 0, nc = 0, bs = 2;
    size_t a_nnz = 0, p_nnz = 0, w_nnz = 0;
    uint32_t *a_ptr = nullptr, *a_col = nullptr;
    double* a64 = nullptr;
    double* dinv64 = nullptr;
    float* dinv32 = nullptr;
    double lmax = 0.0;
    double* t = nullptr;
    uint32_t* agg = nullptr;   // [n / bs] each node's aggregate, or AMG_NONE
    uint32_t *p_ptr = nullptr, *p_col = nullptr;
    double* p64 = nullptr;
    uint32_t *w_ptr = nullptr, *w_col = nullptr;
    double* w64 = nullptr;
    uint32_t *pt_ptr = nullptr, *pt_row = nullptr, *pt_pos = nullptr;
    BellDev ab, pb, tb;        // the operator (below the finest level), P, P^T
    // tiles for the level's smoothing in two launches, or none; the cycle then
    // leaves its correction in d0 instead of x
    Tiles tiles;
    float* out() const { return tiles.n ? d0 : x; }
    // V-cycle vectors: right-hand side and solution of this level (the
    // finest level's come from the caller), residual, two directions
    float *b = nullptr, *x = nullptr, *r = nullptr, *d0 = nullptr, *d1 = nullptr;
    // Chebyshev smoothing on [lambda/30, 1.1 lambda]
    float inv_theta = 0.f, c1[AMG_MAX_DEGREE] = {}, c2[AMG_MAX_DEGREE] = {};
    int degree = AMG_DEGREE;   // smoothing steps before and after (amg_level_degree)
};

struct AmgDev {
    std::vector<AmgDevLevel> lv;
    float* cinv = nullptr;          // coarsest inverse, n x n
    double* ones = nullptr;         // [finest n + 2] the flexible CG's unit scaling
    double* pow_x = nullptr;        // power iteration: [finest n + 2] x, y
    double* pow_y = nullptr;
    double* scal = nullptr;         // [2 levels] 1 / norm and norm of the power iteration
    double* partials = nullptr;     // [MAX_GRID] reduction partials
    double* dense = nullptr;        // the coarsest matrix, its inverse, I - A A^-1, n x n each,
                                    // and n flags
    size_t bytes = 0;
    // more than one level: the finest is smoothed on the matrix's fp16
    // scaled copy, in scaled variables, and its P values are stored as
    // D^1/2 P (FP32)
    bool scaled16 = false;
    size_t bottom = 0;              // the level k_amg_bottom starts from, or 0
    // what the hierarchy was built from besides the mesh: k_block_nzbits of K
    // at that time (null until the build is complete), and a word for the
    // comparison with the current ones
    uint8_t* nzbits = nullptr;
    uint32_t* differ = nullptr;
};

namespace {

template <class T, class Al>
int up(T** d, const std::vector<T, Al>& h, size_t& bytes) {
    const size_t nb = (h.size() + 1) * sizeof(T);
    NBX_HIP(hipMalloc(d, nb));
    bytes += nb;
    if (!h.empty()) NBX_HIP(hipMemcpy(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
    return NBX_OK;
}
template <class T>
int alloc(T** d, size_t n, size_t& bytes) {
    const size_t nb = (n + 2) * sizeof(T);
    NBX_HIP(hipMalloc(d, nb));
    bytes += nb;
    return NBX_OK;
}

// ---- numeric phase ----------------------------------------------------------

// the slice holding slot sl of a sliced layout: the last s < slices with
// slice_ptr[s] <= sl
__device__ __forceinline__ uint32_t slice_of(const uint32_t* __restrict__ slice_ptr,
                                             uint32_t slices, size_t sl) {
    uint32_t lo = 0, hi = slices;
    while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (slice_ptr[mid] <= sl) lo = mid; else hi = mid;
    }
    return lo;
}

// The finest level's CSR values from the 2x2-block layout, one thread per
// slot: block k of node v holds entries (i, j) of rows 2v + i at positions
// a_ptr[2v + i] + 2k + j (the CSR the host built from the same layout)
__global__ __launch_bounds__(BLOCK) void k_amg_fine_vals(Sell2 K, const uint32_t* __restrict__ a_ptr,
                                                         double* __restrict__ a) {
    const size_t sl = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    if (sl >= K.n_blocks) return;
    const uint32_t s = slice_of(K.slice_ptr, K.n_slices, sl);
    const size_t off = sl - K.slice_ptr[s];
    const uint32_t v = s * SLICE + (uint32_t)(off % SLICE);
    const uint32_t k = (uint32_t)(off / SLICE);
    if (v >= K.n_nodes || k >= K.rowlen[v]) return;
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            a[a_ptr[2 * (size_t)v + i] + 2 * (size_t)k + j] = K.val[ent(K.n_blocks, sl, i, j)];
}
// bit 2 i + j: entry (i, j) of slot sl's block is nonzero
__device__ __forceinline__ uint8_t block_nzbits(const Sell2& K, size_t sl) {
    uint32_t b = 0;
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            if (K.val[ent(K.n_blocks, sl, i, j)] != 0.0) b |= 1u << (2 * i + j);
    return (uint8_t)b;
}
__global__ __launch_bounds__(BLOCK) void k_block_nzbits(Sell2 K, uint8_t* __restrict__ bits) {
    const size_t sl = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    if (sl < K.n_blocks) bits[sl] = block_nzbits(K, sl);
}
// sets *differ when a slot's nonzero entries are others than bits says; one
// pass over K's blocks, bound by their bytes (7.5 MB at 256x128)
__global__ __launch_bounds__(BLOCK) void k_block_nzbits_differ(Sell2 K,
                                                               const uint8_t* __restrict__ bits,
                                                               uint32_t* differ) {
    const size_t sl = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    if (sl < K.n_blocks && block_nzbits(K, sl) != bits[sl]) *differ = 1;
}

// D^-1 (0 where the diagonal is not positive: an unknown with no coarse or
// smoothing part)
__global__ __launch_bounds__(BLOCK) void k_amg_dinv(const uint32_t* __restrict__ ptr,
                                                    const uint32_t* __restrict__ col,
                                                    const double* __restrict__ a,
                                                    double* __restrict__ d64,
                                                    float* __restrict__ d32, uint32_t n) {
    const uint32_t i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    double d = 0.0;
    for (uint32_t e = ptr[i]; e < ptr[i + 1]; ++e)
        if (col[e] == i) d = a[e];
    const double v = d > 0.0 ? 1.0 / d : 0.0;
    d64[i] = v;
    d32[i] = (float)v;
}

// power iteration on D^-1 A: x_0 = +-1 from a hash of the index (amg_sign),
// normalised by the first step
__global__ __launch_bounds__(BLOCK) void k_amg_pow_init(double* __restrict__ x, uint32_t n) {
    const uint32_t i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    uint32_t h = i * 2654435761u;
    h ^= h >> 15;
    h *= 2246822519u;
    h ^= h >> 13;
    x[i] = (h & 1u) ? 1.0 : -1.0;
}
// y = D^-1 A (x * s) and the y.y partials.  s = 1 / ||x||: from the step
// before's partials (prev), which every workgroup sums itself; on levels of
// more than ALL_PARTS workgroups from *scale, left by k_amg_pow_fin; or, on the
// first step, s0.  Eight lanes per row, rows strided over the grid (at most
// MAX_GRID workgroups, one partial each).  A step of a small level is a launch
// and a chain of loads, so the summing kernel between two steps cost as much
// again (15 of 2.3 us and their launches a level, of 4.5 us steps).
constexpr int POW_LANES = 8;
constexpr int POW_STEPS = 15;
__global__ __launch_bounds__(BLOCK) void k_amg_pow_step(
    const uint32_t* __restrict__ ptr, const uint32_t* __restrict__ col,
    const double* __restrict__ a, const double* __restrict__ dinv, const double* __restrict__ x,
    double* __restrict__ y, const double* __restrict__ prev, const double* __restrict__ scale,
    double s0, double* __restrict__ partials, uint32_t n) {
    double sc = s0;
    if (prev) {
        __shared__ double sums[1][ALL_PARTS / WAVE];
        double tot[1];
        AllSum<1> all;
        all.load(prev, gridDim.x);
        all.total(gridDim.x, tot, sums);
        const double nr = sqrt(tot[0]);
        sc = nr > 0.0 ? 1.0 / nr : 0.0;
    } else if (scale) {
        sc = *scale;
    }
    double acc[1] = {0.0};
    const size_t gid = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t lane = (uint32_t)(gid % POW_LANES);
    const size_t stride = (size_t)gridDim.x * BLOCK / POW_LANES;
    const size_t rows = ((size_t)n + stride - 1) / stride * stride;   // every group runs alike
    for (size_t r = gid / POW_LANES; r < rows; r += stride) {
        const bool valid = r < n;
        double s = 0.0;
        if (valid)
            for (uint32_t e = ptr[r] + lane; e < ptr[r + 1]; e += POW_LANES) s += a[e] * x[col[e]];
#pragma unroll
        for (int off = POW_LANES / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, POW_LANES);
        if (valid && lane == 0) {
            const double v = dinv[r] * (s * sc);
            y[r] = v;
            acc[0] += v * v;
        }
    }
    __shared__ double red[1][BLOCK / WAVE];
    block_sum<1>(acc, red);
    put_partials<1>(acc, partials);
}
// scal[0] = 1 / sqrt(sum), scal[1] = sqrt(sum)
__global__ __launch_bounds__(FIN) void k_amg_pow_fin(const double* partials, unsigned np,
                                                     double* scal) {
    double tot[1];
    fin_sum<1>(partials, np, tot);
    if (threadIdx.x == 0) {
        const double nr = sqrt(tot[0]);
        scal[0] = nr > 0.0 ? 1.0 / nr : 0.0;
        scal[1] = nr;
    }
}

// ---- the coarsest level's inverse --------------------------------------------
// A^-1 of the coarsest level (at most AMG_COARSEST unknowns) by symmetric
// sweeps (Goodnight 1979): sweeping k turns a_kk into -1 / a_kk, a_ik into
// a_ik / a_kk and a_ij into a_ij - a_ik a_kj / a_kk; all swept, A is -A^-1.
// The pivots are the Cholesky factor's, and an unknown whose pivot is not
// above 1e-13 of the largest diagonal entry is dropped (zero row and column).
// One workgroup holds the matrix in registers, the lower half of its 32 x 32
// blocks; a step passes column k through LDS and costs one barrier.  Bound by
// its n steps of LDS reads, a division and a barrier: 142 us at 162 unknowns
// (190 with all entries).  The sweeps' error is up to 84 times that of a
// Cholesky factor's inverse in FP64 (3.0 on average over the coarsest levels of
// 60 systems of 200 to 200,000 unknowns; with void elements, condition numbers
// of 1e11, 4e-6 where FP32 rounds to 2e-8), so one step of Newton's iteration
// X + X (I - A X) follows, its residual in doubled precision, a workgroup a row
// (9.6 + 7.9 us at 162 unknowns): then the stored inverse is A^-1 rounded to FP32
// in all 60, which the Cholesky inverse was in 53.
constexpr int SWEEP_SIDE = 32, SWEEP_TB = SWEEP_SIDE * SWEEP_SIDE;
constexpr int SWEEP_NB = (AMG_COARSEST + SWEEP_SIDE - 1) / SWEEP_SIDE;

// The dense matrix from its CSR rows, a wavefront per row
__global__ __launch_bounds__(WAVE) void k_dense_rows(const uint32_t* __restrict__ ptr,
                                                     const uint32_t* __restrict__ col,
                                                     const double* __restrict__ a,
                                                     double* __restrict__ out, uint32_t n) {
    __shared__ double row[AMG_COARSEST];
    const uint32_t i = blockIdx.x;
    for (uint32_t j = threadIdx.x; j < n; j += WAVE) row[j] = 0.0;
    __syncthreads();
    for (uint32_t e = ptr[i] + threadIdx.x; e < ptr[i + 1]; e += WAVE) row[col[e]] = a[e];
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < n; j += WAVE) out[(size_t)i * n + j] = row[j];
}

// entry (i, j) of A symmetrised (P^T A P rounds slightly unsymmetrically)
__device__ __forceinline__ double dense_sym(const double* __restrict__ a, uint32_t n, uint32_t i,
                                            uint32_t j) {
    return i == j ? a[(size_t)i * n + i] : 0.5 * (a[(size_t)i * n + j] + a[(size_t)j * n + i]);
}

// inv = A^-1 by sweeps.  Thread (tx, ty) holds the entries (ty + 32 p, tx + 32 q)
// with q <= p; column k is those of the column from row block k / 32 on and
// those of row k before it.
template <int NB>
__global__ __launch_bounds__(SWEEP_TB) void k_dense_sweep(const double* __restrict__ a,
                                                          double* __restrict__ inv, uint32_t n) {
    __shared__ double colk[2][NB * SWEEP_SIDE], big[SWEEP_TB / WAVE];
    const uint32_t tx = threadIdx.x % SWEEP_SIDE, ty = threadIdx.x / SWEEP_SIDE;
    double v[NB][NB], dmax = 0.0;   // (the entries q > p are never used)
#pragma unroll
    for (int p = 0; p < NB; ++p)
#pragma unroll
        for (int q = 0; q <= p; ++q) {
            const uint32_t i = ty + p * SWEEP_SIDE, j = tx + q * SWEEP_SIDE;
            v[p][q] = 0.0;
            if (i < n && j < n) v[p][q] = dense_sym(a, n, i, j);
            if (i == j) dmax = fmax(dmax, v[p][q]);
        }
    for (int off = WAVE / 2; off > 0; off >>= 1) dmax = fmax(dmax, __shfl_xor(dmax, off));
    if (threadIdx.x % WAVE == 0) big[threadIdx.x / WAVE] = dmax;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < SWEEP_TB / WAVE; ++w) dmax = fmax(dmax, big[w]);
#pragma unroll
    for (int kq = 0; kq < NB; ++kq)
        for (uint32_t kt = 0; kt < SWEEP_SIDE; ++kt) {
            const uint32_t k = kq * SWEEP_SIDE + kt;
            if (k >= n) break;
            double* const ck = colk[k & 1];
            if (tx == kt)
#pragma unroll
                for (int p = kq; p < NB; ++p) ck[ty + p * SWEEP_SIDE] = v[p][kq];
            if (ty == kt)
#pragma unroll
                for (int q = 0; q < kq; ++q) ck[tx + q * SWEEP_SIDE] = v[kq][q];
            __syncthreads();
            const double piv = ck[k];
            const bool drop = !(piv > 1e-13 * dmax);
            const double d = drop ? 0.0 : 1.0 / piv;
            double cj[NB];
#pragma unroll
            for (int q = 0; q < NB; ++q) cj[q] = ck[tx + q * SWEEP_SIDE];
#pragma unroll
            for (int p = 0; p < NB; ++p) {
                const double f = ck[ty + p * SWEEP_SIDE] * d;
#pragma unroll
                for (int q = 0; q <= p; ++q) v[p][q] = fma(-f, cj[q], v[p][q]);
                if (p >= kq && tx == kt) v[p][kq] = ty + p * SWEEP_SIDE == k ? -d : f;   // column k
            }
            if (ty == kt)   // row k
#pragma unroll
                for (int q = 0; q <= kq; ++q)
                    if (tx + q * SWEEP_SIDE != k) v[kq][q] = cj[q] * d;
        }
#pragma unroll
    for (int p = 0; p < NB; ++p)
#pragma unroll
        for (int q = 0; q <= p; ++q) {
            const uint32_t i = ty + p * SWEEP_SIDE, j = tx + q * SWEEP_SIDE;
            // (of a diagonal block's two entries that rounding may leave
            // different, the lower one for both)
            if (i < n && j <= i)
                inv[(size_t)i * n + j] = inv[(size_t)j * n + i] = -v[p][q];
        }
}

// R = I - A X by compensated dot products, a workgroup per row, every column by
// REFINE_PARTS threads with REFINE_AHEAD loads under way each (bound by the loads'
// latency: one thread a column 18 and 16 us for the two kernels, four 14.7 and 11.6); far[i]: the row is not small enough for a step of Newton's iteration
// (rows of dropped unknowns, whose X is zero, do not count)
constexpr uint32_t REFINE_PARTS = 4, REFINE_AHEAD = 14;
static_assert(AMG_COARSEST + REFINE_PARTS * REFINE_AHEAD <= BLOCK, "row[] is zero past n");
// f(a row's entry p, column j's) for the p of a part, then for entries of 0
template <class F>
__device__ __forceinline__ void refine_dot(const double* row, const double* __restrict__ m,
                                           uint32_t n, uint32_t j, uint32_t part, F&& f) {
    for (uint32_t p0 = part; p0 < n; p0 += REFINE_PARTS * REFINE_AHEAD) {
        double v[REFINE_AHEAD];
#pragma unroll
        for (uint32_t u = 0; u < REFINE_AHEAD; ++u) {
            const uint32_t p = p0 + u * REFINE_PARTS;
            v[u] = p < n ? m[(size_t)p * n + j] : 0.0;
        }
#pragma unroll
        for (uint32_t u = 0; u < REFINE_AHEAD; ++u) f(row[p0 + u * REFINE_PARTS], v[u]);
    }
}
__global__ __launch_bounds__(REFINE_PARTS * BLOCK) void k_dense_residual(
    const double* __restrict__ a, const double* __restrict__ x, double* __restrict__ r,
    uint32_t* __restrict__ far, uint32_t n) {
    __shared__ double row[BLOCK], ps[REFINE_PARTS][BLOCK], pc[REFINE_PARTS][BLOCK],
        red[BLOCK / WAVE];
    const uint32_t i = blockIdx.x, j = threadIdx.x % BLOCK, part = threadIdx.x / BLOCK;
    if (part == 0) row[j] = j < n ? -dense_sym(a, n, i, j) : 0.0;
    __syncthreads();
    if (j < n) {
        double s = part == 0 && i == j ? 1.0 : 0.0, c = 0.0;
        refine_dot(row, x, n, j, part, [&](double av, double xv) { dot2_add(av, xv, s, c); });
        ps[part][j] = s;
        pc[part][j] = c;
    }
    __syncthreads();
    double e = 0.0;
    if (part == 0 && j < n) {
        double s = ps[0][j], c = pc[0][j];
        for (uint32_t q = 1; q < REFINE_PARTS; ++q) {
            double t, d;
            two_sum64(s, ps[q][j], t, d);
            s = t;
            c += d + pc[q][j];
        }
        r[(size_t)i * n + j] = s + c;
        e = fabs(s + c);
    }
    e = wave_sum(e);
    if (part == 0 && j % WAVE == 0) red[j / WAVE] = e;
    __syncthreads();
    if (threadIdx.x == 0) {
        e = 0.0;
        for (int w = 0; w < BLOCK / WAVE; ++w) e += red[w];
        far[i] = x[(size_t)i * n + i] != 0.0 && !(e < 0.1);
    }
}
// inv = X + X R in FP32 (X alone where a row of R is far from 0), likewise
__global__ __launch_bounds__(REFINE_PARTS * BLOCK) void k_dense_refine(
    const double* __restrict__ x, const double* __restrict__ r, const uint32_t* __restrict__ far,
    float* __restrict__ inv, uint32_t n) {
    __shared__ double row[BLOCK], ps[REFINE_PARTS][BLOCK];
    const uint32_t i = blockIdx.x, j = threadIdx.x % BLOCK, part = threadIdx.x / BLOCK;
    if (part == 0) row[j] = j < n ? x[(size_t)i * n + j] : 0.0;
    const bool skip = __syncthreads_or(part == 0 && j < n && far[j]);
    if (j <= i) {
        double s = 0.0;
        if (!skip) refine_dot(row, r, n, j, part, [&](double xv, double rv) { s += xv * rv; });
        ps[part][j] = s;
    }
    __syncthreads();
    if (part != 0 || j > i) return;
    double s = ps[0][j];
    for (uint32_t q = 1; q < REFINE_PARTS; ++q) s += ps[q][j];
    inv[(size_t)i * n + j] = inv[(size_t)j * n + i] = (float)(row[j] + s);
}
static_assert(AMG_COARSEST <= BLOCK, "a thread per column");

// P = T - omega D^-1 A T: SMOOTH_SLOTS threads per node, each taking every
// SMOOTH_SLOTS-th aggregate column group of the node's P rows (its R rows
// share one A and one P pattern; a group is the three columns of one
// aggregate) and summing, in entry order, each row's A entries whose column
// node belongs to that aggregate
constexpr int SMOOTH_SLOTS = 8;
template <int R>
__global__ __launch_bounds__(BLOCK) void k_amg_smooth_p(
    const uint32_t* __restrict__ a_ptr, const uint32_t* __restrict__ a_col,
    const double* __restrict__ a, const double* __restrict__ dinv, const double* __restrict__ t,
    const uint32_t* __restrict__ agg, const uint32_t* __restrict__ p_ptr,
    const uint32_t* __restrict__ p_col, double* __restrict__ p, const double* __restrict__ lmax,
    uint32_t nodes) {
    const double omega = 4.0 / (3.0 * *lmax);
    const size_t tid = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t I = (uint32_t)(tid / SMOOTH_SLOTS);
    if (I >= nodes) return;
    const uint32_t i0 = R * I;
    const uint32_t ng = (p_ptr[i0 + 1] - p_ptr[i0]) / 3;
    double od[R];
    uint32_t ao[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        od[r] = omega * dinv[i0 + r];
        ao[r] = a_ptr[i0 + r] - a_ptr[i0];   // row r's entry e + ao[r] pairs with e
    }
    for (uint32_t gi = (uint32_t)(tid % SMOOTH_SLOTS); gi < ng; gi += SMOOTH_SLOTS) {
        const uint32_t qo = 3 * gi;          // the group's offset in each row
        const uint32_t ga = p_col[p_ptr[i0] + qo] / 3;   // its aggregate
        const bool own = agg[I] == ga;
        double acc[R][3];
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int m = 0; m < 3; ++m) acc[r][m] = 0.0;
            if (own)
#pragma unroll
                for (int m = 0; m < 3; ++m) acc[r][m] += t[3 * (size_t)(i0 + r) + m];
        }
        for (uint32_t e = a_ptr[i0]; e < a_ptr[i0 + 1]; ++e) {
            if (agg[a_col[e] / R] != ga) continue;
            const uint32_t j = a_col[e];
            double tj[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) tj[m] = t[3 * (size_t)j + m];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const double coef = od[r] * a[e + ao[r]];
#pragma unroll
                for (int m = 0; m < 3; ++m) acc[r][m] -= coef * tj[m];
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int m = 0; m < 3; ++m) p[p_ptr[i0 + r] + qo + m] = acc[r][m];
    }
}

// Block values from a CSR whose R rows per block row share one pattern of
// C-column groups: block k of block row I holds the rows' k-th groups
// (scaled by 1 / dis of the row when dis is given: D^1/2 P on the finest
// level in the scaled variables).
template <int R, int C>
__global__ __launch_bounds__(BLOCK) void k_bell_fill(BellDev B, const uint32_t* __restrict__ ptr,
                                                     const double* __restrict__ v,
                                                     const double* __restrict__ dis) {
    const uint32_t I = blockIdx.x * BLOCK + threadIdx.x;
    if (I >= B.rows) return;
    const size_t base = (size_t)B.slice_ptr[I >> 6] + (I & 63);
    const int len = B.len[I];
    for (int r = 0; r < R; ++r) {
        const size_t row = (size_t)R * I + r;
        const uint32_t off = ptr[row];
        const double sc = dis ? 1.0 / dis[row] : 1.0;
        for (int k = 0; k < len; ++k)
            for (int c = 0; c < C; ++c)
                B.val[(size_t)(r * C + c) * B.slots + base + (size_t)k * SLICE] =
                    (float)(v[off + (size_t)C * k + c] * sc);
    }
}
// P^T's blocks from P's values through the P^T lists: block k of aggregate
// a is node J = bcol; its value (c, r) is P(R J + r, 3 a + c), the
// (R k + r)-th entry of column 3 a + c's list.  One thread per slot of the
// layout (padding slots return).
template <int R>
__global__ __launch_bounds__(BLOCK) void k_bell_fill_t(BellDev B, uint32_t slices,
                                                       const uint32_t* __restrict__ pt_ptr,
                                                       const uint32_t* __restrict__ pt_pos,
                                                       const double* __restrict__ p,
                                                       const double* __restrict__ dis) {
    const size_t sl = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    if (sl >= B.slots) return;
    // the slice holding slot sl: the last s with slice_ptr[s] <= sl
    uint32_t lo = 0, hi = slices;
    while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (B.slice_ptr[mid] <= sl) lo = mid; else hi = mid;
    }
    const size_t off = sl - B.slice_ptr[lo];
    const uint32_t a = lo * SLICE + (uint32_t)(off % SLICE);
    const uint32_t k = (uint32_t)(off / SLICE);
    if (a >= B.rows || k >= B.len[a]) return;
    const uint32_t J = B.bcol[sl];
    for (int c = 0; c < 3; ++c)
        for (int r = 0; r < R; ++r) {
            const uint32_t q = pt_pos[pt_ptr[3 * (size_t)a + c] + (size_t)R * k + r];
            const double sc = dis ? 1.0 / dis[(size_t)R * J + r] : 1.0;
            B.val[(size_t)(c * R + r) * B.slots + sl] = (float)(p[q] * sc);
        }
}

// W = A P and A_c = P^T W, one thread per output block.  The host built
// every pattern in groups: A's rows of one node (R rows: R = 2 on the finest
// level, 3 below) share its pattern of R-column groups, P's, W's and A_c's
// rows share patterns of 3-column groups (aggregates), all ascending; W's
// row holds every aggregate of every P row its A row reaches, A_c's row
// every aggregate of every W row of a node holding it.  An output block sums
// its block products in a fixed order (the neighbour blocks, or the nodes
// holding the aggregate, ascending): no atomics, and runs are reproducible.

// the block row whose blocks start at or before block t: the last i with
// ptr[stride i] <= per t (ptr ascending, rows in [0, rows))
__device__ __forceinline__ uint32_t block_row(const uint32_t* __restrict__ ptr, uint32_t stride,
                                              size_t per, size_t t, uint32_t rows) {
    uint32_t lo = 0, hi = rows;   // invariant: ptr[stride lo] <= per t < ptr[stride hi]
    while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if ((size_t)ptr[(size_t)stride * mid] <= per * t) lo = mid; else hi = mid;
    }
    return lo;
}
// position of group b3 (a multiple of 3) in the ascending groups
// col[b], col[b + 3], ..., col[b + 3 (len - 1)], or len
__device__ __forceinline__ uint32_t find_group(const uint32_t* __restrict__ col, uint32_t b,
                                               uint32_t len, uint32_t b3) {
    uint32_t lo = 0, hi = len;
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (col[b + 3 * mid] < b3) lo = mid + 1; else hi = mid;
    }
    return lo < len && col[b + 3 * lo] == b3 ? lo : len;
}

// W(I, b) = sum over neighbour blocks J of A(I, J) P(J, b).  LANES
// consecutive lanes take an output block (each sums every LANES-th
// neighbour, then a butterfly adds the lanes' sums): more lanes on the small
// levels, whose few output blocks each sum many products.
template <int R, int LANES>
__global__ __launch_bounds__(BLOCK) void k_amg_w(const uint32_t* __restrict__ a_ptr,
                                                 const uint32_t* __restrict__ a_col,
                                                 const double* __restrict__ a,
                                                 const uint32_t* __restrict__ p_ptr,
                                                 const uint32_t* __restrict__ p_col,
                                                 const double* __restrict__ p,
                                                 const uint32_t* __restrict__ w_ptr,
                                                 const uint32_t* __restrict__ w_col,
                                                 double* __restrict__ w, uint32_t nodes,
                                                 size_t blocks) {
    const size_t tid = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    const size_t t = tid / LANES;
    const uint32_t lane = (uint32_t)(tid % LANES);
    if (t >= blocks) return;   // (a whole group: blocks end at a group boundary)
    const uint32_t I = block_row(w_ptr, R, 3 * R, t, nodes);
    const uint32_t j = (uint32_t)(t - w_ptr[(size_t)R * I] / (3 * R));
    const uint32_t b3 = w_col[w_ptr[(size_t)R * I] + 3 * j];
    uint32_t ar[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ar[r] = a_ptr[(size_t)R * I + r];
    const uint32_t al = (a_ptr[(size_t)R * I + 1] - ar[0]) / R;
    double acc[R][3] = {};
    for (uint32_t k = lane; k < al; k += LANES) {
        const uint32_t J = a_col[ar[0] + R * k] / R;
        const uint32_t p0 = p_ptr[(size_t)R * J];
        const uint32_t kk = find_group(p_col, p0, (p_ptr[(size_t)R * J + 1] - p0) / 3, b3);
        if (kk == (p_ptr[(size_t)R * J + 1] - p0) / 3) continue;
        double pk[R][3];
#pragma unroll
        for (int c = 0; c < R; ++c)
#pragma unroll
            for (int m = 0; m < 3; ++m) pk[c][m] = p[p_ptr[(size_t)R * J + c] + 3 * kk + m];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                double s = 0.0;
#pragma unroll
                for (int c = 0; c < R; ++c) s += a[ar[r] + R * k + c] * pk[c][m];
                acc[r][m] += s;
            }
    }
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int m = 0; m < 3; ++m) acc[r][m] += __shfl_xor(acc[r][m], off, LANES);
    if (lane != 0) return;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < 3; ++m) w[w_ptr[(size_t)R * I + r] + 3 * j + m] = acc[r][m];
}

// A_c(a, b) = sum over the nodes J holding aggregate a of P(J, a)^T W(J, b),
// LANES lanes per output block as in k_amg_w
template <int R, int LANES>
__global__ __launch_bounds__(BLOCK) void k_amg_galerkin(
    const uint32_t* __restrict__ pt_ptr, const uint32_t* __restrict__ pt_row,
    const uint32_t* __restrict__ pt_pos, const double* __restrict__ p,
    const uint32_t* __restrict__ w_ptr, const uint32_t* __restrict__ w_col,
    const double* __restrict__ w, const uint32_t* __restrict__ c_ptr,
    const uint32_t* __restrict__ c_col, double* __restrict__ ac, uint32_t aggs, size_t blocks) {
    const size_t tid = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    const size_t t = tid / LANES;
    const uint32_t lane = (uint32_t)(tid % LANES);
    if (t >= blocks) return;   // (a whole group)
    const uint32_t A = block_row(c_ptr, 3, 9, t, aggs);
    const uint32_t j = (uint32_t)(t - c_ptr[3 * (size_t)A] / 9);
    const uint32_t b3 = c_col[c_ptr[3 * (size_t)A] + 3 * j];
    uint32_t tr[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) tr[m] = pt_ptr[3 * (size_t)A + m];
    const uint32_t hl = (pt_ptr[3 * (size_t)A + 1] - tr[0]) / R;
    double acc[3][3] = {};
    for (uint32_t h = lane; h < hl; h += LANES) {
        const uint32_t J = pt_row[tr[0] + R * h] / R;
        const uint32_t w0 = w_ptr[(size_t)R * J];
        const uint32_t wl = (w_ptr[(size_t)R * J + 1] - w0) / 3;
        const uint32_t q = find_group(w_col, w0, wl, b3);
        if (q == wl) continue;
        double wq[R][3], ph[R][3];
#pragma unroll
        for (int c = 0; c < R; ++c)
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                wq[c][n] = w[w_ptr[(size_t)R * J + c] + 3 * q + n];
                ph[c][n] = p[pt_pos[tr[n] + R * h + c]];
            }
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                double s = 0.0;
#pragma unroll
                for (int c = 0; c < R; ++c) s += ph[c][m] * wq[c][n];
                acc[m][n] += s;
            }
    }
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1)
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int n = 0; n < 3; ++n) acc[m][n] += __shfl_xor(acc[m][n], off, LANES);
    if (lane != 0) return;
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int n = 0; n < 3; ++n) ac[c_ptr[3 * (size_t)A + m] + 3 * j + n] = acc[m][n];
}

// ---- V-cycle (FP32) ----------------------------------------------------------
// A group of LANES consecutive lanes takes a block row: each lane sums every
// LANES-th block, the group adds the lanes' sums by a butterfly, and the
// group's first lane does the row's update.  The order of the additions is
// fixed by the pattern, so runs are reproducible.

template <int LANES>
__device__ __forceinline__ float group_sum(float s) {
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, LANES);
    return s;
}

// ---- block sliced ELL products (FP32) ---------------------------------------

template <int R, int C>
struct Bell {
    uint32_t slots, width;
    const uint32_t* __restrict__ slice_ptr;
    const uint16_t* __restrict__ len;
    const uint32_t* __restrict__ bcol;
    const float* __restrict__ val;
};
template <int R, int C>
Bell<R, C> bell(const BellDev& B) {
    return Bell<R, C>{(uint32_t)B.slots, B.width, B.slice_ptr, B.len, B.bcol, B.val};
}

// What a kernel of the cycle reads before its product.  On the coarse levels
// such a kernel is a chain of dependent loads, each a trip past the L2 (the
// kernel before it has just written them): the stop flag, the slice and
// length, the columns and values, x, and what the update of the row reads.
// They go out in three rounds: the flag with the slice, the length and the
// row's own values (KEEP holds them before the branch on the flag, below
// which the compiler would sink them), four blocks of a lane at once, their
// x; on a level of one slice width the first round needs no slice or length,
// and the blocks' loads follow it without a wait.  Outer iteration, five or
// six trips before -> this, us: 96x48 56.5 -> 53, 150x75 67.5 -> 62.6,
// 512x256 141 -> 127, 1024x512 260 -> 237, 2048x1024 628 -> 598 (there bound
// by the bytes of its two finest levels).
#define KEEP(v) asm volatile("" : "+v"(v))
struct BellHead {
    uint32_t slice, row, len, done;   // the slice's first slot, the row in it
};
template <int R, int C>
__device__ __forceinline__ BellHead bell_head(const Bell<R, C>& B, uint32_t I, const PcgState* st) {
    uint32_t slice = (I >> 6) * SLICE * B.width, len = B.width;
    if (!B.width) {
        slice = B.slice_ptr[I >> 6];
        len = B.len[I];
    }
    uint32_t zero = 0;   // in a vector register: the flag goes out with the other loads, not
    KEEP(zero);          // through the scalar cache, whose trip the branch would wait for
    return {slice, I & 63, len, (&st->done)[zero]};
}
template <int R>
__device__ __forceinline__ void load_rows(const float* __restrict__ p, uint32_t I, float (&v)[R]) {
#pragma unroll
    for (int m = 0; m < R; ++m) v[m] = p[(size_t)R * I + m];
}
__device__ __forceinline__ void keep(BellHead& h) {
    KEEP(h.len);
    KEEP(h.slice);
    KEEP(h.done);
}
template <int R, class... Rest>
__device__ __forceinline__ void keep(BellHead& h, float (&v)[R], Rest&... rest) {
#pragma unroll
    for (int m = 0; m < R; ++m) KEEP(v[m]);
    keep(h, rest...);
}

// y = (block row) x, x indexed by C per block column, as a group of LANES
// lanes sums it: lane l adds blocks l, l + LANES, ..., and a butterfly the
// lanes' sums.  PHYS lanes do it, each the sums of LANES / PHYS of them, with
// DEPTH blocks (their columns and values) loaded before the dependent gathers;
// every lane of the group gets the result.
template <int R, int C, int LANES, int PHYS = LANES, int DEPTH = 4>
__device__ __forceinline__ void bell_row(const Bell<R, C>& B, const BellHead& h, uint32_t lane,
                                         const float* __restrict__ x, float (&y)[R]) {
    constexpr int V = LANES / PHYS;
    static_assert(DEPTH % V == 0, "a block's accumulator follows from its place");
    float s[V][R] = {};
    const uint32_t base = h.slice + h.row;
    for (uint32_t k0 = lane; k0 < h.len; k0 += DEPTH * PHYS) {
        uint32_t J[DEPTH];
        float a[DEPTH][R * C], xv[DEPTH][C];
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            if (k0 + u * PHYS < h.len) {
                const uint32_t sl = base + (k0 + u * PHYS) * SLICE;
                J[u] = B.bcol[sl];
#pragma unroll
                for (int m = 0; m < R * C; ++m) a[u][m] = B.val[(size_t)m * B.slots + sl];
            }
        }
#pragma unroll
        for (int u = 0; u < DEPTH; ++u)
            if (k0 + u * PHYS < h.len)
#pragma unroll
                for (int c = 0; c < C; ++c) xv[u][c] = x[(size_t)C * J[u] + c];
#pragma unroll
        for (int u = 0; u < DEPTH; ++u)
            if (k0 + u * PHYS < h.len)
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int c = 0; c < C; ++c) s[u % V][r] += a[u][r * C + c] * xv[u][c];
    }
#pragma unroll
    for (int o = V / 2; o > 0; o >>= 1)
#pragma unroll
        for (int v = 0; v < o; ++v)
#pragma unroll
            for (int r = 0; r < R; ++r) s[v][r] += s[v + o][r];
#pragma unroll
    for (int r = 0; r < R; ++r) y[r] = group_sum<PHYS>(s[0][r]);
}

// the group's block row and lane; groups past the last row take that row
// again without storing it (rows >= 1: a branch here would put another trip
// before the first loads)
#define BELL_ROW(LANES, rows)                                       \
    const size_t gid_ = (size_t)blockIdx.x * BLOCK + threadIdx.x;  \
    const uint32_t lane = (uint32_t)(gid_ % LANES);                \
    const bool store = lane == 0 && gid_ / LANES < (rows);         \
    const uint32_t I = min((uint32_t)(gid_ / LANES), (rows) - 1u)

// Chebyshev smoothing below the finest level, a group per aggregate (3
// rows).  The start (r = D^-1 b, d = r / theta, x = d) rides in the
// restriction that writes b; the post-smoothing start takes A x.
template <int LANES, int PHYS>
__global__ __launch_bounds__(BLOCK) void k_bsm_init(Bell<3, 3> A, const float* __restrict__ dinv,
                                                    const float* __restrict__ b,
                                                    const float* __restrict__ x,
                                                    float* __restrict__ r, float* __restrict__ d,
                                                    float inv_theta, const PcgState* st,
                                                    uint32_t rows) {
    BELL_ROW(PHYS, rows);
    BellHead h = bell_head(A, I, st);
    float ax[3], di[3], bi[3];
    load_rows(dinv, I, di);
    load_rows(b, I, bi);
    keep(h, di, bi);
    if (__builtin_amdgcn_readfirstlane(h.done)) return;
    bell_row<3, 3, LANES, PHYS, (LANES / PHYS > 4 ? LANES / PHYS : 4)>(A, h, lane, x, ax);
    if (!store) return;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const size_t i = 3 * (size_t)I + m;
        const float ri = di[m] * (bi[m] - ax[m]);
        r[i] = ri;
        d[i] = ri * inv_theta;
    }
}

// r -= D^-1 A d_in; d_out = c1 d_in + c2 r; x += d_out (and d_in when ADD_IN)
template <bool ADD_IN, int LANES, int PHYS>
__global__ __launch_bounds__(BLOCK) void k_bsm_step(Bell<3, 3> A, const float* __restrict__ dinv,
                                                    const float* __restrict__ din,
                                                    float* __restrict__ dout,
                                                    float* __restrict__ r, float* __restrict__ x,
                                                    float c1, float c2, const PcgState* st,
                                                    uint32_t rows) {
    BELL_ROW(PHYS, rows);
    BellHead h = bell_head(A, I, st);
    float ad[3], dv[3], d0[3], r0[3], x0[3];
    load_rows(dinv, I, dv);
    load_rows(din, I, d0);
    load_rows(r, I, r0);
    load_rows(x, I, x0);
    keep(h, dv, d0, r0, x0);
    if (__builtin_amdgcn_readfirstlane(h.done)) return;
    bell_row<3, 3, LANES, PHYS, (LANES / PHYS > 4 ? LANES / PHYS : 4)>(A, h, lane, din, ad);
    if (!store) return;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const size_t i = 3 * (size_t)I + m;
        const float ri = r0[m] - dv[m] * ad[m];
        const float dn = c1 * d0[m] + c2 * ri;
        r[i] = ri;
        dout[i] = dn;
        x[i] = x0[m] + (ADD_IN ? d0[m] + dn : dn);
    }
}

template <int LANES, int PHYS>
__global__ __launch_bounds__(BLOCK) void k_bresidual(Bell<3, 3> A, const float* __restrict__ b,
                                                     const float* __restrict__ x,
                                                     float* __restrict__ r, const PcgState* st,
                                                     uint32_t rows) {
    BELL_ROW(PHYS, rows);
    BellHead h = bell_head(A, I, st);
    float ax[3], bi[3];
    load_rows(b, I, bi);
    keep(h, bi);
    if (__builtin_amdgcn_readfirstlane(h.done)) return;
    bell_row<3, 3, LANES, PHYS, (LANES / PHYS > 4 ? LANES / PHYS : 4)>(A, h, lane, x, ax);
    if (!store) return;
#pragma unroll
    for (int m = 0; m < 3; ++m) r[3 * (size_t)I + m] = bi[m] - ax[m];
}

// b_c = P^T r, a group per aggregate; INIT: also the next level's
// smoothing start from x = 0 (r_c = D_c^-1 b_c, d_c = r_c / theta_c, x_c = d_c)
template <int R, bool INIT, int LANES, int PHYS>
__global__ __launch_bounds__(BLOCK) void k_brestrict(Bell<3, R> T, const float* __restrict__ r,
                                                     float* __restrict__ bc,
                                                     const float* __restrict__ dinv_c,
                                                     float* __restrict__ xc,
                                                     float* __restrict__ rc,
                                                     float* __restrict__ dc, float inv_theta_c,
                                                     const PcgState* st, uint32_t aggs) {
    BELL_ROW(PHYS, aggs);
    BellHead h = bell_head(T, I, st);
    float y[3], di[3] = {};
    if constexpr (INIT) {
        load_rows(dinv_c, I, di);
        keep(h, di);
    } else {
        keep(h);
    }
    if (__builtin_amdgcn_readfirstlane(h.done)) return;
    bell_row<3, R, LANES, PHYS, (LANES / PHYS > 4 ? LANES / PHYS : 4)>(T, h, lane, r, y);
    if (!store) return;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const size_t i = 3 * (size_t)I + m;
        bc[i] = y[m];
        if constexpr (INIT) {
            const float ri = di[m] * y[m];
            const float d = ri * inv_theta_c;
            rc[i] = ri;
            dc[i] = d;
            xc[i] = d;
        }
    }
}

// x += P x_c (ADD), or x = P x_c; a group per node
template <int R, bool ADD, int LANES, int PHYS>
__global__ __launch_bounds__(BLOCK) void k_bprolong(Bell<R, 3> P, const float* __restrict__ xc,
                                                    float* __restrict__ x, const PcgState* st,
                                                    uint32_t rows) {
    BELL_ROW(PHYS, rows);
    BellHead h = bell_head(P, I, st);
    float y[R], x0[R] = {};
    if constexpr (ADD) {
        load_rows(x, I, x0);
        keep(h, x0);
    } else {
        keep(h);
    }
    if (__builtin_amdgcn_readfirstlane(h.done)) return;
    bell_row<R, 3, LANES, PHYS, (LANES / PHYS > 4 ? LANES / PHYS : 4)>(P, h, lane, xc, y);
    if (!store) return;
#pragma unroll
    for (int m = 0; m < R; ++m) x[(size_t)R * I + m] = ADD ? x0[m] + y[m] : y[m];
}

// x = C^-1 b on the coarsest level (n <= AMG_COARSEST), one workgroup
constexpr int DENSE_BLOCK = 256;
__global__ __launch_bounds__(DENSE_BLOCK) void k_amg_dense(const float* __restrict__ cinv,
                                                           const float* __restrict__ b,
                                                           float* __restrict__ x,
                                                           const PcgState* st, uint32_t n) {
    if (st->done) return;
    __shared__ float sb[AMG_COARSEST];
    for (uint32_t j = threadIdx.x; j < n; j += DENSE_BLOCK) sb[j] = b[j];
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += DENSE_BLOCK) {
        float s = 0.f;
        for (uint32_t j = 0; j < n; ++j) s += cinv[(size_t)i * n + j] * sb[j];
        x[i] = s;
    }
}

// ---- the bottom of the V-cycle in one workgroup -------------------------------
// A smoothing step on a level of a few hundred unknowns costs a launch and a
// chain of dependent loads (3.5-4 us), and the last smoothed level takes 8-13
// such launches per cycle with the dense solve below it.  One workgroup of 512
// or 1,024 threads does them all, down to the dense solve and back up, when
// that level has at most 1,024 unknowns.  Its operator is read once and kept in
// registers (a thread holds a scalar row, padded with zero blocks to HELD, so
// that a product's LDS reads go out together), every vector lives in LDS, and a
// step costs one barrier; the products (0.5 us) and the loads of P, P^T and C^-1
// bound it.  Every sum keeps the order of the kernels of one step each, so the
// cycle's result is the same to the bit.  The kernel and the outer iteration
// around it, with the launches it replaces and with it (cantilevers): 357
// unknowns (150x75) 14 us, 104 -> 71; 726 (64x32) 62 -> 43; 969 (256x128)
// 118 -> 95; 288 (512x256) 17 us, 184 -> 150; 312 (2048x1024) 25 us,
// 661 -> 630.  With two rows a thread in 512 threads 64x32 42.1 instead of
// 40.6 now, 256x128 78.4 instead of 76; more unknowns than that (three rows a
// thread spill) take as long as the launches.
// Threads take the scalar rows of equal component r of consecutive block
// rows, so that a wavefront's loads of a block position are coalesced.
struct BottomLevel {
    Bell<3, 3> A, P, T;
    const float* dinv;
    int p_lanes, t_lanes;               // lanes per row of P and T
    uint32_t rows, degree;              // block rows
    float inv_theta, c1[AMG_MAX_DEGREE], c2[AMG_MAX_DEGREE];
};
struct Bottom {
    BottomLevel lv;
    uint32_t nco;
    const float* cinv;
    const float* b;
    float* x;
};
// one thread's scalar row on a level: component r of block row I, thread
// r rows + I
template <int HELD, int LANES>   // HELD: blocks of a row, none longer
struct BottomRows {
    uint32_t at;   // the scalar row's place in LDS (3 I + r), or none
    float dinv;
    static constexpr uint32_t NO_ROW = 0xffffffffu;
    __device__ __forceinline__ bool on() const { return at != NO_ROW; }
    float v[HELD][3];
    uint32_t col[HELD / 2];   // two 16-bit places (3 J) per word
    // component r of block row I: its values, and with COLS the columns as
    // they stand
    template <bool COLS>
    __device__ __forceinline__ void load_row(const BottomLevel& L, uint32_t I, uint32_t r,
                                             bool valid) {
        dinv = valid ? L.dinv[3 * (size_t)I + r] : 0.f;
        size_t base = (size_t)(I >> 6) * SLICE * L.A.width + (I & 63);
        int len = valid ? (int)L.A.width : 0;
        if (valid && !L.A.width) {
            base = (size_t)L.A.slice_ptr[I >> 6] + (I & 63);
            len = L.A.len[I];
        }
#pragma unroll
        for (int k = 0; k < HELD; ++k) {
#pragma unroll
            for (int c = 0; c < 3; ++c) v[k][c] = 0.f;
            if (k < len) {
                const size_t sl = base + (size_t)k * SLICE;
                if constexpr (COLS) col[k / 2] |= (3 * L.A.bcol[sl]) << (16 * (k & 1));
#pragma unroll
                for (int c = 0; c < 3; ++c) v[k][c] = L.A.val[(size_t)(3 * r + c) * L.A.slots + sl];
            }
        }
    }
    __device__ __forceinline__ void load(const BottomLevel& L) {
        const uint32_t r = threadIdx.x / L.rows, I = threadIdx.x - r * L.rows;
        const bool valid = r < 3;
        at = valid ? 3 * I + r : NO_ROW;
#pragma unroll
        for (int k = 0; k < HELD / 2; ++k) col[k] = 0;
        load_row<true>(L, I, r, valid);
    }
    // (A x) of the row, summed as bell_row's LANES lanes sum it
    __device__ __forceinline__ float product(const float* x) const {
        float y[LANES] = {};
#pragma unroll
        for (int k = 0; k < HELD; ++k) {
            const float* xk = x + ((col[k / 2] >> (16 * (k & 1))) & 0xffffu);
            float& t = y[k % LANES];
            t += v[k][0] * xk[0];
            t += v[k][1] * xk[1];
            t += v[k][2] * xk[2];
        }
#pragma unroll
        for (int o = LANES / 2; o > 0; o >>= 1)
#pragma unroll
            for (int l = 0; l < o; ++l) y[l] += y[l + o];
        return y[0];
    }
    __device__ __forceinline__ float scaled(const float* x) const { return dinv * product(x); }
};
// Vectors of a level in LDS: right-hand side, solution, residual (or the
// second direction), direction.
struct BottomVec {
    float *b, *x, *r, *d;
};
// x = 0 start and degree - 1 steps, then the residual b - A x into v.r
template <int HELD, int LANES>
__device__ __forceinline__ void bottom_down(const BottomLevel& L,
                                            const BottomRows<HELD, LANES>& R, const BottomVec& v) {
    float rr = 0.f, xx = 0.f, dd = 0.f;
    if (R.on()) {
        rr = R.dinv * v.b[R.at];
        dd = rr * L.inv_theta;
        xx = dd;
        v.d[R.at] = dd;
    }
    float *din = v.d, *dout = v.r;
    for (uint32_t k = 1; k < L.degree; ++k) {
        __syncthreads();
        if (R.on()) {
            rr -= R.scaled(din);
            dd = L.c1[k] * dd + L.c2[k] * rr;
            xx += dd;
            dout[R.at] = dd;
        }
        float* t = din;
        din = dout;
        dout = t;
    }
    if (R.on()) v.x[R.at] = xx;
    __syncthreads();
    if (R.on()) v.r[R.at] = v.b[R.at] - R.product(v.x);
    __syncthreads();
}
// post-smoothing from v.x
template <int HELD, int LANES>
__device__ __forceinline__ void bottom_up(const BottomLevel& L, const BottomRows<HELD, LANES>& R,
                                          const BottomVec& v) {
    float rr = 0.f, xx = 0.f, dd = 0.f;
    if (R.on()) {
        xx = v.x[R.at];
        rr = R.dinv * (v.b[R.at] - R.product(v.x));
        dd = rr * L.inv_theta;
        v.d[R.at] = dd;
    }
    float *din = v.d, *dout = v.r;
    for (uint32_t k = 1; k < L.degree; ++k) {
        __syncthreads();
        if (R.on()) {
            rr -= R.scaled(din);
            const float dn = L.c1[k] * dd + L.c2[k] * rr;
            xx += k == 1 ? dd + dn : dn;
            dd = dn;
            dout[R.at] = dn;
        }
        float* t = din;
        din = dout;
        dout = t;
    }
    __syncthreads();
    if (R.on()) v.x[R.at] = xx;
    __syncthreads();
}
// y = B x, or y += B x (ADD); LANES lanes per block row
template <bool ADD, int LANES>
__device__ __forceinline__ void bottom_apply(const Bell<3, 3>& B, uint32_t rows, const float* x,
                                             float* y) {
    const uint32_t lane = threadIdx.x % LANES;
    for (uint32_t I = threadIdx.x / LANES; I < rows; I += blockDim.x / LANES) {
        float t[3];
        bell_row<3, 3, LANES, LANES, 2>(B, BellHead{B.slice_ptr[I >> 6], I & 63, B.len[I], 0}, lane,
                                        x, t);
        if (lane == 0)
#pragma unroll
            for (int r = 0; r < 3; ++r) y[3 * I + r] = ADD ? y[3 * I + r] + t[r] : t[r];
    }
    __syncthreads();
}
template <bool ADD>
__device__ __forceinline__ void bottom_apply(const Bell<3, 3>& B, int lanes, uint32_t rows,
                                             const float* x, float* y) {
    switch (lanes) {
        case 1: bottom_apply<ADD, 1>(B, rows, x, y); break;
        case 2: bottom_apply<ADD, 2>(B, rows, x, y); break;
        case 4: bottom_apply<ADD, 4>(B, rows, x, y); break;
        case 8: bottom_apply<ADD, 8>(B, rows, x, y); break;
        default: bottom_apply<ADD, 16>(B, rows, x, y); break;
    }
}
template <int TB, int HELD, int LANES>
__global__ __launch_bounds__(TB) void k_amg_bottom(Bottom B, const PcgState* st) {
    if (st->done) return;
    extern __shared__ float lds[];
    const BottomLevel& L0 = B.lv;
    const uint32_t n = 3 * L0.rows;
    const BottomVec v{lds, lds + n, lds + 2 * n, lds + 3 * n};
    float *bc = lds + 4 * n, *xc = bc + B.nco;
    BottomRows<HELD, LANES> R0;
    R0.load(L0);
    for (uint32_t i = threadIdx.x; i < n; i += TB) v.b[i] = B.b[i];
    __syncthreads();
    bottom_down(L0, R0, v);
    bottom_apply<false>(L0.T, L0.t_lanes, B.nco / 3, v.r, bc);
    // x = C^-1 b (C^-1 is symmetric: its columns are read as rows)
    if (threadIdx.x < B.nco) {
        const float* c = B.cinv + threadIdx.x;
        float t = 0.f;
#pragma unroll 24
        for (uint32_t j = 0; j < B.nco; ++j) t += c[(size_t)j * B.nco] * bc[j];
        xc[threadIdx.x] = t;
    }
    __syncthreads();
    bottom_apply<true>(L0.P, L0.p_lanes, L0.rows, xc, v.x);
    bottom_up(L0, R0, v);
    for (uint32_t i = threadIdx.x; i < n; i += TB) B.x[i] = v.x[i];
}

// ---- a level between the finest and the bottom, on tiles ------------------------
// Such a level takes 2 degree + 3 launches of one step each per cycle. On tiles
// (tiles.hip) of its graph with `degree` rings it takes two, with the
// restriction between them: k_amg_down all steps before the coarse correction
// and the residual, k_amg_up the prolongation and all steps after.  A tile's
// rows are held as k_amg_bottom holds its own; a step is taken on the rows whose
// neighbours' last step this workgroup has, so each leaves a ring behind.
// Sums keep the order of the kernels of one step: same bits.
// Bound by the launch and the loads of the rows (about 200 listed for 57 owned
// at degree 2, 300 for 20 at degree 4).  One scalar row a thread: with two in
// 512 threads 120 us per outer iteration at 512x256 instead of 115.  Launch per
// step -> tiles, us per outer iteration: 96x48 56.1 -> 49.1, 150x75 64.7 ->
// 56.6, 256x128 84.1 -> 78.0, 512x256 137 -> 115, 1024x512 232 -> 210,
// 2048x1024 572 -> 563.
template <int HELD, int LANES>
struct TileHeld : BottomRows<HELD, LANES> {
    uint32_t I, r, act;  // block row, component, rings inside (0: the outermost)
    uint32_t own, all;   // rows owned, rows listed
    // false: the solve has ended, or the tile owns nothing
    __device__ __forceinline__ bool load(const BottomLevel& L, const Tiles& T, const PcgState* st) {
        const uint32_t tile = xcd_remap(blockIdx.x, gridDim.x);
        uint32_t zero = 0;
        KEEP(zero);
        uint32_t ro = T.roff[(size_t)tile * (T.rings + 1) + min(threadIdx.x % WAVE, T.rings)];
        uint32_t done = (&st->done)[zero];
        KEEP(ro);
        KEEP(done);
        own = __builtin_amdgcn_readlane(ro, 0);
        all = __builtin_amdgcn_readlane(ro, T.rings);
        if (__builtin_amdgcn_readfirstlane(done) || !own) return false;
        r = threadIdx.x / all;
        const uint32_t e = threadIdx.x - r * all;
        const bool valid = r < 3;
        act = 0;   // rings that hold the row, so products it may take
        for (uint32_t k = 0; k < T.rings; ++k)
            act += e < (uint32_t)__builtin_amdgcn_readlane(ro, k);
        if (!valid) act = 0;
        this->at = valid ? 3 * e + r : this->NO_ROW;
        I = valid ? T.ids[(size_t)tile * T.ext + e] : 0;
#pragma unroll
        for (int k = 0; k < HELD / 2; ++k) {
            uint32_t w = 0;
            if (act && k < (int)T.W2) w = T.lcol[((size_t)tile * T.W2 + k) * T.ext + e];
            this->col[k] = (3 * (w & 0xffffu)) | ((3 * (w >> 16)) << 16);
        }
        this->template load_row<false>(L, I, r, act != 0);
        if (valid) this->dinv = L.dinv[3 * (size_t)I + r];
        return true;
    }
    __device__ __forceinline__ bool owned() const { return this->on() && this->at < 3 * own; }
    __device__ __forceinline__ size_t global() const { return 3 * (size_t)I + r; }
};
template <int TB, int HELD, int LANES>
__global__ __launch_bounds__(TB) void k_amg_down(BottomLevel L, Tiles T,
                                                 const float* __restrict__ b,
                                                 float* __restrict__ x, float* __restrict__ r,
                                                 const PcgState* st) {
    extern __shared__ float lds[];
    TileHeld<HELD, LANES> R;
    if (!R.load(L, T, st)) return;
    float *din = lds, *dout = lds + 3 * R.all, *xs = lds + 6 * R.all;
    float bb = 0.f, rr = 0.f, xx = 0.f, dd = 0.f;
    if (R.on()) {
        bb = b[R.global()];
        rr = R.dinv * bb;
        dd = rr * L.inv_theta;
        xx = dd;
        din[R.at] = dd;
    }
    for (uint32_t k = 1; k < L.degree; ++k) {
        __syncthreads();
        if (k <= R.act) {
            rr -= R.scaled(din);
            dd = L.c1[k] * dd + L.c2[k] * rr;
            xx += dd;
            dout[R.at] = dd;
        }
        float* t = din;
        din = dout;
        dout = t;
    }
    if (R.on()) xs[R.at] = xx;
    __syncthreads();
    if (R.owned()) {
        r[R.global()] = bb - R.product(xs);
        x[R.global()] = xx;
    }
}
template <int TB, int HELD, int LANES>
__global__ __launch_bounds__(TB) void k_amg_up(BottomLevel L, Tiles T,
                                               const float* __restrict__ b,
                                               const float* __restrict__ x,
                                               const float* __restrict__ xc,
                                               float* __restrict__ out, const PcgState* st) {
    extern __shared__ float lds[];
    TileHeld<HELD, LANES> R;
    if (!R.load(L, T, st)) return;
    float *din = lds, *dout = lds + 3 * R.all, *xs = lds + 6 * R.all;
    float rr = 0.f, xx = 0.f, dd = 0.f;
    if (R.on()) {   // x + P xc, by one lane a row
        const uint32_t I = R.I;
        const Bell<3, 3>& P = L.P;
        uint32_t base = (I >> 6) * SLICE * P.width + (I & 63), len = P.width;
        if (!P.width) {
            base = P.slice_ptr[I >> 6] + (I & 63);
            len = P.len[I];
        }
        const float* const val = P.val + (size_t)(3 * R.r) * P.slots;
        float y = 0.f;
        for (uint32_t k0 = 0; k0 < len; k0 += 4) {
            float a[4][3], v[4][3];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u)
                if (k0 + u < len) {
                    const uint32_t sl = base + (k0 + u) * SLICE;
                    const float* const xj = xc + 3 * (size_t)P.bcol[sl];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        a[u][c] = val[(size_t)c * P.slots + sl];
                        v[u][c] = xj[c];
                    }
                }
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u)
                if (k0 + u < len)
#pragma unroll
                    for (int c = 0; c < 3; ++c) y += a[u][c] * v[u][c];
        }
        xx = x[R.global()] + y;
        xs[R.at] = xx;
    }
    __syncthreads();
    if (R.act) {
        rr = R.dinv * (b[R.global()] - R.product(xs));
        dd = rr * L.inv_theta;
        din[R.at] = dd;
    }
    for (uint32_t k = 1; k < L.degree; ++k) {
        __syncthreads();
        if (k < R.act) {
            rr -= R.scaled(din);
            const float dn = L.c1[k] * dd + L.c2[k] * rr;
            xx += k == 1 ? dd + dn : dn;
            dd = dn;
            dout[R.at] = dn;
        }
        float* t = din;
        din = dout;
        dout = t;
    }
    if (R.owned()) out[R.global()] = xx;
}

}  // namespace


void amg_free(AmgDev* A) {
    if (!A) return;
    for (AmgDevLevel& L : A->lv) {
        void* ps[] = {L.a_ptr, L.a_col, L.a64, L.dinv64, L.dinv32, L.t, L.agg, L.p_ptr,
                      L.p_col, L.p64, L.w_ptr, L.w_col, L.w64, L.pt_ptr,
                      L.pt_row, L.pt_pos, L.b, L.x, L.r, L.d0, L.d1};
        for (void* p : ps)
            if (p) (void)hipFree(p);
        for (BellDev* B : {&L.ab, &L.pb, &L.tb}) {
            void* qs[] = {B->slice_ptr, B->len, B->bcol, B->val};
            for (void* q : qs)
                if (q) (void)hipFree(q);
        }
        tiles_free(L.tiles);
    }
    void* ps[] = {A->cinv, A->ones,     A->pow_x,  A->pow_y,
                  A->scal, A->partials, A->nzbits, A->differ, A->dense};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    delete A;
}

constexpr size_t BELL_SMALL = 65536;   // slots (2.6 MB)
constexpr uint32_t BELL_LARGE = 32768;   // block rows

// The block sliced-ELL pattern of `rows` block rows: len_of(I) blocks in
// row I, col_of(I, k) the k-th block's column; uploaded with room for R x C
// FP32 values per slot.  NBX_ERR_ARG when a row has more blocks than the
// format holds (65,535) or the layout more than 2^32 slots.
template <int R, int C, class Len, class Col>
static int bell_upload(uint32_t rows, Len len_of, Col col_of, BellDev& B, size_t& bytes) {
    const uint32_t ns = (rows + SLICE - 1) / SLICE;
    std::vector<uint32_t> sp(ns + 1, 0);
    std::vector<uint16_t> len(rows, 0);
    for (uint32_t sl = 0; sl < ns; ++sl) {
        uint32_t w = 0;
        for (uint32_t I = sl * SLICE; I < std::min<uint32_t>(rows, (sl + 1) * SLICE); ++I) {
            const uint32_t l = len_of(I);
            if (l > 0xffffu) {
                set_last_error("AMG: a block row of %u blocks", l);
                return NBX_ERR_ARG;
            }
            len[I] = (uint16_t)l;
            w = std::max(w, l);
        }
        if ((uint64_t)sp[sl] + (uint64_t)w * SLICE > 0xffffffffull) {
            set_last_error("AMG: block layout beyond 2^32 slots");
            return NBX_ERR_ARG;
        }
        sp[sl + 1] = sp[sl] + w * SLICE;
    }
    std::vector<uint32_t> bcol(sp[ns], 0);
    // One width for all slices where that adds little or the level is small:
    // a row's place then follows from its index, without the loads of its
    // slice and length before its blocks' (96x48 58 -> 53 us per outer
    // iteration, 512x256 130 -> 127, 2048x1024 608 -> 598).  Padding blocks are
    // zero, on the row's own first column: they add +0 to sums that are never -0.
    for (uint16_t l : len) B.wmax = std::max<uint32_t>(B.wmax, l);
    const size_t same = (size_t)ns * SLICE * B.wmax;
    if (same <= 0xffffffffull && (same <= sp[ns] + (size_t)sp[ns] / 8 || same <= BELL_SMALL)) {
        B.width = B.wmax;
        for (uint32_t sl = 0; sl <= ns; ++sl) sp[sl] = sl * SLICE * B.width;
        bcol.assign(same, 0);
    }
    for (uint32_t I = 0; I < rows; ++I) {
        const uint32_t w = len[I] ? std::max<uint32_t>(B.width, len[I]) : 0;
        for (uint32_t k = 0; k < w; ++k)
            bcol[sp[I / SLICE] + (size_t)k * SLICE + I % SLICE] = col_of(I, k < len[I] ? k : 0);
    }
    B.rows = rows;
    B.slots = sp[ns];
    // about three blocks per lane (1, 2, 4, 8 or 16 lanes)
    size_t used = 0;
    for (uint32_t I = 0; I < rows; ++I) used += len[I];
    const double avg = rows ? (double)used / rows : 0.0;
    B.lanes = 1;
    while (B.lanes < 16 && avg / (2 * B.lanes) >= 2.5) B.lanes *= 2;
    NBX_TRY(up(&B.slice_ptr, sp, bytes));
    NBX_TRY(up(&B.len, len, bytes));
    NBX_TRY(up(&B.bcol, bcol, bytes));
    NBX_TRY(alloc(&B.val, B.slots * R * C, bytes));
    if (B.width) NBX_HIP(hipMemset(B.val, 0, B.slots * R * C * sizeof(float)));
    return NBX_OK;
}

// Whether the R rows of every block row share one pattern of complete
// C-column groups (what the block layout stores).
static bool grouped(uint32_t rows, int R, int C, const HostVec<uint32_t>& ptr,
                    const HostVec<uint32_t>& col) {
    for (uint32_t I = 0; I < rows; ++I) {
        const uint32_t b0 = ptr[(size_t)R * I], l = ptr[(size_t)R * I + 1] - b0;
        if (l % C) return false;
        for (int r = 1; r < R; ++r) {
            const uint32_t br = ptr[(size_t)R * I + r];
            if (ptr[(size_t)R * I + r + 1] - br != l) return false;
            for (uint32_t q = 0; q < l; ++q)
                if (col[br + q] != col[b0 + q]) return false;
        }
        for (uint32_t q = 0; q < l; q += C)
            for (int c = 1; c < C; ++c)
                if (col[b0 + q + c] != col[b0 + q] + c || col[b0 + q] % C) return false;
    }
    return true;
}

// Most scalar rows of level L that a workgroup holds, one a thread: 1,024 of up
// to 14 blocks (the coarse levels of structured T3 meshes have 11-13), 512 of
// up to 24; 0 where the rows do not fit.  Rows of 5 to 20 blocks on average,
// that is 2 or 4 lanes in the kernels of one step: thinner and denser levels
// are too rare to pay for more forms.
static uint32_t held_rows(const AmgDevLevel& L) {
    if (L.ab.lanes != 2 && L.ab.lanes != 4) return 0;
    return L.ab.wmax <= 14 ? 1024 : L.ab.wmax <= 24 ? 512 : 0;
}
static bool bottom_fits(const AmgDevLevel& L) { return L.n <= held_rows(L); }
// f(threads, HELD, LANES) for a workgroup of `rows` scalar rows of level V
template <class F>
static void with_row_form(const AmgDevLevel& V, uint32_t rows, F&& f) {
    using std::integral_constant;
    auto lanes = [&](auto tb, auto held) {
        if (V.ab.lanes == 2)
            f(tb, held, integral_constant<int, 2>{});
        else
            f(tb, held, integral_constant<int, 4>{});
    };
    if (V.ab.wmax > 14)
        lanes(integral_constant<int, 512>{}, integral_constant<int, 24>{});
    else if (rows <= 512)
        lanes(integral_constant<int, 512>{}, integral_constant<int, 14>{});
    else
        lanes(integral_constant<int, 1024>{}, integral_constant<int, 14>{});
}

// The mean place of each aggregate's nodes (the next level's nodes)
static std::vector<double> mean_places(const AmgHostLevel& h, const std::vector<double>& xy) {
    std::vector<double> out(2 * (size_t)(h.nc / 3), 0.0), cnt(h.nc / 3, 0.0);
    for (uint32_t i = 0; i < h.n / h.bs; ++i) {
        const uint32_t a = h.agg[i];
        if (a >= h.nc / 3) continue;   // in no aggregate
        out[2 * (size_t)a] += xy[2 * (size_t)i];
        out[2 * (size_t)a + 1] += xy[2 * (size_t)i + 1];
        cnt[a] += 1.0;
    }
    for (size_t a = 0; a < cnt.size(); ++a)
        for (int c = 0; c < 2; ++c) out[2 * a + c] /= std::max(cnt[a], 1.0);
    return out;
}

// Tiles of a level of fewer than BELL_LARGE block rows (larger ones are bound by
// bytes, of which the rings read more), at most 256, which run at once (a tile
// takes a CU: 19,608 rows of degree 4 in 990 tiles take 644 us per outer
// iteration instead of 563 with a launch per step), of about 8 rows at least
// (a launch takes as long as its largest tile: 16 rows 1-2 us more).
static int level_tiles(AmgDevLevel& L, const std::vector<double>& xy, hipStream_t s) {
    // (a row's P by one lane, as the prolongation's kernel sums it)
    const uint32_t limit = L.pb.lanes == 1 ? held_rows(L) / 3 : 0;
    const uint32_t rows = L.n / 3, rings = (uint32_t)L.degree;
    if (!limit || rows >= BELL_LARGE || rows < 64) return NBX_OK;
    const uint32_t cells = std::max(std::min(256u, rows / 8), 1u);
    double2* d = nullptr;
    NBX_HIP(hipMalloc(&d, (size_t)rows * sizeof(double2)));
    hipError_t e = copy_on(d, xy.data(), (size_t)rows * sizeof(double2), hipMemcpyHostToDevice, s);
    int rc = NBX_OK;
    std::vector<TileAttempt> attempts{{cells, rings, rings}};
    if (cells < 256) attempts.push_back({std::min(256u, 2 * cells), rings, rings});
    if (e == hipSuccess)
        rc = tiles_build(L.tiles, TileRows<uint16_t>{L.ab.slice_ptr, L.ab.len, L.ab.bcol}, rows,
                         L.ab.wmax, d, attempts, limit, s);
    (void)hipFree(d);
    NBX_HIP(e);
    return rc;
}

// Symbolic hierarchy of the system's current K (pattern, Dirichlet rows,
// node coordinates), uploaded; replaces any previous one.
static int amg_symbolic(FemSys& S) {
    amg_free(S.K.amg);
    S.K.amg = nullptr;
    S.K.amg_current = false;
    const uint32_t n = 2 * S.nn;
    const size_t nnz = S.K.s.n_valid * 4;
    if ((size_t)n > (size_t)MAX_GRID * BLOCK || nnz > 0xffffffffull) {
        set_last_error("AMG: %u unknowns (at most %u) or %zu nonzeros", n,
                       (unsigned)(MAX_GRID * BLOCK), nnz);
        return NBX_ERR_ARG;
    }
    // the finest pattern and its nonzero entries, from the block layout's
    // columns and one flag byte per block (the values stay on the device)
    const Sell2& K = S.K.s;
    std::vector<uint32_t> sp(K.n_slices + 1);
    std::vector<uint8_t> len(S.nn + 1);
    HostVec<uint32_t> bc(K.n_blocks + 1);
    HostVec<uint8_t> bits(K.n_blocks + 1);
    std::vector<double> xy(2 * (size_t)S.nn);
    struct Bits {   // kept with the hierarchy once that is complete
        uint8_t* d = nullptr;
        ~Bits() { if (d) (void)hipFree(d); }
    } dbits;
    NBX_HIP(hipMalloc(&dbits.d, K.n_blocks + 1));
    hipLaunchKernelGGL(k_block_nzbits, dim3(grid_for(K.n_blocks)), dim3(BLOCK), 0, S.s, K, dbits.d);
    NBX_HIP(hipGetLastError());
    NBX_HIP(hipMemcpyAsync(bits.data(), dbits.d, K.n_blocks, hipMemcpyDeviceToHost, S.s));
    NBX_HIP(hipStreamSynchronize(S.s));
    NBX_HIP(hipMemcpyAsync(sp.data(), K.slice_ptr, (K.n_slices + 1) * 4, hipMemcpyDeviceToHost,
                           S.s));
    if (S.nn) NBX_HIP(hipMemcpyAsync(len.data(), K.rowlen, S.nn, hipMemcpyDeviceToHost, S.s));
    NBX_HIP(hipMemcpyAsync(bc.data(), K.bcol, K.n_blocks * 4, hipMemcpyDeviceToHost, S.s));
    NBX_HIP(copy_on(xy.data(), S.nod, xy.size() * sizeof(double), hipMemcpyDeviceToHost, S.s));
    HostVec<uint32_t> rp, col;
    HostVec<uint8_t> nzf;
    amg_expand_blocks(S.nn, sp.data(), len.data(), bc.data(), bits.data(), rp, col, nzf);
    if (rp.size() != (size_t)n + 1 || col.size() != nnz) {
        set_last_error("AMG: the block layout holds %zu entries, the pattern %zu", col.size(), nnz);
        return NBX_ERR_ARG;
    }
    AmgHost H;
    const int hb = amg_build_host(n, rp.data(), col.data(), nzf.data(), xy.data(), H);
    if (hb == -2) {
        set_last_error("AMG: host memory ran out building the hierarchy");
        return NBX_ERR_ARG;
    }
    if (hb) {
        set_last_error("AMG: the matrix is not a 2-dof node pattern");
        return NBX_ERR_ARG;
    }
    if (H.lv.back().n > AMG_COARSEST) {
        set_last_error("AMG: coarsening stopped at %u unknowns (at most %u are solved directly)",
                       H.lv.back().n, AMG_COARSEST);
        return NBX_ERR_ARG;
    }
    AmgDev* A = new AmgDev();
    S.K.amg = A;
    A->lv.resize(H.lv.size());
    const size_t nl = H.lv.size();
    for (size_t l = 0; l < nl; ++l) {
        const AmgHostLevel& h = H.lv[l];
        const uint32_t bs = l == 0 ? 2 : 3;
        const bool ok = h.n % bs == 0 && grouped(h.n / bs, (int)bs, (int)bs, h.a_ptr, h.a_col) &&
                        (l + 1 == nl || (h.nc % 3 == 0 &&
                                          grouped(h.n / bs, (int)bs, 3, h.p_ptr, h.p_col) &&
                                          grouped(h.n / bs, (int)bs, 3, h.w_ptr, h.w_col)));
        if (!ok) {
            set_last_error("AMG: level %zu is not in %ux%u / %ux3 node blocks", l, bs, bs, bs);
            return NBX_ERR_ARG;
        }
    }
    for (size_t l = 0; l < nl; ++l) {
        const AmgHostLevel& h = H.lv[l];
        AmgDevLevel& L = A->lv[l];
        if (l > 0) xy = mean_places(H.lv[l - 1], xy);
        L.n = h.n;
        L.nc = h.nc;
        L.bs = l == 0 ? 2 : 3;
        L.degree = amg_level_degree(l);
        L.a_nnz = h.a_col.size();
        NBX_TRY(up(&L.a_ptr, h.a_ptr, A->bytes));
        NBX_TRY(up(&L.a_col, h.a_col, A->bytes));
        NBX_TRY(alloc(&L.a64, L.a_nnz, A->bytes));
        if (l > 0 && l + 1 < nl) {
            const uint32_t* ap = h.a_ptr.data();
            const uint32_t* ac = h.a_col.data();
            auto alen = [&](uint32_t I) { return (ap[3 * (size_t)I + 1] - ap[3 * (size_t)I]) / 3; };
            auto acol = [&](uint32_t I, uint32_t k) { return ac[ap[3 * (size_t)I] + 3 * k] / 3; };
            NBX_TRY((bell_upload<3, 3>(h.n / 3, alen, acol, L.ab, A->bytes)));
        }
        NBX_TRY(alloc(&L.dinv64, L.n, A->bytes));
        NBX_TRY(alloc(&L.dinv32, L.n, A->bytes));
        NBX_TRY(alloc(&L.r, L.n, A->bytes));
        NBX_TRY(alloc(&L.d0, L.n, A->bytes));
        NBX_TRY(alloc(&L.d1, L.n, A->bytes));
        if (l > 0) {
            NBX_TRY(alloc(&L.b, L.n, A->bytes));
            NBX_TRY(alloc(&L.x, L.n, A->bytes));
        }
        if (l + 1 < H.lv.size()) {
            L.p_nnz = h.p_col.size();
            L.w_nnz = h.w_col.size();
            const uint32_t R = L.bs;
            const uint32_t* pp = h.p_ptr.data();
            const uint32_t* pc = h.p_col.data();
            const uint32_t* tp = h.pt_ptr.data();
            const uint32_t* tr = h.pt_row.data();
            auto plen = [&](uint32_t I) { return (pp[R * (size_t)I + 1] - pp[R * (size_t)I]) / 3; };
            auto pcol = [&](uint32_t I, uint32_t k) { return pc[pp[R * (size_t)I] + 3 * k] / 3; };
            auto tlen = [&](uint32_t a) { return (tp[3 * (size_t)a + 1] - tp[3 * (size_t)a]) / R; };
            auto tcol = [&](uint32_t a, uint32_t k) { return tr[tp[3 * (size_t)a] + R * k] / R; };
            if (R == 2) {
                NBX_TRY((bell_upload<2, 3>(L.n / 2, plen, pcol, L.pb, A->bytes)));
                NBX_TRY((bell_upload<3, 2>(L.nc / 3, tlen, tcol, L.tb, A->bytes)));
            } else {
                NBX_TRY((bell_upload<3, 3>(L.n / 3, plen, pcol, L.pb, A->bytes)));
                NBX_TRY((bell_upload<3, 3>(L.nc / 3, tlen, tcol, L.tb, A->bytes)));
                // (the last smoothed level: with the dense solve, where it can)
                if (l + 2 < nl || !bottom_fits(L)) NBX_TRY(level_tiles(L, xy, S.s));
            }
            NBX_TRY(up(&L.t, h.t, A->bytes));
            NBX_TRY(up(&L.agg, h.agg, A->bytes));
            NBX_TRY(up(&L.p_ptr, h.p_ptr, A->bytes));
            NBX_TRY(up(&L.p_col, h.p_col, A->bytes));
            NBX_TRY(alloc(&L.p64, L.p_nnz, A->bytes));
            NBX_TRY(up(&L.w_ptr, h.w_ptr, A->bytes));
            NBX_TRY(up(&L.w_col, h.w_col, A->bytes));
            NBX_TRY(alloc(&L.w64, L.w_nnz, A->bytes));
            NBX_TRY(up(&L.pt_ptr, h.pt_ptr, A->bytes));
            NBX_TRY(up(&L.pt_row, h.pt_row, A->bytes));
            NBX_TRY(up(&L.pt_pos, h.pt_pos, A->bytes));
        }
    }
    // the last smoothed level in one workgroup with the dense solve
    if (nl >= 3 && bottom_fits(A->lv[nl - 2])) A->bottom = nl - 2;
    const uint32_t nco = A->lv.back().n;
    NBX_TRY(alloc(&A->cinv, (size_t)nco * nco, A->bytes));
    NBX_TRY(alloc(&A->ones, n, A->bytes));
    NBX_TRY(alloc(&A->pow_x, n, A->bytes));
    NBX_TRY(alloc(&A->pow_y, n, A->bytes));
    NBX_TRY(alloc(&A->scal, 2 * nl, A->bytes));
    NBX_TRY(alloc(&A->dense, 3 * (size_t)nco * nco + nco, A->bytes));
    NBX_TRY(alloc(&A->partials, (size_t)MAX_GRID, A->bytes));
    std::vector<double> ones(n + 2, 1.0);
    NBX_HIP(hipMemcpy(A->ones, ones.data(), ones.size() * sizeof(double), hipMemcpyHostToDevice));
    NBX_TRY(alloc(&A->differ, 1, A->bytes));
    std::swap(A->nzbits, dbits.d);
    return NBX_OK;
}

// Whether K's current entries (their nonzeros: the mesh stays) are the ones
// the hierarchy was built from, so that building it again would give the same.
static int amg_same_entries(FemSys& S, bool* same) {
    *same = false;
    const AmgDev* A = S.K.amg;
    if (!A || !A->nzbits) return NBX_OK;
    uint32_t differ = 0;
    NBX_HIP(hipMemcpyAsync(A->differ, &differ, sizeof differ, hipMemcpyHostToDevice, S.s));
    hipLaunchKernelGGL(k_block_nzbits_differ, dim3(grid_for(S.K.s.n_blocks)), dim3(BLOCK), 0, S.s,
                       S.K.s, A->nzbits, A->differ);
    NBX_HIP(hipGetLastError());
    NBX_HIP(copy_on(&differ, A->differ, sizeof differ, hipMemcpyDeviceToHost, S.s));
    *same = differ == 0;
    return NBX_OK;
}

// f(LANES, PHYS) for a block layout: the lanes a row's sum is formed by, and
// the lanes that form it.  Large levels are bound by bytes: there one lane
// takes a row, so that a wavefront reads 256 bytes in a row of each plane
// instead of 32 or 64 (2048x1024: the finest restriction 51.5 -> 44 us, level
// 1's products 5% less, 586 -> 572 us per outer iteration, 1024x512 239 -> 231).
// Smaller levels need the wavefronts.
template <class F>
static void with_bl(const BellDev& B, F&& f) {
    std::integral_constant<int, 1> one;
    const bool large = B.rows >= BELL_LARGE;
    auto go = [&](auto ln) {
        if (large)
            f(ln, one);
        else
            f(ln, ln);
    };
    switch (B.lanes) {
        case 1: f(one, one); break;
        case 2: go(std::integral_constant<int, 2>{}); break;
        case 4: go(std::integral_constant<int, 4>{}); break;
        case 8: go(std::integral_constant<int, 8>{}); break;
        default: f(std::integral_constant<int, 16>{}, std::integral_constant<int, 16>{}); break;
    }
}
// f(integral_constant R) for a level's rows per node
template <class F>
static void with_bs(uint32_t bs, F&& f) {
    if (bs == 2)
        f(std::integral_constant<int, 2>{});
    else
        f(std::integral_constant<int, 3>{});
}

// f(integral_constant LANES) for the numeric phase's products: lanes per
// output block, more on the small levels (0 blocks: one lane)
template <class F>
static void with_out_lanes(size_t blocks, F&& f) {
    if (blocks == 0)
        f(std::integral_constant<int, 1>{});
    else if (blocks >= (size_t)1 << 14)
        f(std::integral_constant<int, 4>{});
    else
        f(std::integral_constant<int, 16>{});
}

// cinv of the coarsest level's current values
template <int NB>
static void launch_sweep(AmgDev* A, uint32_t n, hipStream_t s) {
    if constexpr (NB < SWEEP_NB)
        if (n > NB * SWEEP_SIDE) return launch_sweep<NB + 1>(A, n, s);
    hipLaunchKernelGGL(k_dense_sweep<NB>, dim3(1), dim3(SWEEP_TB), 0, s, A->dense,
                       A->dense + (size_t)n * n, n);
}
static int coarsest_inverse(AmgDev* A, hipStream_t s) {
    const AmgDevLevel& L = A->lv.back();
    if (!L.n) return NBX_OK;
    hipLaunchKernelGGL(k_dense_rows, dim3(L.n), dim3(WAVE), 0, s, L.a_ptr, L.a_col, L.a64, A->dense,
                       L.n);
    launch_sweep<1>(A, L.n, s);
    double *const x = A->dense + (size_t)L.n * L.n, *const r = x + (size_t)L.n * L.n;
    uint32_t* const far = (uint32_t*)(r + (size_t)L.n * L.n);
    const dim3 rows(L.n), tb(REFINE_PARTS * BLOCK);
    hipLaunchKernelGGL(k_dense_residual, rows, tb, 0, s, A->dense, x, r, far, L.n);
    hipLaunchKernelGGL(k_dense_refine, rows, tb, 0, s, x, r, far, A->cinv, L.n);
    NBX_HIP(hipGetLastError());
    return NBX_OK;
}

// Numeric phase for the current values of K.
static int amg_numeric(FemSys& S) {
    AmgDev* A = S.K.amg;
    const hipStream_t s = S.s;
    AmgDevLevel& L0 = A->lv[0];
    hipLaunchKernelGGL(k_amg_fine_vals, dim3(grid_for(S.K.s.n_blocks)), dim3(BLOCK), 0, s, S.K.s,
                       L0.a_ptr, L0.a64);
    NBX_HIP(hipGetLastError());
    for (size_t l = 0; l < A->lv.size(); ++l) {
        AmgDevLevel& L = A->lv[l];
        const unsigned g = grid_for(L.n);
        hipLaunchKernelGGL(k_amg_dinv, dim3(g), dim3(BLOCK), 0, s, L.a_ptr, L.a_col, L.a64,
                           L.dinv64, L.dinv32, L.n);
        // (the finest level's smoothing reads the fp16 scaled copy; the
        // coarser levels' operators are filled in block form by the level
        // above)
        if (l + 1 == A->lv.size()) break;
        // lambda_max(D^-1 A): POW_STEPS power steps from a fixed start, x.x = n
        // (the coarsest level, solved directly, needs none)
        hipLaunchKernelGGL(k_amg_pow_init, dim3(g), dim3(BLOCK), 0, s, A->pow_x, L.n);
        double *px = A->pow_x, *py = A->pow_y, *scal = A->scal + 2 * l;
        const unsigned gp = std::min<size_t>(grid_for((size_t)L.n * POW_LANES), (size_t)MAX_GRID);
        const bool fold = gp <= ALL_PARTS;
        const double s0 = 1.0 / sqrt((double)L.n);
        for (int it = 0; it < POW_STEPS; ++it) {
            double* const part = A->partials + (fold ? (it & 1) * ALL_PARTS : 0);
            const double* const prev =
                fold && it ? A->partials + ((it - 1) & 1) * ALL_PARTS : nullptr;
            hipLaunchKernelGGL(k_amg_pow_step, dim3(gp), dim3(BLOCK), 0, s, L.a_ptr, L.a_col, L.a64,
                               L.dinv64, px, py, prev, it ? scal : nullptr, s0, part, L.n);
            if (!fold || it + 1 == POW_STEPS)
                hipLaunchKernelGGL(k_amg_pow_fin, dim3(1), dim3(FIN), 0, s, part, gp, scal);
            std::swap(px, py);
        }
        NBX_HIP(hipGetLastError());
        AmgDevLevel& C = A->lv[l + 1];
        with_bs(L.bs, [&](auto rr) {
            constexpr int R = decltype(rr)::value;
            hipLaunchKernelGGL(k_amg_smooth_p<R>,
                               dim3(grid_for((size_t)(L.n / R) * SMOOTH_SLOTS)), dim3(BLOCK), 0,
                               s, L.a_ptr, L.a_col, L.a64, L.dinv64, L.t, L.agg, L.p_ptr,
                               L.p_col, L.p64, scal + 1, L.n / R);
        });
        // P and P^T in block form (D^1/2 P on the finest level when it is
        // smoothed in the scaled variables)
        const double* pdis = l == 0 && A->scaled16 ? S.K.dis : nullptr;
        if (L.bs == 2) {
            hipLaunchKernelGGL((k_bell_fill<2, 3>), dim3(grid_for(L.pb.rows)), dim3(BLOCK), 0, s,
                               L.pb, L.p_ptr, L.p64, pdis);
            hipLaunchKernelGGL((k_bell_fill_t<2>), dim3(grid_for(L.tb.slots)), dim3(BLOCK), 0, s,
                               L.tb, (L.tb.rows + SLICE - 1) / SLICE, L.pt_ptr, L.pt_pos, L.p64,
                               pdis);
        } else {
            hipLaunchKernelGGL((k_bell_fill<3, 3>), dim3(grid_for(L.pb.rows)), dim3(BLOCK), 0, s,
                               L.pb, L.p_ptr, L.p64, pdis);
            hipLaunchKernelGGL((k_bell_fill_t<3>), dim3(grid_for(L.tb.slots)), dim3(BLOCK), 0, s,
                               L.tb, (L.tb.rows + SLICE - 1) / SLICE, L.pt_ptr, L.pt_pos, L.p64,
                               pdis);
        }
        const uint32_t nodes = L.n / L.bs, aggs = L.nc / 3;
        const size_t wblocks = L.w_nnz / (3 * L.bs), cblocks = C.a_nnz / 9;
        with_bs(L.bs, [&](auto rr) {
            constexpr int R = decltype(rr)::value;
            // (the finest level's W blocks sum about nine products each: one
            // lane per block measured fastest there)
            with_out_lanes(R == 2 ? 0 : wblocks, [&](auto ln) {
                constexpr int LN = decltype(ln)::value;
                hipLaunchKernelGGL((k_amg_w<R, LN>), dim3(grid_for(wblocks * LN)), dim3(BLOCK), 0,
                                   s, L.a_ptr, L.a_col, L.a64, L.p_ptr, L.p_col, L.p64, L.w_ptr,
                                   L.w_col, L.w64, nodes, wblocks);
            });
            with_out_lanes(cblocks, [&](auto ln) {
                constexpr int LN = decltype(ln)::value;
                hipLaunchKernelGGL((k_amg_galerkin<R, LN>), dim3(grid_for(cblocks * LN)),
                                   dim3(BLOCK), 0, s, L.pt_ptr, L.pt_row, L.pt_pos, L.p64, L.w_ptr,
                                   L.w_col, L.w64, C.a_ptr, C.a_col, C.a64, aggs, cblocks);
            });
        });
        if (C.ab.rows)
            hipLaunchKernelGGL((k_bell_fill<3, 3>), dim3(grid_for(C.ab.rows)), dim3(BLOCK), 0, s,
                               C.ab, C.a_ptr, C.a64, (const double*)nullptr);
        NBX_HIP(hipGetLastError());
    }
    NBX_TRY(coarsest_inverse(A, s));
    // the smoothers' coefficients, from all levels' lambda_max at once
    std::vector<double> scal(2 * A->lv.size());
    NBX_HIP(copy_on(scal.data(), A->scal, scal.size() * sizeof(double), hipMemcpyDeviceToHost, s));
    for (size_t l = 0; l + 1 < A->lv.size(); ++l) {
        AmgDevLevel& L = A->lv[l];
        L.lmax = scal[2 * l + 1];
        if (!(L.lmax > 0.0) || !std::isfinite(L.lmax)) {
            set_last_error("AMG: lambda_max(D^-1 A) of level %zu is %g", l, L.lmax);
            return NBX_ERR_BREAKDOWN;
        }
        const double hi = 1.1 * L.lmax, lo = L.lmax / 30.0;
        const double theta = 0.5 * (hi + lo), delta = 0.5 * (hi - lo), sigma = theta / delta;
        double rho = 1.0 / sigma;
        L.inv_theta = (float)(1.0 / theta);
        for (int k = 1; k < L.degree; ++k) {
            const double rn = 1.0 / (2.0 * sigma - rho);
            L.c1[k] = (float)(rn * rho);
            L.c2[k] = (float)(2.0 * rn / delta);
            rho = rn;
        }
    }
    return NBX_OK;
}

int amg_prepare(FemSys& S) {
    // New boundary conditions may eliminate other unknowns; where K's nonzero
    // entries are those of the last build (an optimisation that applies the
    // same supports to every new K), the hierarchy stands: 0.03 ms in place of
    // 21 ms of host work at 256x128.
    if (S.K.amg && !S.amg_symbolic_current)
        NBX_TRY(amg_same_entries(S, &S.amg_symbolic_current));
    if (!S.K.amg || !S.amg_symbolic_current) {
        // (the host arrays of a large system can exhaust host memory: an
        // error, not an exception through the C interface)
        int rc;
        try {
            rc = amg_symbolic(S);
        } catch (const std::bad_alloc&) {
            set_last_error("AMG: host memory ran out building the hierarchy");
            rc = NBX_ERR_ARG;
        }
        if (rc != NBX_OK) return rc;
        S.amg_symbolic_current = true;
    }
    if (!S.K.amg_current) {
        // the finest level's smoothing reads the fp16 Jacobi-scaled copy
        // (a FEM matrix always has one: its scaled entries lie in [-1, 1])
        AmgDev* A = S.K.amg;
        A->scaled16 = false;
        if (A->lv.size() > 1) {
            NBX_TRY(mat_make_off16(S.K, S.s));
            if (!S.K.has_off16 || !S.K.has_scale) {
                set_last_error("AMG: the matrix has no fp16 Jacobi-scaled copy for the finest "
                               "level's smoothing");
                return NBX_ERR_ARG;
            }
            A->scaled16 = true;
        }
        NBX_TRY(amg_numeric(S));
        S.K.amg_current = true;
    }
    return NBX_OK;
}

AmgFine amg_fine(const AmgDev* A) {
    AmgFine f;
    if (!A || !A->scaled16 || A->lv.size() < 2) return f;
    const AmgDevLevel& L = A->lv[0];
    f.scaled16 = true;
    const double hi = 1.1 * L.lmax, lo = L.lmax / 30.0;
    f.inv_theta = 1.0 / (0.5 * (hi + lo));
    f.c = L.d0;
    return f;
}

const double* amg_ones(const AmgDev* A) { return A->ones; }
uint32_t amg_levels(const AmgDev* A) { return (uint32_t)A->lv.size(); }


// b_{l+1} = P_l^T r_l, with the next level's smoothing start unless that
// level is the coarsest
static void restrict_to(AmgDev* A, size_t l, const float* r, const PcgState* st, hipStream_t s) {
    AmgDevLevel& V = A->lv[l];
    AmgDevLevel& W = A->lv[l + 1];
    const bool init = l + 2 < A->lv.size() && l + 1 != A->bottom && !W.tiles.n;
    with_bs(V.bs, [&](auto R) {
        constexpr int RR = decltype(R)::value;
        with_bl(V.tb, [&](auto ln, auto ph) {
            constexpr int LN = decltype(ln)::value, PH = decltype(ph)::value;
            const unsigned g = grid_for((size_t)V.tb.rows * PH);
            if (init)
                hipLaunchKernelGGL((k_brestrict<RR, true, LN, PH>), dim3(g), dim3(BLOCK), 0, s,
                                   bell<3, RR>(V.tb), r, W.b, W.dinv32, W.x, W.r, W.d0,
                                   W.inv_theta, st, V.tb.rows);
            else
                hipLaunchKernelGGL((k_brestrict<RR, false, LN, PH>), dim3(g), dim3(BLOCK), 0, s,
                                   bell<3, RR>(V.tb), r, W.b, W.dinv32, W.x, W.r, W.d0,
                                   W.inv_theta, st, V.tb.rows);
        });
    });
}

// x_l (+)= P_l x_{l+1}
static void prolong_from(AmgDev* A, size_t l, float* x, bool add, const PcgState* st,
                         hipStream_t s) {
    AmgDevLevel& V = A->lv[l];
    const float* xc = A->lv[l + 1].out();
    with_bs(V.bs, [&](auto R) {
        constexpr int RR = decltype(R)::value;
        with_bl(V.pb, [&](auto ln, auto ph) {
            constexpr int LN = decltype(ln)::value, PH = decltype(ph)::value;
            const unsigned g = grid_for((size_t)V.pb.rows * PH);
            if (add)
                hipLaunchKernelGGL((k_bprolong<RR, true, LN, PH>), dim3(g), dim3(BLOCK), 0, s,
                                   bell<RR, 3>(V.pb), xc, x, st, V.pb.rows);
            else
                hipLaunchKernelGGL((k_bprolong<RR, false, LN, PH>), dim3(g), dim3(BLOCK), 0, s,
                                   bell<RR, 3>(V.pb), xc, x, st, V.pb.rows);
        });
    });
}

static BottomLevel level_args(const AmgDevLevel& V) {
    BottomLevel L{};
    L.A = bell<3, 3>(V.ab);
    L.P = bell<3, 3>(V.pb);
    L.T = bell<3, 3>(V.tb);
    L.dinv = V.dinv32;
    L.p_lanes = V.pb.lanes;
    L.t_lanes = V.tb.lanes;
    L.rows = V.n / 3;
    L.degree = (uint32_t)V.degree;
    L.inv_theta = V.inv_theta;
    std::copy(V.c1, V.c1 + AMG_MAX_DEGREE, L.c1);
    std::copy(V.c2, V.c2 + AMG_MAX_DEGREE, L.c2);
    return L;
}

static void tile_down(const AmgDevLevel& V, const float* b, float* x, const PcgState* st,
                      hipStream_t s) {
    const size_t lds = 9 * (size_t)V.tiles.most * sizeof(float);
    with_row_form(V, 3 * V.tiles.most, [&](auto tb, auto held, auto ln) {
        constexpr int TB = decltype(tb)::value, HELD = decltype(held)::value;
        hipLaunchKernelGGL((k_amg_down<TB, HELD, decltype(ln)::value>), dim3(V.tiles.n), dim3(TB),
                           lds, s, level_args(V), V.tiles, b, x, V.r, st);
    });
}
static void tile_up(const AmgDevLevel& V, const float* b, const float* x, const float* xc,
                    const PcgState* st, hipStream_t s) {
    const size_t lds = 9 * (size_t)V.tiles.most * sizeof(float);
    with_row_form(V, 3 * V.tiles.most, [&](auto tb, auto held, auto ln) {
        constexpr int TB = decltype(tb)::value, HELD = decltype(held)::value;
        hipLaunchKernelGGL((k_amg_up<TB, HELD, decltype(ln)::value>), dim3(V.tiles.n), dim3(TB),
                           lds, s, level_args(V), V.tiles, b, x, xc, V.d0, st);
    });
}

// The one-workgroup part: level A->bottom and the dense solve below it.
static void bottom_cycle(AmgDev* A, const float* b, float* x, const PcgState* st, hipStream_t s) {
    Bottom B{};
    const AmgDevLevel& C = A->lv.back();
    const AmgDevLevel& V = A->lv[A->bottom];
    B.lv = level_args(V);
    B.nco = C.n;
    B.cinv = A->cinv;
    B.b = b;
    B.x = x;
    const size_t lds = (4 * (size_t)V.n + 2 * (size_t)C.n) * sizeof(float);
    with_row_form(V, V.n, [&](auto tb, auto held, auto ln) {
        constexpr int TB = decltype(tb)::value, HELD = decltype(held)::value;
        hipLaunchKernelGGL((k_amg_bottom<TB, HELD, decltype(ln)::value>), dim3(1), dim3(TB), lds, s,
                           B, st);
    });
}

// The V-cycle from level l0 >= 1 down, x = M^-1 b on that level (b, x: that
// level's arrays; the finest level is smoothed by the flexible CG's own
// kernels on the fp16 copy).  The restriction has already started the
// pre-smoothing (r, d0, x) of each level that takes a launch per step; levels
// on tiles take two launches, and the last ones one workgroup.  A level's
// correction is in its out().  A one-level hierarchy is its dense solve alone
// (l0 = 0).
static void cycle_from(AmgDev* A, size_t l0, const float* b, float* x, const PcgState* st,
                       hipStream_t s) {
    const size_t L = A->lv.size();
    const size_t low = A->bottom ? std::max(A->bottom, l0) : L - 1;   // the last part's level
    for (size_t l = l0; l < low; ++l) {
        AmgDevLevel& V = A->lv[l];
        const float* bl = l == l0 ? b : V.b;
        float* xl = l == l0 ? x : V.x;
        if (V.tiles.n) {
            tile_down(V, bl, xl, st, s);
            restrict_to(A, l, V.r, st, s);
            continue;
        }
        float *din = V.d0, *dout = V.d1;
        with_bl(V.ab, [&](auto ln, auto ph) {
            constexpr int LN = decltype(ln)::value, PH = decltype(ph)::value;
            const unsigned g = grid_for((size_t)V.ab.rows * PH);
            for (int k = 1; k < V.degree; ++k) {
                hipLaunchKernelGGL((k_bsm_step<false, LN, PH>), dim3(g), dim3(BLOCK), 0, s,
                                   bell<3, 3>(V.ab), V.dinv32, din, dout, V.r, xl, V.c1[k],
                                   V.c2[k], st, V.ab.rows);
                std::swap(din, dout);
            }
            hipLaunchKernelGGL((k_bresidual<LN, PH>), dim3(g), dim3(BLOCK), 0, s, bell<3, 3>(V.ab), bl,
                               xl, V.r, st, V.ab.rows);
        });
        restrict_to(A, l, V.r, st, s);
    }
    if (A->bottom) {
        AmgDevLevel& V = A->lv[low];
        bottom_cycle(A, low == l0 ? b : V.b, low == l0 ? x : V.x, st, s);
    } else {
        AmgDevLevel& C = A->lv[L - 1];
        hipLaunchKernelGGL(k_amg_dense, dim3(1), dim3(DENSE_BLOCK), 0, s, A->cinv,
                           L == l0 + 1 ? b : C.b, L == l0 + 1 ? x : C.x, st, C.n);
    }
    for (size_t l = low; l-- > l0;) {
        AmgDevLevel& V = A->lv[l];
        const float* bl = l == l0 ? b : V.b;
        float* xl = l == l0 ? x : V.x;
        if (V.tiles.n) {
            tile_up(V, bl, xl, A->lv[l + 1].out(), st, s);
            continue;
        }
        prolong_from(A, l, xl, true, st, s);
        float *din = V.d0, *dout = V.d1;
        with_bl(V.ab, [&](auto ln, auto ph) {
            constexpr int LN = decltype(ln)::value, PH = decltype(ph)::value;
            const unsigned g = grid_for((size_t)V.ab.rows * PH);
            hipLaunchKernelGGL((k_bsm_init<LN, PH>), dim3(g), dim3(BLOCK), 0, s, bell<3, 3>(V.ab),
                               V.dinv32, bl, xl, V.r, V.d0, V.inv_theta, st, V.ab.rows);
            for (int k = 1; k < V.degree; ++k) {
                if (k == 1)
                    hipLaunchKernelGGL((k_bsm_step<true, LN, PH>), dim3(g), dim3(BLOCK), 0, s,
                                       bell<3, 3>(V.ab), V.dinv32, din, dout, V.r, xl, V.c1[k],
                                       V.c2[k], st, V.ab.rows);
                else
                    hipLaunchKernelGGL((k_bsm_step<false, LN, PH>), dim3(g), dim3(BLOCK), 0, s,
                                       bell<3, 3>(V.ab), V.dinv32, din, dout, V.r, xl, V.c1[k],
                                       V.c2[k], st, V.ab.rows);
                std::swap(din, dout);
            }
        });
    }
}

// z = C^-1 r for a one-level hierarchy (the finest level is the coarsest)
int amg_vcycle(AmgDev* A, const float* b, float* x, const PcgState* st, hipStream_t s) {
    if (A->lv.size() != 1) {
        set_last_error("AMG: the V-cycle of a multi-level hierarchy runs on the fp16 copy");
        return NBX_ERR_ARG;
    }
    cycle_from(A, 0, b, x, st, s);
    NBX_HIP(hipGetLastError());
    return NBX_OK;
}

int amg_coarse_correction(AmgDev* A, const float* r, float* c, const PcgState* st,
                          hipStream_t s) {
    restrict_to(A, 0, r, st, s);
    cycle_from(A, 1, A->lv[1].b, A->lv[1].x, st, s);
    prolong_from(A, 0, c, false, st, s);
    NBX_HIP(hipGetLastError());
    return NBX_OK;
}

}  // namespace nbx
