// Conjugate-gradient solvers for gfx950, device resident.
//
// * Jacobi-preconditioned CG with the reference's recurrences and stop test
//   (solver_bot/sparse/solvers/cg_precond_jacobi.c:13-90).  Three kernels per
//   iteration: SpMV + p.w, the g update + g.q and g.g, and the x and
//   direction update (x += alpha p reads the p that the direction update
//   reads anyway, so the vectors cross HBM 12 times per iteration, not 13).
//   Reducing kernels write one partial per workgroup; a one-workgroup
//   finalize kernel sums them in index order and computes alpha, beta and the
//   stop decision on the GPU (runs are reproducible, and no device-scope fence
//   or atomic sits in the loop); the host only polls a done flag between
//   batches of iterations.  Small and medium systems take two kernels per
//   iteration, whose workgroups each add the partials themselves (k_cg_dir).
// * Mixed precision: CG on the Jacobi-scaled FP32 copy D^-1/2 K D^-1/2 with
//   FP32 vectors and compensated FP32 dot products, and FP64 reliable updates
//   (Sleijpen & van der Vorst 1996): when the iterated residual has dropped
//   by delta, the FP32 correction is folded into the FP64 solution u, the
//   true residual b - K u is recomputed with the FP64 matrix, and the FP32
//   recurrence continues from it without restarting the Krylov directions.
//   A restarted variant (inner tolerance per sweep) is kept for comparison.
//   CG on the symmetrically Jacobi-scaled system is Jacobi-PCG in other
//   variables.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>
#include <string.h>
#include <algorithm>
#include <type_traits>
#include <vector>

#include "rows.hpp"

namespace nbx {

// ---------------------------------------------------------------------------
// FP64 Jacobi PCG, reference semantics
// ---------------------------------------------------------------------------
// init: g = A x - b; q = g / Aii; p = -q; gg = g.g; rz = g.q
//   (cg_precond_jacobi.c:33-43)
template <class Op>
__global__ __launch_bounds__(BLOCK) void k_pcg_init(Op op, const typename Op::V* __restrict__ b,
                                                    const typename Op::V* __restrict__ x,
                                                    typename Op::V* __restrict__ g,
                                                    typename Op::V* __restrict__ p,
                                                    const typename Op::V* __restrict__ diag,
                                                    PcgState* st, double* partials, uint32_t n) {
    using V = typename Op::V;
    double acc[2] = {0.0, 0.0};
    const Chunk c = my_chunk(n);
    for (size_t u = c.beg + threadIdx.x; u < c.end; u += BLOCK) {
        const V gv = subu(op.row((uint32_t)u, x), b[u]);
        const V q = divu(gv, diag[u]);
        g[u] = gv;
        p[u] = negu(q);
        acc[0] += dotu(gv, gv);
        acc[1] += dotu(gv, q);
    }
    __shared__ double red[2][BLOCK / WAVE];
    block_sum<2>(acc, red);
    put_partials<2>(acc, partials);
}

__global__ __launch_bounds__(FIN) void k_fin_init(PcgState* st, const double* partials, unsigned np) {
    double tot[2];
    fin_sum<2>(partials, np, tot);
    if (threadIdx.x == 0) {
        const double gg = tot[0];
        st->rz = tot[1];
        st->gg_cur = gg;
        st->gg_prev = gg;
        st->gg0 = gg;
        st->k = 0;
        if (!(gg > st->tol2 && 0u < st->max_iter)) {
            st->done = 1;
            st->tol_reached = sqrt(gg);
            st->status = gg > st->tol2 ? 1u : 0u;
        }
    }
}

// w = A p; pw = p.w; alpha = rz / pw   (cg_precond_jacobi.c:50-59)
template <class Op>
__global__ __launch_bounds__(BLOCK) void k_pcg_A(Op op, const typename Op::V* __restrict__ p,
                                                 typename Op::V* __restrict__ w, PcgState* st,
                                                 double* partials, uint32_t n) {
    if (st->done) return;
    double acc[1] = {0.0};
    const Chunk c = my_chunk(n);
    for (size_t u = c.beg + threadIdx.x; u < c.end; u += BLOCK) {
        const typename Op::V wv = op.row((uint32_t)u, p);
        w[u] = wv;
        acc[0] += dotu(p[u], wv);
    }
    __shared__ double red[1][BLOCK / WAVE];
    block_sum<1>(acc, red);
    put_partials<1>(acc, partials);
}

// The finalize kernels read the state they need together with the partials
// and test `done` afterwards: one memory round trip instead of three in a
// row (state, partials, state).  The partials buffer holds 4 x MAX_GRID
// values, so the reads stay in it whatever the state says; a finished
// solve ignores the sums.
__global__ __launch_bounds__(FIN) void k_fin_A(PcgState* st, const double* partials, unsigned np) {
    const uint32_t done = st->done, j = st->k;   // this is iteration j
    const double rz = st->rz;
    double tot[1];
    fin_sum<1>(partials, np, tot);
    if (done) return;
    if (threadIdx.x == 0) {
        st->pw = tot[0];
        st->alpha = rz / tot[0];
        st->alpha_hist[j & 3u] = st->alpha;
    }
}

__global__ __launch_bounds__(FIN) void k_fin_B(PcgState* st, const double* partials, unsigned np) {
    const uint32_t done = st->done, k = st->k + 1, max_iter = st->max_iter;
    const double rz = st->rz, gg_prev = st->gg_cur, tol2 = st->tol2;
    double tot[2];
    fin_sum<2>(partials, np, tot);
    if (done) return;
    if (threadIdx.x == 0) {
        st->beta = tot[0] / rz;
        st->rz = tot[0];
        st->gg_prev = gg_prev;
        st->gg_cur = tot[1];
        st->k = k;
        if (!(gg_prev > tol2 && k < max_iter)) {
            st->done = 1;
            st->tol_reached = sqrt(gg_prev);
            st->status = gg_prev > tol2 ? 1u : 0u;
        }
    }
}

// g += alpha w; q = g / Aii; rz' = g.q; gg' = g.g, then the lagged stop test
// (cg_precond_jacobi.c:63-70, :75); x is left to the direction kernel.
template <class V, bool NT>
__global__ __launch_bounds__(BLOCK) void k_pcg_B(V* __restrict__ g, const V* __restrict__ w,
                                                  const V* __restrict__ diag, PcgState* st,
                                                  double* partials, uint32_t n) {
    if (st->done) return;
    const double alpha = st->alpha;
    double acc[2] = {0.0, 0.0};
    const Chunk c = my_chunk(n);
    for (size_t u = c.beg + threadIdx.x; u < c.end; u += BLOCK) {
        const V gv = axpyu(ldv<NT>(&g[u]), alpha, ldv<NT>(&w[u]));
        stv<NT>(&g[u], gv);
        const V q = divu(gv, ldv<NT>(&diag[u]));
        acc[0] += dotu(gv, q);
        acc[1] += dotu(gv, gv);
    }
    __shared__ double red[2][BLOCK / WAVE];
    block_sum<2>(acc, red);
    put_partials<2>(acc, partials);
}

// The four direction buffers of the FP64 PCG: p_j lives in p[j % 4].
template <class V>
struct PBufs {
    V* p[4];
};

// p_{j+1} = -q + beta p_j  (cg_precond_jacobi.c:72-74) into the next of four
// direction buffers, and x += alpha p (:62) for four iterations at a time:
// iteration j reads p_j from buffer j % 4 and writes p_{j+1} into buffer
// (j + 1) % 4, which still holds p_{j-3}.  Iterations j % 4 = 0, 1, 2 leave
// x alone; iteration j % 4 = 3 (FLUSH) applies
// x = (((x + a_{j-3} p_{j-3}) + a_{j-2} p_{j-2}) + a_{j-1} p_{j-1}) + a_j p_j,
// the same roundings in the same order as one update per iteration, so x is
// bit-identical, and x is read and written every fourth iteration only.
// Once the stop test has fired this kernel no longer runs, and k_pcg_tail
// applies the updates still pending.
template <class V, bool NT, bool FLUSH>
__global__ __launch_bounds__(BLOCK) void k_pcg_C(V* __restrict__ x, PBufs<V> P, uint32_t j,
                                                  const V* __restrict__ g,
                                                  const V* __restrict__ diag, PcgState* st,
                                                  uint32_t n) {
    if (st->done) return;
    const double alpha = st->alpha, beta = st->beta;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    if constexpr (FLUSH) {
        a0 = st->alpha_hist[0];
        a1 = st->alpha_hist[1];
        a2 = st->alpha_hist[2];
    }
    const V* __restrict__ p = P.p[j & 3u];
    V* __restrict__ p_next = P.p[(j + 1) & 3u];
    const Chunk c = my_chunk(n);
    for (size_t u = c.beg + threadIdx.x; u < c.end; u += BLOCK) {
        const V pu = ldv<NT>(&p[u]);
        if constexpr (FLUSH) {
            // j % 4 = 3: p_{j-3} is in p_next (read before p_{j+1} replaces
            // it), p_{j-2} in P.p[1], p_{j-1} in P.p[2]
            V xv = ldv<NT>(&x[u]);
            xv = axpyu(xv, a0, ldv<NT>(&p_next[u]));
            xv = axpyu(xv, a1, ldv<NT>(&P.p[1][u]));
            xv = axpyu(xv, a2, ldv<NT>(&P.p[2][u]));
            stv<NT>(&x[u], axpyu(xv, alpha, pu));
        }
        const V q = divu(ldv<NT>(&g[u]), ldv<NT>(&diag[u]));
        p_next[u] = pupd(q, beta, pu);   // gathered by the next SpMV: cached store
    }
}

// The x updates still pending when the loop has stopped (cg_precond_jacobi.c:
// 62): iteration J = k - 1 did not reach k_pcg_C, and the updates of the
// iterations 4 floor(J / 4) .. J are pending, applied in ascending order.
// Nothing if no iteration ran.
template <class V>
__global__ __launch_bounds__(BLOCK) void k_pcg_tail(V* __restrict__ x, PBufs<V> P,
                                                    const PcgState* st, uint32_t n) {
    const uint32_t k = st->k;
    if (k == 0) return;
    const uint32_t last = (k - 1) & 3u;   // buffers 0 .. last hold p of the pending ones
    const Chunk c = my_chunk(n);
    for (size_t u = c.beg + threadIdx.x; u < c.end; u += BLOCK) {
        V xv = x[u];
        for (uint32_t i = 0; i <= last; ++i) xv = axpyu(xv, st->alpha_hist[i], P.p[i][u]);
        x[u] = xv;
    }
}

// ---------------------------------------------------------------------------
// FP64 Jacobi PCG in two kernels per iteration (small and medium systems)
// ---------------------------------------------------------------------------
// Up to a few hundred thousand rows an iteration of the five kernels above is
// bound by their launches and by the chains of dependent loads in each (3-4
// us a kernel), not by bytes.  Two kernels do the same iteration:
//   k_cg_dir     sums the previous update's partials (g.q and g.g), which
//                gives beta and the stop decision; forms p_j = -q + beta
//                p_{j-1} of a row and of its neighbours on the fly, stores
//                its own, w = A p_j and the partials of p_j.w;
//   k_cg_update  sums those, which gives alpha; x += alpha p, g += alpha w,
//                q = g / Aii and the partials of g.q and g.g.
// Every workgroup sums all partials itself, in the same order, so all have
// the same scalars and no one-workgroup kernel stands between (G partials
// read by G workgroups: at most 1,024 of each, a few us of L2 traffic at the
// largest).  k_cg_dir issues its row's loads before that sum, whose latency
// then hides them.  The state alternates between two slots: a launch reads
// one and its first workgroup writes the other, so no workgroup reads what
// another one of the same launch writes.  Products, vectors, sums (a partial
// per 256 rows, wave sums of 64 partials, those in index order) and the stop
// test are formed by the same operations in the same order as in the five
// kernels, so the results are the same bit for bit.

// q of the coming direction and the direction before it, side by side: the
// product gathers both of a neighbour in one place.
template <class V>
struct __attribute__((aligned(16))) CgPair {
    V q, p;
};

// p_j of one row from q and p_{j-1}
struct CgDir {
    double beta;
    bool first;
    template <class V>
    __device__ __forceinline__ V operator()(const CgPair<V>& d) const {
        return first ? negu(d.q) : pupd(d.q, beta, d.p);
    }
};

// beta and the stop decision before iteration k (the test of k_fin_init and
// k_fin_B) from the sums of the update before it; false when the solve has
// ended.  Called by every thread of every workgroup, with the same results.
__device__ __forceinline__ bool cg_next(const PcgState* __restrict__ sin, PcgState* sout,
                                        const AllSum<2>& upd, bool first,
                                        double (*red)[ALL_PARTS / WAVE], CgDir& dir) {
    const uint32_t ended = sin->done, max_iter = sin->max_iter;
    const uint32_t k = first ? 0u : sin->k + 1u;
    const double tol2 = sin->tol2, rz = sin->rz, gg_cur = sin->gg_cur;
    double tot[2];
    upd.total(gridDim.x, tot, red);
    const double gg_prev = first ? tot[1] : gg_cur;
    const bool go = gg_prev > tol2 && k < max_iter;
    dir.beta = first ? 0.0 : tot[0] / rz;
    dir.first = first;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sout->tol2 = tol2;
        sout->max_iter = max_iter;
        sout->gg0 = first ? tot[1] : sin->gg0;
        if (ended) {   // (the state goes on from slot to slot)
            sout->k = sin->k;
            sout->done = 1;
            sout->status = sin->status;
            sout->tol_reached = sin->tol_reached;
        } else {
            sout->k = k;
            sout->beta = dir.beta;
            sout->rz = tot[0];
            sout->gg_prev = gg_prev;
            sout->gg_cur = tot[1];
            sout->done = go ? 0u : 1u;
            sout->status = gg_prev > tol2 ? 1u : 0u;
            sout->tol_reached = sqrt(gg_prev);
        }
    }
    return !ended && go;
}

// The flexible CG's direction: p = z + beta p (p = z on the first step), beta
// and the restart from the sums (z.w, r.z) as k_fin_fcg_dots forms them.
struct FcgDir {
    double beta;
    bool first;
    __device__ __forceinline__ double2 operator()(const CgPair<double2>& d) const {
        return first ? d.q : axpyu(d.q, beta, d.p);
    }
};
__device__ __forceinline__ bool cg_next(const PcgState* __restrict__ sin, PcgState* sout,
                                        const AllSum<2>& dots, bool first,
                                        double (*red)[ALL_PARTS / WAVE], FcgDir& dir) {
    const uint32_t ended = sin->done;
    const double alpha = sin->alpha, rz_old = sin->rz;
    double tot[2];
    dots.total(gridDim.x, tot, red);
    const double rz = tot[1];
    dir.beta = first ? 0.0 : -alpha * tot[0] / rz_old;
    dir.first = first;
    const bool restart = !(rz > 0.0) || !isfinite(rz) || !isfinite(dir.beta);
    if (restart) dir.beta = 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sout->done = ended;
        if (!ended) {
            sout->k = sin->k;
            sout->max_iter = sin->max_iter;
            sout->tol2 = sin->tol2;
            sout->gg0 = sin->gg0;
            sout->beta = dir.beta;
            sout->rz = rz;
            sout->breakdown = sin->breakdown + (restart ? 1u : 0u);
        }
    }
    return !ended;
}

// A row's loads ahead of beta, then the product with p formed on the fly;
// blocks beyond the ones held ahead are loaded MORE at a time when they are
// used.  us per iteration with five kernels, with the rest of a row a block at
// a time and MORE at a time: symmetric, 10,000 nodes of 101 blocks 39.5, 42.2,
// 33.0; 60,000 of 51 38.2, 47.7, 32.6; 120,000 of 27 36.8, 39.1, 34.8; full
// rows, 10,000 of 101 45.2, 57.2, 34.1; 120,000 of 27 38.7, 34.8, 32.9.
constexpr int MORE = 4;
template <class Op>
struct CgRow;
// the symmetric copy, with U lower and U upper blocks loaded ahead
template <int U>
struct OpSymU : OpSymC {};
template <>
struct CgRow<OpS2> {
    static constexpr int U = 7;   // an interior row of a T3 mesh
    const Sell2& A;
    size_t base = 0;
    int len = 0;
    uint32_t w[U];
    dv2 a[U], b[U];
    CgPair<double2> x[U];
    __device__ __forceinline__ void load(uint32_t v, const CgPair<double2>* __restrict__ d) {
        const dv2* __restrict__ pa = reinterpret_cast<const dv2*>(A.val);
        const dv2* __restrict__ pb = reinterpret_cast<const dv2*>(A.val + 2 * A.n_blocks);
        base = (size_t)A.slice_ptr[v >> 6] + (v & 63);
        len = A.rowlen[v];
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (k < len) {
                const size_t i = base + (size_t)k * SLICE;
                w[k] = A.bcol[i];
                a[k] = pa[i];
                b[k] = pb[i];
            }
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (k < len) x[k] = d[w[k]];
    }
    template <class D>
    __device__ __forceinline__ double2 product(const D& dir, double2,
                                               const CgPair<double2>* __restrict__ d) const {
        double s0 = 0.0, s1 = 0.0;
        auto add = [&](dv2 ka, dv2 kb, double2 v) {
            s0 = s0 + ka.x * v.x;
            s0 = s0 + ka.y * v.y;
            s1 = s1 + kb.x * v.x;
            s1 = s1 + kb.y * v.y;
        };
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (k < len) add(a[k], b[k], dir(x[k]));
        const dv2* __restrict__ pa = reinterpret_cast<const dv2*>(A.val);
        const dv2* __restrict__ pb = reinterpret_cast<const dv2*>(A.val + 2 * A.n_blocks);
        for (int k0 = U; k0 < len; k0 += MORE) {
            uint32_t wk[MORE];
            dv2 ka[MORE], kb[MORE];
            CgPair<double2> xk[MORE];
#pragma unroll
            for (int k = 0; k < MORE; ++k)
                if (k0 + k < len) {
                    const size_t i = base + (size_t)(k0 + k) * SLICE;
                    wk[k] = A.bcol[i];
                    ka[k] = pa[i];
                    kb[k] = pb[i];
                }
#pragma unroll
            for (int k = 0; k < MORE; ++k)
                if (k0 + k < len) xk[k] = d[wk[k]];
#pragma unroll
            for (int k = 0; k < MORE; ++k)
                if (k0 + k < len) add(ka[k], kb[k], dir(xk[k]));
        }
        return make_double2(s0, s1);
    }
};
template <int U>
struct CgRow<OpSymU<U>> {
    const Sym2& Y;
    size_t lbase = 0, ubase = 0;
    int llen = 0, ulen = 0;
    dv2 d01;
    double d11;
    uv2 e[U];
    uint32_t w[U];
    dv2 la[U], lb[U], ua[U], ub[U];
    CgPair<double2> lx[U], ux[U];
    __device__ __forceinline__ void load(uint32_t v, const CgPair<double2>* __restrict__ d) {
        const dv2* __restrict__ pa = reinterpret_cast<const dv2*>(Y.u_val);
        const dv2* __restrict__ pb = reinterpret_cast<const dv2*>(Y.u_val + 2 * Y.n_upper);
        const uv2* __restrict__ li = reinterpret_cast<const uv2*>(Y.l_idx);
        d01 = reinterpret_cast<const dv2*>(Y.d_val)[v];
        d11 = Y.d_val[2 * (size_t)Y.n_nodes + v];
        llen = Y.l_rowlen[v];
        ulen = Y.u_rowlen[v];
        // the entries to hold: the row's own, or, where every slice is as wide
        // as the widest row, the slice's, without waiting for the row length
        int ln = llen, un = ulen;
        if (Y.l_width) {
            lbase = (size_t)(v >> 6) * SLICE * Y.l_width + (v & 63);
            ln = (int)Y.l_width;
        } else {
            lbase = (size_t)Y.l_slice_ptr[v >> 6] + (v & 63);
        }
        if (Y.u_width) {
            ubase = (size_t)(v >> 6) * SLICE * Y.u_width + (v & 63);
            un = (int)Y.u_width;
        } else {
            ubase = (size_t)Y.u_slice_ptr[v >> 6] + (v & 63);
        }
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (k < ln) e[k] = li[lbase + (size_t)k * SLICE];
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (k < un) {
                const size_t i = ubase + (size_t)k * SLICE;
                w[k] = Y.u_bcol[i];
                ua[k] = pa[i];
                ub[k] = pb[i];
            }
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (k < ln) {
                la[k] = pa[e[k].y];
                lb[k] = pb[e[k].y];
                lx[k] = d[e[k].x];
            }
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (k < un) ux[k] = d[w[k]];
    }
    template <class D>
    __device__ __forceinline__ double2 product(const D& dir, double2 pd,
                                               const CgPair<double2>* __restrict__ d) const {
        const dv2* __restrict__ pa = reinterpret_cast<const dv2*>(Y.u_val);
        const dv2* __restrict__ pb = reinterpret_cast<const dv2*>(Y.u_val + 2 * Y.n_upper);
        const uv2* __restrict__ li = reinterpret_cast<const uv2*>(Y.l_idx);
        double s0 = 0.0, s1 = 0.0;
        auto lower = [&](dv2 a, dv2 b, double2 v) {   // [[a.x, b.x], [a.y, b.y]]
            s0 = s0 + a.x * v.x;
            s0 = s0 + b.x * v.y;
            s1 = s1 + a.y * v.x;
            s1 = s1 + b.y * v.y;
        };
        auto upper = [&](dv2 a, dv2 b, double2 v) {
            s0 = s0 + a.x * v.x;
            s0 = s0 + a.y * v.y;
            s1 = s1 + b.x * v.x;
            s1 = s1 + b.y * v.y;
        };
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (k < llen) lower(la[k], lb[k], dir(lx[k]));
        for (int k0 = U; k0 < llen; k0 += MORE) {
            uv2 ck[MORE];
            dv2 ka[MORE], kb[MORE];
            CgPair<double2> xk[MORE];
#pragma unroll
            for (int k = 0; k < MORE; ++k)
                if (k0 + k < llen) ck[k] = li[lbase + (size_t)(k0 + k) * SLICE];
#pragma unroll
            for (int k = 0; k < MORE; ++k)
                if (k0 + k < llen) {
                    ka[k] = pa[ck[k].y];
                    kb[k] = pb[ck[k].y];
                    xk[k] = d[ck[k].x];
                }
#pragma unroll
            for (int k = 0; k < MORE; ++k)
                if (k0 + k < llen) lower(ka[k], kb[k], dir(xk[k]));
        }
        s0 = s0 + d01.x * pd.x;
        s0 = s0 + d01.y * pd.y;
        s1 = s1 + d01.y * pd.x;
        s1 = s1 + d11 * pd.y;
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (k < ulen) upper(ua[k], ub[k], dir(ux[k]));
        for (int k0 = U; k0 < ulen; k0 += MORE) {
            uint32_t wk[MORE];
            dv2 ka[MORE], kb[MORE];
            CgPair<double2> xk[MORE];
#pragma unroll
            for (int k = 0; k < MORE; ++k)
                if (k0 + k < ulen) {
                    const size_t i = ubase + (size_t)(k0 + k) * SLICE;
                    wk[k] = Y.u_bcol[i];
                    ka[k] = pa[i];
                    kb[k] = pb[i];
                }
#pragma unroll
            for (int k = 0; k < MORE; ++k)
                if (k0 + k < ulen) xk[k] = d[wk[k]];
#pragma unroll
            for (int k = 0; k < MORE; ++k)
                if (k0 + k < ulen) upper(ka[k], kb[k], dir(xk[k]));
        }
        return make_double2(s0, s1);
    }
};

// g = A x - b; q = g / Aii; partials g.q, g.g  (cg_precond_jacobi.c:33-43)
template <class Op>
__global__ __launch_bounds__(BLOCK) void k_cg_init(Op op, const typename Op::V* __restrict__ b,
                                                   const typename Op::V* __restrict__ x,
                                                   typename Op::V* __restrict__ g,
                                                   CgPair<typename Op::V>* __restrict__ d,
                                                   const typename Op::V* __restrict__ diag,
                                                   double* partials, uint32_t n) {
    using V = typename Op::V;
    double acc[2] = {0.0, 0.0};
    const Chunk c = my_chunk(n);
    const size_t u = c.beg + threadIdx.x;
    if (u < c.end) {
        const V gv = subu(op.row((uint32_t)u, x), b[u]);
        const V qv = divu(gv, diag[u]);
        g[u] = gv;
        d[u].q = qv;
        acc[0] = dotu(gv, qv);
        acc[1] = dotu(gv, gv);
    }
    __shared__ double red[2][BLOCK / WAVE];
    block_sum<2>(acc, red);
    put_partials<2>(acc, partials);
}

template <class Op, class D>
__global__ __launch_bounds__(BLOCK) void k_cg_dir(Op op,
                                                  const CgPair<typename Op::V>* __restrict__ d,
                                                  CgPair<typename Op::V>* __restrict__ dnew,
                                                  typename Op::V* __restrict__ w,
                                                  const PcgState* __restrict__ sin, PcgState* sout,
                                                  const double* __restrict__ upd, double* dirp,
                                                  uint32_t n, bool first) {
    using V = typename Op::V;
    __shared__ double red[2][ALL_PARTS / WAVE], red2[2][BLOCK / WAVE];
    const Chunk c = my_chunk(n);
    const size_t u = c.beg + threadIdx.x;
    const bool valid = u < c.end;
    AllSum<2> sums;
    sums.load(upd, gridDim.x);
    CgRow<Op> row{op.mat()};
    CgPair<V> own{};
    if (valid) {
        own = d[u];
        row.load((uint32_t)u, d);
    }
    D dir;
    if (!cg_next(sin, sout, sums, first, red, dir)) return;
    double acc[1] = {0.0};
    if (valid) {
        const V pd = dir(own);
        dnew[u].p = pd;
        const V wv = row.product(dir, pd, d);
        w[u] = wv;
        acc[0] = dotu(pd, wv);
    }
    block_sum<1>(acc, red2);
    put_partials<1>(acc, dirp);
}

// The same on scalar CSR.  A workgroup takes 256 rows and walks their entries
// a tile at a time in storage order, so that columns and values are read in
// whole cache lines (one thread per row reads them a row apart); the products
// go through LDS, where each row's thread adds its own in column order, as
// the reference sums a row.  A tile's loads are issued before the sums of
// the tile before it.
// PER entries per thread and tile: 16 take a whole 256-row group of up to 16
// entries a row at once (182 VGPRs, which is no matter while there are two
// workgroups per CU or less), 8 leave more waves to a larger matrix.
// us per iteration (five kernels -> two): 4,290 rows 21 -> 12.4, 41,004 rows
// 20.6 -> 13.1, 90,902 rows 24 -> 13.9 with 16 and 14.3 with 8, 257,442 rows
// 94 -> 21 with 8 and 27 with 16.
// A tile holds few long rows, whose threads add thousands of entries one after
// another while the others wait.  Where a workgroup's rows have 64 entries or
// more on average and none is much longer than the rest, it takes STRIP entries
// of every row at a time instead (8 of 8 bytes are half a cache line, and the
// rest of the line is still cached for the next strip).  us per iteration, five
// kernels -> two with tiles -> with strips: 2,001 rows of 33 entries 29.7 -> 22.3
// (tiles), of 129 59 -> 76 -> 31, of 2,001 1,526 -> 8,297 -> 467; 20,001 of 65 43
// -> 36 -> 22, of 513 365 -> 704 -> 114; 100,001 of 129 197 -> 112 -> 77; every
// tenth of 2,001 rows full, the others of 5 entries, 337 -> 871 -> 310.  Beyond
// CSR_WIDE_ROWS four workgroups a CU hide each other's sums and strips of 4, all
// that their registers leave room for, lose the lines to one another: 250,001 of
// 65 633 -> 89 -> 190, of 257 2,429 -> 466 -> 674; they keep the tiles.  One row
// of 9,000 entries among short ones: 1,183 -> 306 with tiles.
constexpr uint32_t CSR_WIDE_ROWS = 131072;   // PER 16 up to here
constexpr int STRIP = 8;
constexpr uint32_t STRIP_MIN = 64 * BLOCK;   // a workgroup's entries from which strips are taken
constexpr uint32_t STRIP_EVEN = 16;          // ... if they are so many times its longest row's
// The thread's row of a workgroup's 256, by strips (rp: where the rows begin,
// the last one's end after them; prod: STRIP + 1 values a row)
__device__ __forceinline__ double strip_sum(const DevCsr& A, const CgPair<double>* __restrict__ d,
                                            const CgDir& dir, const uint32_t* rp, uint32_t longest,
                                            double* prod) {
    constexpr unsigned AT_ONCE = BLOCK / STRIP, STRIDE = STRIP + 1;   // (a row apart, off the banks)
    const unsigned row0 = threadIdx.x / STRIP, lane = threadIdx.x % STRIP;
    const uint32_t len = rp[threadIdx.x + 1] - rp[threadIdx.x];
    double av[STRIP], s = 0.0;
    CgPair<double> dv[STRIP];
    auto fetch = [&](uint32_t base) {   // (zeros past a row's end)
        uint32_t col[STRIP];
#pragma unroll
        for (int i = 0; i < STRIP; ++i) {
            const unsigned row = row0 + (unsigned)i * AT_ONCE;
            const uint32_t beg = rp[row];
            col[i] = 0;
            av[i] = 0.0;
            if (base + lane < rp[row + 1] - beg) {
                col[i] = A.col[(size_t)beg + base + lane];
                av[i] = A.val[(size_t)beg + base + lane];
            }
        }
#pragma unroll
        for (int i = 0; i < STRIP; ++i) dv[i] = d[col[i]];
    };
    fetch(0);
    for (uint32_t base = 0; base < longest; base += STRIP) {
#pragma unroll
        for (int i = 0; i < STRIP; ++i)
            prod[(row0 + (unsigned)i * AT_ONCE) * STRIDE + lane] = av[i] * dir(dv[i]);
        __syncthreads();
        if (base + STRIP < longest) fetch(base + STRIP);
        for (unsigned t = 0; t < STRIP && base + t < len; t += 4) {   // four reads in flight
            double v[4];
#pragma unroll
            for (unsigned k = 0; k < 4; ++k) v[k] = prod[threadIdx.x * STRIDE + t + k];
#pragma unroll
            for (unsigned k = 0; k < 4; ++k) s = base + t + k < len ? s + v[k] : s;
        }
        __syncthreads();
    }
    return s;
}
template <int PER>
__global__ __launch_bounds__(BLOCK) void k_cg_dir_csr(DevCsr A,
                                                      const CgPair<double>* __restrict__ d,
                                                      CgPair<double>* __restrict__ dnew,
                                                      double* __restrict__ w,
                                                      const PcgState* __restrict__ sin,
                                                      PcgState* sout,
                                                      const double* __restrict__ upd,
                                                      double* dirp, uint32_t n, bool first) {
    constexpr int TILE = PER * BLOCK;
    constexpr bool STRIPS = PER == 16;
    static_assert(!STRIPS || (STRIP + 1) * BLOCK <= TILE, "a strip's products lie in prod");
    __shared__ double red[2][ALL_PARTS / WAVE], prod[TILE], red2[1][BLOCK / WAVE];
    __shared__ uint32_t rp[STRIPS ? BLOCK + 1 : 1], wlen[BLOCK / WAVE];
    const Chunk c = my_chunk(n);
    const size_t u = c.beg + threadIdx.x;
    const bool valid = u < c.end;
    AllSum<2> sums;
    sums.load(upd, gridDim.x);
    const uint32_t e0 = A.rowptr[c.beg], e1 = A.rowptr[c.end];
    uint32_t r0 = e1, r1 = e1;
    CgPair<double> own{};
    if (valid) {
        r0 = A.rowptr[u];
        r1 = A.rowptr[u + 1];
        own = d[u];
    }
    uint32_t longest = 0;   // the longest row's entries where strips are taken
    if constexpr (STRIPS) {
        if (e1 - e0 >= STRIP_MIN) {
            uint32_t m = r1 - r0;
            for (int off = WAVE / 2; off > 0; off >>= 1)
                m = max(m, (uint32_t)__shfl_xor((int)m, off));
            if (threadIdx.x % WAVE == 0) wlen[threadIdx.x / WAVE] = m;
            rp[threadIdx.x] = r0;
            if (threadIdx.x == 0) rp[BLOCK] = e1;
            __syncthreads();
#pragma unroll
            for (int k = 0; k < BLOCK / WAVE; ++k) longest = max(longest, wlen[k]);
            if ((uint64_t)longest * STRIP_EVEN > e1 - e0) longest = 0;
        }
    }
    double av[PER];
    CgPair<double> dv[PER];
    auto fetch = [&](uint64_t base) {
        uint32_t col[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const uint64_t e = base + threadIdx.x + (unsigned)i * BLOCK;
            if (e < e1) {
                col[i] = A.col[e];
                av[i] = A.val[e];
            }
        }
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (base + threadIdx.x + (unsigned)i * BLOCK < e1) dv[i] = d[col[i]];
    };
    if (!longest) fetch(e0);
    CgDir dir;
    if (!cg_next(sin, sout, sums, first, red, dir)) return;
    double s = 0.0;
    if (longest) {
        s = strip_sum(A, d, dir, rp, longest, prod);
    } else {
        for (uint64_t base = e0; base < e1; base += TILE) {
            const uint32_t m = (uint32_t)min((uint64_t)TILE, e1 - base);
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const uint32_t t = threadIdx.x + (unsigned)i * BLOCK;
                if (t < m) prod[t] = av[i] * dir(dv[i]);
            }
            __syncthreads();
            fetch(base + TILE);   // (nothing past the last entry)
            const uint32_t lo = r0 > base ? (uint32_t)(r0 - base) : 0u;
            const uint32_t hi = r1 > base ? (uint32_t)min((uint64_t)m, r1 - base) : 0u;
            for (uint32_t t = lo; t < hi; t += 8) {   // eight reads in flight, added in order
                double v[8];
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k) v[k] = t + k < hi ? prod[t + k] : 0.0;
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k) s = t + k < hi ? s + v[k] : s;
            }
            __syncthreads();
        }
    }
    double acc[1] = {0.0};
    if (valid) {
        const double pd = dir(own);
        dnew[u].p = pd;
        w[u] = s;
        acc[0] = dotu(pd, s);
    }
    block_sum<1>(acc, red2);
    put_partials<1>(acc, dirp);
}
template <class Op>
static void launch_cg_dir(const Op& op, unsigned G, hipStream_t s,
                          const CgPair<typename Op::V>* d, CgPair<typename Op::V>* dnew,
                          typename Op::V* w,
                          const PcgState* sin, PcgState* sout, const double* upd, double* dirp,
                          uint32_t n, bool first) {
    if constexpr (std::is_same<Op, OpCsr>::value) {
        if (n <= CSR_WIDE_ROWS)
            hipLaunchKernelGGL(k_cg_dir_csr<16>, dim3(G), dim3(BLOCK), 0, s, op.A, d, dnew, w, sin,
                               sout, upd, dirp, n, first);
        else
            hipLaunchKernelGGL(k_cg_dir_csr<8>, dim3(G), dim3(BLOCK), 0, s, op.A, d, dnew, w, sin,
                               sout, upd, dirp, n, first);
    } else {
        hipLaunchKernelGGL((k_cg_dir<Op, CgDir>), dim3(G), dim3(BLOCK), 0, s, op, d, dnew, w, sin,
                           sout, upd, dirp, n, first);
    }
}

template <class V>
__global__ __launch_bounds__(BLOCK) void k_cg_update(V* __restrict__ x, V* __restrict__ g,
                                                     CgPair<V>* __restrict__ d,
                                                     const V* __restrict__ w,
                                                     const V* __restrict__ diag,
                                                     const PcgState* __restrict__ st,
                                                     const double* __restrict__ dirp, double* upd,
                                                     uint32_t n) {
    __shared__ double red[2][ALL_PARTS / WAVE], red2[2][BLOCK / WAVE];
    const Chunk c = my_chunk(n);
    const size_t u = c.beg + threadIdx.x;
    const bool valid = u < c.end;
    AllSum<1> sums;
    sums.load(dirp, gridDim.x);
    V xv{}, pv{}, gv{}, wv{}, dv{};
    if (valid) {
        xv = x[u];
        pv = d[u].p;
        gv = g[u];
        wv = w[u];
        dv = diag[u];
    }
    const uint32_t done = st->done;
    const double rz = st->rz;
    double tot[1];
    sums.total(gridDim.x, tot, red);
    if (done) return;
    const double alpha = rz / tot[0];
    double acc[2] = {0.0, 0.0};
    if (valid) {
        x[u] = axpyu(xv, alpha, pv);
        gv = axpyu(gv, alpha, wv);
        g[u] = gv;
        const V qv = divu(gv, dv);
        d[u].q = qv;
        acc[0] = dotu(gv, qv);
        acc[1] = dotu(gv, gv);
    }
    block_sum<2>(acc, red2);
    put_partials<2>(acc, upd);
}

// ---------------------------------------------------------------------------
// mixed precision
// ---------------------------------------------------------------------------
// True residual in FP64 and its scaled FP32 image:
//   r = b - K u; r32 = fl32(dis * r); rr64 = r.r; rr32 = r32.r32
// first: p32 = r32, y32 = 0 (a new CG); otherwise beta = rr32 / rz so that
// the direction update continues the old Krylov sequence.
__global__ __launch_bounds__(BLOCK) void k_mix_residual(Sell2 K, const double2* __restrict__ b,
                                                        const double2* __restrict__ u,
                                                        const double2* __restrict__ dis,
                                                        float2* __restrict__ r32,
                                                        float2* __restrict__ p32,
                                                        float2* __restrict__ y32, PcgState* st,
                                                        double* partials, uint32_t n, int first) {
    if (st->done) return;
    double acc[2] = {0.0, 0.0};
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const double2 ku = row64(K, (uint32_t)i, u);
        const double2 bi = b[i];
        const double2 r = make_double2(bi.x - ku.x, bi.y - ku.y);
        const double2 d = dis[i];
        const float2 rs = make_float2((float)(d.x * r.x), (float)(d.y * r.y));
        r32[i] = rs;
        if (first) {
            p32[i] = rs;
            y32[i] = make_float2(0.f, 0.f);
        }
        acc[0] += r.x * r.x + r.y * r.y;
        acc[1] += (double)rs.x * rs.x + (double)rs.y * rs.y;
    }
    __shared__ double red[2][BLOCK / WAVE];
    block_sum<2>(acc, red);
    put_partials<2>(acc, partials);
}

__global__ __launch_bounds__(FIN) void k_fin_residual(PcgState* st, const double* partials,
                                                      unsigned np, int first) {
    if (st->done) return;
    double tot[2];
    fin_sum<2>(partials, np, tot);
    if (threadIdx.x == 0) {
        const double rr64 = tot[0], rr32 = tot[1];
        st->tol_reached = sqrt(rr64);
        st->gg_cur = rr64;
        if (!(rr64 > st->tol2)) {
            st->done = 1;
            st->status = 0;
        } else if (st->k >= st->max_iter || !isfinite(rr64)) {
            st->done = 1;
            st->status = 1;
        }
        if (!first) st->beta = rr32 / st->rz;
        st->rz = rr32;
        st->maxrr = rr32;
        // the iterated residual at which the true one is predicted to meet
        // the tolerance (ratio of the two norms taken from this update)
        st->conv_rr = rr64 > 0.0 ? 0.5 * st->tol2 * rr32 / rr64 : 0.0;
        st->hold = 0;
        st->updates += 1;
    }
}

// w = Kt p; alpha = rz / (p.w)
__global__ __launch_bounds__(BLOCK) void k_mix_A(Sell2 K, const float2* __restrict__ p,
                                                 float2* __restrict__ w, PcgState* st,
                                                 float* partials, uint32_t n) {
    if (st->done | st->hold) return;
    f32c acc[1] = {{0.f, 0.f}};
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const float2 wv = row32(K, (uint32_t)i, p);
        w[i] = wv;
        const float2 pv = p[i];
        acc[0] = cadd(acc[0], pv.x * wv.x);
        acc[0] = cadd(acc[0], pv.y * wv.y);
    }
    __shared__ f32c red[1][BLOCK / WAVE];
    block_sum<1>(acc, red);
    put_partials<1>(acc, partials);
}

__global__ __launch_bounds__(FIN) void k_fin_mixA(PcgState* st, const float* partials, unsigned np) {
    if (st->done | st->hold) return;
    f32c tot[1];
    fin_sum<1>(partials, np, tot);
    if (threadIdx.x == 0) {
        const double pw = (double)tot[0].s + (double)tot[0].c;
        st->pw = pw;
        st->alpha = st->rz / pw;
        if (!(pw > 0.0) || !isfinite(pw)) {
            st->breakdown = 1;
            st->hold = 1;
        }
    }
}

// y += alpha p; r -= alpha w; rz' = r.r; then continue (beta) or pause for
// a reliable update / the end of a restarted sweep.
__global__ __launch_bounds__(BLOCK) void k_mix_B(float2* __restrict__ y, float2* __restrict__ r,
                                                 const float2* __restrict__ p,
                                                 const float2* __restrict__ w, PcgState* st,
                                                 float* partials, uint32_t n) {
    if (st->done | st->hold) return;
    const float alpha = (float)st->alpha;
    f32c acc[1] = {{0.f, 0.f}};
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const float2 pv = p[i], wv = w[i];
        float2 yv = y[i], rv = r[i];
        yv.x = yv.x + alpha * pv.x;
        yv.y = yv.y + alpha * pv.y;
        rv.x = rv.x - alpha * wv.x;
        rv.y = rv.y - alpha * wv.y;
        y[i] = yv;
        r[i] = rv;
        acc[0] = cadd(acc[0], rv.x * rv.x);
        acc[0] = cadd(acc[0], rv.y * rv.y);
    }
    __shared__ f32c red[1][BLOCK / WAVE];
    block_sum<1>(acc, red);
    put_partials<1>(acc, partials);
}

__global__ __launch_bounds__(FIN) void k_fin_mixB(PcgState* st, const float* partials, unsigned np,
                                                  double delta2, double inner_stop) {
    if (st->done | st->hold) return;
    f32c tot[1];
    fin_sum<1>(partials, np, tot);
    if (threadIdx.x == 0) {
        const double rz = (double)tot[0].s + (double)tot[0].c;
        st->k += 1;
        const bool upd = inner_stop > 0.0 ? !(rz > inner_stop * st->maxrr)   // restarted sweeps
                                          : (rz < delta2 * st->maxrr || rz < st->conv_rr);
        if (upd || st->k >= st->max_iter || !isfinite(rz)) {
            st->hold = 1;
            if (!isfinite(rz)) st->breakdown = 1;
        } else {
            st->beta = rz / st->rz;
            st->rz = rz;
            if (inner_stop <= 0.0 && rz > st->maxrr) st->maxrr = rz;
        }
    }
}

// p = r + beta p
__global__ __launch_bounds__(BLOCK) void k_mix_C(float2* __restrict__ p, const float2* __restrict__ r,
                                                 PcgState* st, uint32_t n) {
    if (st->done | st->hold) return;
    const float beta = (float)st->beta;
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const float2 rv = r[i], pv = p[i];
        p[i] = make_float2(rv.x + beta * pv.x, rv.y + beta * pv.y);
    }
}

// u += dis * y (FP64); y = 0
__global__ __launch_bounds__(BLOCK) void k_mix_update(double2* __restrict__ u,
                                                      const double2* __restrict__ dis,
                                                      float2* __restrict__ y, PcgState* st,
                                                      uint32_t n) {
    if (st->done) return;
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const double2 d = dis[i];
        const float2 yv = y[i];
        double2 uv = u[i];
        uv.x = uv.x + d.x * (double)yv.x;
        uv.y = uv.y + d.y * (double)yv.y;
        u[i] = uv;
        y[i] = make_float2(0.f, 0.f);
    }
}

// ---------------------------------------------------------------------------
// mixed precision: FP64 flexible CG, FP32 Chebyshev-Jacobi preconditioner
// ---------------------------------------------------------------------------
// z = D^-1/2 c(Kt) D^-1/2 r, where c(Kt) s is m steps of the Chebyshev
// iteration for Kt y = s from y = 0 on [lmin, lmax] (Saad, Iterative Methods
// for Sparse Linear Systems, 2nd ed., Alg. 12.1), Kt = D^-1/2 K D^-1/2 in
// FP32.  The outer iteration is CG with the Polak-Ribiere beta (Notay 2000,
// flexible CG), all in FP64 with the FP64 matrix, so FP32 rounding only
// weakens the preconditioner and never the attainable residual.

// first: r = b - K x; otherwise x += alpha p, r -= alpha w.  Then the
// preconditioner's start, P = float2 (scaled, FP32): s = fl32(dis r),
// res = s, d = z = s / theta (d null: neither); P = double2 (unscaled, FP64): res = r,
// d = z = D^-1 r / theta.
template <class P>
__global__ __launch_bounds__(BLOCK) void k_fcg_update(Sell2 K, const double2* __restrict__ b,
                                                      double2* __restrict__ x,
                                                      double2* __restrict__ r,
                                                      const double2* __restrict__ p,
                                                      const double2* __restrict__ w,
                                                      const double2* __restrict__ dis,
                                                      P* __restrict__ res,
                                                      P* __restrict__ d,
                                                      P* __restrict__ z, PcgState* st,
                                                      double* partials, uint32_t n, int first,
                                                      double inv_theta) {
    if (st->done) return;
    const double alpha = st->alpha;
    double acc[1] = {0.0};
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        double2 rv;
        if (first) {
            const double2 ku = row64(K, (uint32_t)i, x);
            const double2 bi = b[i];
            rv = make_double2(bi.x - ku.x, bi.y - ku.y);
        } else {
            x[i] = axpyu(x[i], alpha, p[i]);
            const double2 ro = r[i], wv = w[i];
            rv = make_double2(ro.x - alpha * wv.x, ro.y - alpha * wv.y);
        }
        r[i] = rv;
        const double2 dd = dis[i];
        if constexpr (std::is_same<P, float2>::value) {
            const float2 sv = make_float2((float)(dd.x * rv.x), (float)(dd.y * rv.y));
            const float it = (float)inv_theta;
            res[i] = sv;
            if (d) {
                const float2 dv = make_float2(sv.x * it, sv.y * it);
                d[i] = dv;
                z[i] = dv;
            }
        } else {
            res[i] = rv;
            const double2 dv = make_double2(dd.x * dd.x * rv.x * inv_theta,
                                            dd.y * dd.y * rv.y * inv_theta);
            d[i] = dv;
            z[i] = dv;
        }
        acc[0] += rv.x * rv.x + rv.y * rv.y;
    }
    __shared__ double red[1][BLOCK / WAVE];
    block_sum<1>(acc, red);
    put_partials<1>(acc, partials);
}

__global__ __launch_bounds__(FIN) void k_fin_fcg_update(PcgState* st, const double* partials,
                                                        unsigned np, int first) {
    const uint32_t done = st->done, k = first ? st->k : st->k + 1, max_iter = st->max_iter;
    const double tol2 = st->tol2;
    double tot[1];
    fin_sum<1>(partials, np, tot);
    if (done) return;
    if (threadIdx.x == 0) {
        const double gg = tot[0];
        st->k = k;
        if (first) st->gg0 = gg;
        st->gg_cur = gg;
        st->tol_reached = sqrt(gg);
        if (!(gg > tol2)) {
            st->done = 1;
            st->status = 0;
        } else if (k >= max_iter || !isfinite(gg)) {
            st->done = 1;
            st->status = 1;
        }
    }
}

// one Chebyshev step: res -= Kt d; d' = c1 d + c2 res; z += d'
template <int BITS>
__global__ __launch_bounds__(BLOCK) void k_cheb_step(Sell2 K, const float2* __restrict__ din,
                                                     float2* __restrict__ dout,
                                                     float2* __restrict__ res,
                                                     float2* __restrict__ z, PcgState* st,
                                                     uint32_t n, float c1, float c2) {
    if (st->done) return;
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const float2 t = row_scaled<BITS>(K, (uint32_t)i, din);
        float2 rs = res[i];
        rs.x = rs.x - t.x;
        rs.y = rs.y - t.y;
        const float2 di = din[i];
        const float2 dn = make_float2(c1 * di.x + c2 * rs.x, c1 * di.y + c2 * rs.y);
        float2 zv = z[i];
        zv.x = zv.x + dn.x;
        zv.y = zv.y + dn.y;
        res[i] = rs;
        dout[i] = dn;
        z[i] = zv;
    }
}

// The step on the fp16 copy, with the row sum and the recurrence in FP64
// (vectors stored in FP32).  The FP32 sum loses most of the small result of
// a cancelling stiffness row; with it the outer iteration count jumps up
// and down with the degree (4.2M DOF, degree 28-40: 1006, 940, 1118, 996,
// 711), with FP64 sums it falls steadily (1006, 943, 882, 787, 709) at the
// same cost per step.  NT: non-temporal matrix loads.
// ZM says how z = d_0 + d_1 + ... takes this step's direction:
//   Z_SKIP  not yet (the next step adds it with its own),
//   Z_PAIR  z += d_in + d_out (the previous step's and this one's),
//   Z_ONE   z += d_out.
// Adding the directions in pairs reads and writes z on half the steps
// (16 B per node less on every other step) and rounds z once per pair.
// M: the fp16 matrix, Sell2 (full copy) or Off16 (without diagonal blocks).
enum { Z_SKIP = 0, Z_PAIR = 1, Z_ONE = 2 };
template <bool NT, int ZM, class M>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_cheb_step64(M K, const float2* __restrict__ din,
                                                       float2* __restrict__ dout,
                                                       float2* __restrict__ res,
                                                       float2* __restrict__ z, PcgState* st,
                                                       uint32_t n, double c1, double c2) {
    if (st->done) return;
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const float2 di = din[i];
        const double2 t = cheb_row<NT>(K, (uint32_t)i, din, di);
        const float2 r0 = res[i];
        const double rx = (double)r0.x - t.x, ry = (double)r0.y - t.y;
        const double dx = c1 * (double)di.x + c2 * rx, dy = c1 * (double)di.y + c2 * ry;
        res[i] = make_float2((float)rx, (float)ry);
        dout[i] = make_float2((float)dx, (float)dy);
        if constexpr (ZM != Z_SKIP) {
            const float2 zv = z[i];
            const double ax = ZM == Z_PAIR ? (double)di.x + dx : dx;
            const double ay = ZM == Z_PAIR ? (double)di.y + dy : dy;
            z[i] = make_float2((float)((double)zv.x + ax), (float)((double)zv.y + ay));
        }
    }
}

// Step k of 1..last (z = d_0 on entry): even steps add d_{k-1} + d_k, odd
// steps wait for the next one, except the last, which adds d_k alone.
template <bool NT, class M>
static void launch_cheb_step64(uint32_t k, uint32_t last, unsigned G, hipStream_t s, const M& K,
                               const float2* din, float2* dout, float2* res, float2* z,
                               PcgState* st, uint32_t n, double c1, double c2) {
    if (k % 2 == 0)
        hipLaunchKernelGGL((k_cheb_step64<NT, Z_PAIR, M>), dim3(G), dim3(BLOCK), 0, s, K, din, dout,
                           res, z, st, n, c1, c2);
    else if (k == last)
        hipLaunchKernelGGL((k_cheb_step64<NT, Z_ONE, M>), dim3(G), dim3(BLOCK), 0, s, K, din, dout,
                           res, z, st, n, c1, c2);
    else
        hipLaunchKernelGGL((k_cheb_step64<NT, Z_SKIP, M>), dim3(G), dim3(BLOCK), 0, s, K, din, dout,
                           res, z, st, n, c1, c2);
}

// Several Chebyshev steps in one launch, a workgroup per tile (tiles.hip).
// Up to about 150k nodes a step of k_cheb_step64 is bound by the launch and
// the chain of dependent loads (4 us whatever the size), above that by the
// matrix and vectors it reads; both are paid here once for S steps.  Step
// t = 1 .. S is taken on the tile's rows within S - t rings of the owned
// ones, so each row's neighbours were computed by the same workgroup one
// step earlier; the directions live in LDS (two buffers, widened to FP64
// once), each thread keeps its row (the fp16 values widened to FP32, 16-bit
// positions), residual and z in registers, and a step costs one barrier.
// Halo rows are computed by every tile that lists them.
// Bound by the FP64 pipe and the barriers on small systems (1.35 us per step
// at 33k nodes, outer kernels included, against 4.9), by bytes on large ones
// (about 63 B per node and step against 105: 24.0 against 36.5 us at 2.1M
// nodes).  Where one tile a CU is all there is, the row's values are widened to
// FP64 once, which saves 24 conversions of some 66 FP64 operations a row and
// step (33k nodes 59.1 -> 54.9 us per outer iteration); that takes 84 VGPRs
// instead of 62 and leaves 5 waves per SIMD instead of 8, so more tiles hold
// FP32 (2.1M nodes: 24.0 against 28 us a step, 45k in 283 tiles 71.6 against
// 80.3 per outer iteration).  Held as packed fp16 they cost a second
// conversion per product (24.2 us).
// The arithmetic of a row is k_cheb_step64's: the same sums in the same
// order, an fp16 value times an FP32 entry being exact in FP64, so that the
// fused multiply-add rounds as the separate add does.  Results are the same
// bit for bit.  Residuals and directions are read from one buffer and written
// to another: the halo rows of a tile are owned by its neighbours.
// FULL: every row holds W blocks (the uniform layout).
constexpr uint32_t CHEB_SMAX = 8;   // most rings (steps) of a tile
struct ChebSteps {
    uint32_t steps, k0, last;   // steps k0 .. k0 + steps - 1 of 1 .. last
    double c1[CHEB_SMAX], c2[CHEB_SMAX];
};
// V: the components that a row's values are held in.
template <int W, bool FULL, class V>
__global__ __launch_bounds__(1024) void k_cheb_tiles(Off16 O, Tiles T, ChebSteps cs,
                                                     const float2* __restrict__ din,
                                                     float2* __restrict__ dout,
                                                     const float2* __restrict__ rin,
                                                     float2* __restrict__ rout,
                                                     float2* __restrict__ z, const PcgState* st) {
    extern __shared__ double2 sd[];   // [2][T.ext]
    const uint32_t S = cs.steps, i = threadIdx.x, ext = T.ext;
    const uint32_t t = xcd_remap(blockIdx.x, gridDim.x);
    // The stop flag, the ring offsets (one a lane), the thread's node and its
    // columns go out together; the row's values follow in a second trip instead
    // of a fourth (501x247 100.4 -> 96.9 us per outer iteration).  Large systems,
    // bound by bytes, read the columns of the rows that need them: not those of
    // the outermost ring (1024x512 278 us, 282 with them).
    const bool ahead = T.rings > 3;
    uint32_t ro = T.roff[(size_t)t * (T.rings + 1) + min(i % WAVE, T.rings)];
    uint32_t v = T.ids[(size_t)t * ext + i];
    uint32_t pc[(W + 1) / 2], zero = 0;
#pragma unroll
    for (int q = 0; q < (W + 1) / 2; ++q)
        pc[q] = ahead && (FULL || q < (int)T.W2) ? T.lcol[((size_t)t * T.W2 + q) * ext + i] : 0u;
    asm volatile("" : "+v"(zero));   // (a vector load: no wait on the scalar cache)
    uint32_t done = (&st->done)[zero];
#pragma unroll
    for (int q = 0; q < (W + 1) / 2; ++q) asm volatile("" : "+v"(pc[q]));
    asm volatile("" : "+v"(ro), "+v"(v), "+v"(done));
    if (__builtin_amdgcn_readfirstlane(done)) return;
    const uint32_t own = __builtin_amdgcn_readlane(ro, 0), all = __builtin_amdgcn_readlane(ro, S);
    // a row of ring r takes part in the first S - r steps
    uint32_t act = 0;
    for (uint32_t r = 0; r < S; ++r) act += i < (uint32_t)__builtin_amdgcn_readlane(ro, r);
    typedef V V4 __attribute__((ext_vector_type(4)));
    V4 av[W];
    hv2 od = {};
    float2 rs = {}, zv = {};
    int len = W;
    if (i < all) {
        const float2 d0 = din[v];
        sd[i] = make_double2((double)d0.x, (double)d0.y);
        if (act) {
            size_t g;
            if (FULL || O.width)
                g = (size_t)(v >> 6) * SLICE * O.width + (v & 63);
            else
                g = (size_t)O.slice_ptr[v >> 6] + (v & 63);
            if constexpr (!FULL) len = O.width ? (int)O.width : (int)O.rowlen[v];
            const hv4* __restrict__ val = reinterpret_cast<const hv4*>(O.val);
            if (!ahead)
#pragma unroll
                for (int q = 0; q < (W + 1) / 2; ++q)
                    if (FULL || 2 * q < len) pc[q] = T.lcol[((size_t)t * T.W2 + q) * ext + i];
#pragma unroll
            for (int k = 0; k < W; ++k)
                if (FULL || k < len) {
                    const hv4 h = val[g + (size_t)k * SLICE];
                    av[k] = V4{(V)h.x, (V)h.y, (V)h.z, (V)h.w};
                }
            od = reinterpret_cast<const hv2*>(O.od)[v];
            rs = rin[v];
        }
        if (i < own) zv = z[v];
    }
    __syncthreads();
    uint32_t cur = 0;
    for (uint32_t s = 1; s <= S; ++s) {
        if (s <= act) {
            const double2* __restrict__ d = sd + cur * ext;
            const double c1 = cs.c1[s - 1], c2 = cs.c2[s - 1];
            const uint32_t k = cs.k0 + s - 1;
            const double2 di = d[i];
            double s0 = di.x + (double)od.x * di.y;
            double s1 = (double)od.y * di.x + di.y;
#pragma unroll
            for (int q = 0; q < W; ++q) {
                if (FULL || q < len) {
                    const double2 xv = d[(pc[q / 2] >> (16 * (q & 1))) & 0xffffu];
                    // (opaque per step, or FP64 copies of the row are hoisted)
                    if constexpr (sizeof(V) == 4) asm volatile("" : "+v"(av[q]));
                    s0 = fma((double)av[q].x, xv.x, s0);
                    s0 = fma((double)av[q].y, xv.y, s0);
                    s1 = fma((double)av[q].z, xv.x, s1);
                    s1 = fma((double)av[q].w, xv.y, s1);
                }
            }
            const double rx = (double)rs.x - s0, ry = (double)rs.y - s1;
            const double dx = c1 * di.x + c2 * rx, dy = c1 * di.y + c2 * ry;
            rs = make_float2((float)rx, (float)ry);
            sd[(cur ^ 1u) * ext + i] = make_double2((double)(float)dx, (double)(float)dy);
            // z as launch_cheb_step64 adds it: even steps the pair, the last
            // odd step its own direction (stored for the owned rows only)
            const bool pair = (k & 1u) == 0u;
            if (pair || k == cs.last) {
                const double ax = pair ? di.x + dx : dx;
                const double ay = pair ? di.y + dy : dy;
                zv = make_float2((float)((double)zv.x + ax), (float)((double)zv.y + ay));
            }
        }
        __syncthreads();
        cur ^= 1u;
    }
    if (i < own) {
        rout[v] = rs;
        const double2 dn = sd[cur * ext + i];
        dout[v] = make_float2((float)dn.x, (float)dn.y);
        z[v] = zv;
    }
}

static void launch_cheb_tiles(const Off16& O, const Tiles& T, const ChebSteps& cs,
                              const float2* din, float2* dout, const float2* rin, float2* rout,
                              float2* z, const PcgState* st, hipStream_t s) {
    const dim3 g(T.n), b(T.ext);
    const size_t lds = 2 * (size_t)T.ext * sizeof(double2);
    if (O.width == 6 && T.n <= NUM_CU)
        hipLaunchKernelGGL((k_cheb_tiles<6, true, double>), g, b, lds, s, O, T, cs, din, dout, rin,
                           rout, z, st);
    else if (O.width == 6)
        hipLaunchKernelGGL((k_cheb_tiles<6, true, float>), g, b, lds, s, O, T, cs, din, dout, rin,
                           rout, z, st);
    else
        hipLaunchKernelGGL((k_cheb_tiles<TILE_WMAX, false, float>), g, b, lds, s, O, T, cs, din,
                           dout, rin, rout, z, st);
}

// One step of the all-FP64 preconditioner (precond_bits = 64): the same
// Chebyshev recurrence on the FP64 matrix itself (the symmetric copy the
// FP64 products read, or the full one), vectors and arithmetic in FP64, in
// unscaled variables: res -= K d; d' = c1 d + c2 D^-1 res; z += d'.  With
// d = D^-1/2 d~ and res = D^1/2 res~ this is the scaled step on
// D^-1/2 K D^-1/2 exactly; z then holds D^-1/2 z~, the preconditioned
// residual.  ZM as in k_cheb_step64.
template <class Op, int ZM>
__global__ __launch_bounds__(BLOCK) void k_cheb_step_f64(Op op, const double2* __restrict__ din,
                                                         double2* __restrict__ dout,
                                                         double2* __restrict__ res,
                                                         double2* __restrict__ z,
                                                         const double2* __restrict__ dis,
                                                         PcgState* st, uint32_t n, double c1,
                                                         double c2) {
    if (st->done) return;
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const double2 t = op.row((uint32_t)i, din);
        const double2 r0 = res[i], di = din[i], dd = dis[i];
        const double rx = r0.x - t.x, ry = r0.y - t.y;
        const double dx = c1 * di.x + c2 * (dd.x * dd.x * rx);
        const double dy = c1 * di.y + c2 * (dd.y * dd.y * ry);
        res[i] = make_double2(rx, ry);
        dout[i] = make_double2(dx, dy);
        if constexpr (ZM != Z_SKIP) {
            const double2 zv = z[i];
            const double ax = ZM == Z_PAIR ? di.x + dx : dx;
            const double ay = ZM == Z_PAIR ? di.y + dy : dy;
            z[i] = make_double2(zv.x + ax, zv.y + ay);
        }
    }
}

template <class Op>
static void launch_cheb_step_f64(uint32_t k, uint32_t last, unsigned G, hipStream_t s, const Op& op,
                                 const double2* din, double2* dout, double2* res, double2* z,
                                 const double2* dis, PcgState* st, uint32_t n, double c1,
                                 double c2) {
    if (k % 2 == 0)
        hipLaunchKernelGGL((k_cheb_step_f64<Op, Z_PAIR>), dim3(G), dim3(BLOCK), 0, s, op, din, dout,
                           res, z, dis, st, n, c1, c2);
    else if (k == last)
        hipLaunchKernelGGL((k_cheb_step_f64<Op, Z_ONE>), dim3(G), dim3(BLOCK), 0, s, op, din, dout,
                           res, z, dis, st, n, c1, c2);
    else
        hipLaunchKernelGGL((k_cheb_step_f64<Op, Z_SKIP>), dim3(G), dim3(BLOCK), 0, s, op, din, dout,
                           res, z, dis, st, n, c1, c2);
}

// the preconditioned residual z64: dis z (scaled FP32 z) or z itself
// (unscaled FP64 z)
__device__ __forceinline__ double2 z_unscaled(const float2* z, const double2* dis, size_t i) {
    const double2 dd = dis[i];
    const float2 zv = z[i];
    return make_double2(dd.x * (double)zv.x, dd.y * (double)zv.y);
}
__device__ __forceinline__ double2 z_unscaled(const double2* z, const double2*, size_t i) {
    return z[i];
}

// partials z64.w (Polak-Ribiere numerator) and r.z64
template <class P>
__global__ __launch_bounds__(BLOCK) void k_fcg_dots(const P* __restrict__ z,
                                                    const double2* __restrict__ dis,
                                                    const double2* __restrict__ w,
                                                    const double2* __restrict__ r, PcgState* st,
                                                    double* partials, uint32_t n, int first) {
    if (st->done) return;
    double acc[2] = {0.0, 0.0};
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const double2 zz = z_unscaled(z, dis, i);
        if (!first) acc[0] += dotu(zz, w[i]);
        acc[1] += dotu(r[i], zz);
    }
    __shared__ double red[2][BLOCK / WAVE];
    block_sum<2>(acc, red);
    put_partials<2>(acc, partials);
}

__global__ __launch_bounds__(FIN) void k_fin_fcg_dots(PcgState* st, const double* partials,
                                                      unsigned np, int first) {
    const uint32_t done = st->done;
    const double alpha = st->alpha, rz_old = st->rz;
    double tot[2];
    fin_sum<2>(partials, np, tot);
    if (done) return;
    if (threadIdx.x == 0) {
        const double zw = tot[0], rz = tot[1];
        double beta = first ? 0.0 : -alpha * zw / rz_old;
        if (!(rz > 0.0) || !isfinite(rz) || !isfinite(beta)) {
            // the preconditioned residual lost positivity: restart the
            // direction (p = z) and count the event
            beta = 0.0;
            st->breakdown += 1;
        }
        st->beta = beta;
        st->rz = rz;
    }
}

// p = z64 + beta p  (p = z64 on the first step)
template <class P>
__global__ __launch_bounds__(BLOCK) void k_fcg_p(const P* __restrict__ z,
                                                 const double2* __restrict__ dis,
                                                 double2* __restrict__ p, PcgState* st,
                                                 uint32_t n, int first) {
    if (st->done) return;
    const double beta = st->beta;
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const double2 zz = z_unscaled(z, dis, i);
        p[i] = first ? zz : axpyu(zz, beta, p[i]);
    }
}

// The flexible CG's outer iteration without one-workgroup kernels, up to
// cg2_nodes: k_cg_dir<.., FcgDir> (the direction and w = K p), this
// update, the preconditioner, then k_fcg2_dots; 3 kernels in place of 7 around
// the preconditioner (2-3 us each).  Every workgroup sums the partials of the
// kernel before it, as in the two-kernel PCG, with the same results bit for
// bit as the separate kernels.  State slots: k_cg_dir reads s0 and writes s1,
// the update reads s1 and leaves alpha in s0, the preconditioner's kernels
// read s1, k_fcg2_dots reads s1 and writes s0 (all but alpha).  The stop test
// runs in k_fcg2_dots, so the iteration that meets the tolerance still runs
// its preconditioner.
// FIRST: r = b - K x; otherwise x += alpha p, r -= alpha w.
template <bool FIRST>
__global__ __launch_bounds__(BLOCK) void k_fcg2_update(
    Sell2 K, const double2* __restrict__ b, double2* __restrict__ x, double2* __restrict__ r,
    const CgPair<double2>* __restrict__ d, const double2* __restrict__ w,
    const double2* __restrict__ dis, float2* __restrict__ res, float2* __restrict__ dz,
    float2* __restrict__ z, PcgState* s0, const PcgState* __restrict__ s1,
    const double* __restrict__ dirp, double* rrp, uint32_t n, double inv_theta) {
    __shared__ double red[1][ALL_PARTS / WAVE], red2[1][BLOCK / WAVE];
    const Chunk c = my_chunk(n);
    const size_t i = c.beg + threadIdx.x;
    const bool valid = i < c.end;
    AllSum<1> sums;
    if constexpr (!FIRST) sums.load(dirp, gridDim.x);
    double2 xv{}, pv{}, rv{}, wv{}, dd{};
    if (valid) {
        dd = dis[i];
        if constexpr (!FIRST) {
            xv = x[i];
            pv = d[i].p;
            rv = r[i];
            wv = w[i];
        }
    }
    double alpha = 0.0;
    if constexpr (!FIRST) {
        const uint32_t done = s1->done;
        const double rz = s1->rz;
        double tot[1];
        sums.total(gridDim.x, tot, red);
        if (done) return;
        alpha = rz / tot[0];
        if (blockIdx.x == 0 && threadIdx.x == 0) s0->alpha = alpha;
    }
    double acc[1] = {0.0};
    if (valid) {
        if constexpr (FIRST) {
            const double2 ku = row64(K, (uint32_t)i, x);
            const double2 bi = b[i];
            rv = make_double2(bi.x - ku.x, bi.y - ku.y);
        } else {
            x[i] = axpyu(xv, alpha, pv);
            rv = make_double2(rv.x - alpha * wv.x, rv.y - alpha * wv.y);
        }
        r[i] = rv;
        const float2 sv = make_float2((float)(dd.x * rv.x), (float)(dd.y * rv.y));
        const float it = (float)inv_theta;
        res[i] = sv;
        if (dz) {
            const float2 dv = make_float2(sv.x * it, sv.y * it);
            dz[i] = dv;
            z[i] = dv;
        }
        acc[0] += rv.x * rv.x + rv.y * rv.y;
    }
    block_sum<1>(acc, red2);
    put_partials<1>(acc, rrp);
}

// The stop test on r.r (as k_fin_fcg_update); false when the solve has ended
__device__ __forceinline__ bool fcg2_goes_on(PcgState* s0, const PcgState* __restrict__ s1,
                                             const AllSum<1>& sums, double (&tot)[1],
                                             double (*red)[ALL_PARTS / WAVE], bool first) {
    const uint32_t ended = s1->done, max_iter = s1->max_iter;
    const uint32_t k = first ? s1->k : s1->k + 1u;
    const double tol2 = s1->tol2;
    sums.total(gridDim.x, tot, red);
    if (ended) return false;   // (s0 holds the end of the solve)
    const double gg = tot[0];
    const bool met = !(gg > tol2), stop = met || k >= max_iter || !isfinite(gg);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        s0->k = k;
        s0->max_iter = max_iter;
        s0->tol2 = tol2;
        s0->gg0 = first ? gg : s1->gg0;
        s0->gg_cur = gg;
        s0->tol_reached = sqrt(gg);
        s0->rz = s1->rz;
        s0->breakdown = s1->breakdown;
        s0->done = stop ? 1u : 0u;
        s0->status = met ? 0u : 1u;
    }
    return !stop;
}

// ... and z64 = dis z for the next direction; partials z64.w and r.z64.
__global__ __launch_bounds__(BLOCK) void k_fcg2_dots(const float2* __restrict__ z,
                                                     const double2* __restrict__ dis,
                                                     const double2* __restrict__ w,
                                                     const double2* __restrict__ r,
                                                     CgPair<double2>* __restrict__ d, PcgState* s0,
                                                     const PcgState* __restrict__ s1,
                                                     const double* __restrict__ rrp, double* dots,
                                                     uint32_t n, bool first) {
    __shared__ double red[1][ALL_PARTS / WAVE], red2[2][BLOCK / WAVE];
    const Chunk c = my_chunk(n);
    const size_t i = c.beg + threadIdx.x;
    const bool valid = i < c.end;
    AllSum<1> sums;
    sums.load(rrp, gridDim.x);
    double2 zz{}, wv{}, rv{};
    if (valid) {
        zz = z_unscaled(z, dis, i);
        if (!first) wv = w[i];
        rv = r[i];
    }
    double tot[1];
    if (!fcg2_goes_on(s0, s1, sums, tot, red, first)) return;
    double acc[2] = {0.0, 0.0};
    if (valid) {
        d[i].q = zz;
        if (!first) acc[0] += dotu(zz, wv);
        acc[1] += dotu(rv, zz);
    }
    block_sum<2>(acc, red2);
    put_partials<2>(acc, dots);
}

// One V-cycle of the multigrid preconditioner whose finest level is
// smoothed on the fp16 scaled copy K~ = D^-1/2 K D^-1/2, in scaled variables
// (z~ = D^1/2 z, res~ = D^-1/2 res): Chebyshev smoothing of degree 1 in K~ is
// that in D^-1 K.  The flexible-CG update leaves res = r~ alone; then
//   k_amg_residual  r1 = r~ - K~ z0, the first smoothing step z0 = r~ / theta
//                   formed from r~ wherever it is read;
//   the coarse levels  c = P~ M_c^-1 P~^T r1 (P~ = D^1/2 P);
//   k_amg_post      z = z0 + c + d with d = (r1 - K~ c) / theta, the post-
//                   smoothing; k_amg_post2 does k_fcg2_dots's work as well.
// As steps of the general Chebyshev kernel these wrote z0 and d, a direction
// of zeros and the last residual: 84 MB more at 2.1M nodes (598 -> 587 us per
// outer iteration).  Up to 262,144 nodes, where a launch costs 3.3 us: 64x32
// 43.4 -> 41.5, 96x48 58.4 -> 55.1, 150x75 67.8 -> 64.2, 512x256 141 -> 135.
// The dot products in k_amg_post of the large systems too: 603 (82 VGPRs, or
// their vectors' loads after the product).
template <bool NT, class M>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_amg_residual(M K, const float2* __restrict__ res,
                                                        float2* __restrict__ r1, float it,
                                                        const PcgState* __restrict__ st,
                                                        uint32_t n) {
    if (st->done) return;
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK) {
        const float2 r0 = res[i];
        const double2 t = cheb_row<NT>(K, (uint32_t)i, Scaled32{res, it},
                                       make_float2(r0.x * it, r0.y * it));
        r1[i] = make_float2((float)((double)r0.x - t.x), (float)((double)r0.y - t.y));
    }
}
template <bool NT, class M>
__device__ __forceinline__ float2 amg_post_row(const M& K, size_t i, const float2* __restrict__ cc,
                                               float2 r0, float2 r1, double inv_theta) {
    const float it = (float)inv_theta;
    const float2 ci = cc[i];
    const double2 t = cheb_row<NT>(K, (uint32_t)i, cc, ci);
    const double dx = inv_theta * ((double)r1.x - t.x), dy = inv_theta * ((double)r1.y - t.y);
    return make_float2((float)((double)(r0.x * it) + ((double)ci.x + dx)),
                       (float)((double)(r0.y * it) + ((double)ci.y + dy)));
}
template <bool NT, class M>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_amg_post(
    M K, const float2* __restrict__ cc, const float2* __restrict__ res,
    const float2* __restrict__ r1, float2* __restrict__ z, const PcgState* __restrict__ st,
    uint32_t n, double inv_theta) {
    if (st->done) return;
    const Chunk c = my_chunk(n);
    for (size_t i = c.beg + threadIdx.x; i < c.end; i += BLOCK)
        z[i] = amg_post_row<NT>(K, i, cc, res[i], r1[i], inv_theta);
}
template <bool NT, class M>
__global__ __launch_bounds__(BLOCK) void k_amg_post2(
    M K, const float2* __restrict__ cc, const float2* __restrict__ res,
    const float2* __restrict__ r1, const double2* __restrict__ dis, const double2* __restrict__ w,
    const double2* __restrict__ r, CgPair<double2>* __restrict__ d, PcgState* s0,
    const PcgState* __restrict__ s1, const double* __restrict__ rrp, double* dots, uint32_t n,
    bool first, double inv_theta) {
    __shared__ double red[1][ALL_PARTS / WAVE], red2[2][BLOCK / WAVE];
    const Chunk c = my_chunk(n);
    const size_t i = c.beg + threadIdx.x;
    const bool valid = i < c.end;
    AllSum<1> sums;
    sums.load(rrp, gridDim.x);
    double2 zz{}, wv{}, rv{};
    if (valid) {
        const double2 dd = dis[i];
        if (!first) wv = w[i];
        rv = r[i];
        const float2 zv = amg_post_row<NT>(K, i, cc, res[i], r1[i], inv_theta);
        zz = make_double2(dd.x * (double)zv.x, dd.y * (double)zv.y);
    }
    double tot[1];
    if (!fcg2_goes_on(s0, s1, sums, tot, red, first)) return;
    double acc[2] = {0.0, 0.0};
    if (valid) {
        d[i].q = zz;
        if (!first) acc[0] += dotu(zz, wv);
        acc[1] += dotu(rv, zz);
    }
    block_sum<2>(acc, red2);
    put_partials<2>(acc, dots);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static int poll_state(Workspace& w, hipStream_t s) {
    NBX_HIP(hipMemcpyAsync(w.h_st, w.st, sizeof(PcgState), hipMemcpyDeviceToHost, s));
    NBX_HIP(hipStreamSynchronize(s));
    return NBX_OK;
}

static int sampled_ms(Workspace& w, uint32_t n, double* avg) {
    double tot = 0.0;
    for (uint32_t i = 0; i < n; ++i) {
        float t = 0.f;
        NBX_HIP(hipEventElapsedTime(&t, w.sev[2 * i], w.sev[2 * i + 1]));
        tot += t;
    }
    *avg = n ? tot / n : 0.0;
    return NBX_OK;
}

// A fixed sequence of kernel launches captured once and replayed with
// hipGraphLaunch.  The solvers' repeated steps launch the same kernels with
// the same arguments every time (their state lives on the device), so one
// replay issues a step's kernels with one host call instead of one per
// kernel: the same kernels in the same order as launched one by one, so the
// same results.  The sequences hold kernel launches only.
struct Replay {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    Replay() = default;
    Replay(const Replay&) = delete;
    Replay& operator=(const Replay&) = delete;
    ~Replay() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
    }
};

template <class F>
static int capture(hipStream_t s, F&& launches, Replay& r) {
    NBX_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed));
    launches();
    const hipError_t le = hipGetLastError();
    const hipError_t ee = hipStreamEndCapture(s, &r.graph);
    if (le != hipSuccess || ee != hipSuccess) {
        set_last_error("stream capture of the solver's steps: %s",
                       hipGetErrorString(le != hipSuccess ? le : ee));
        return NBX_ERR_HIP;
    }
    NBX_HIP(hipGraphInstantiate(&r.exec, r.graph, nullptr, nullptr, 0));
    return NBX_OK;
}

// diag: the Jacobi diagonal, or all ones for unpreconditioned CG (q = g/1
// is g exactly, so the same kernels give conjugate_gradient.c:13-77).
template <class Op>
static int pcg_run(const Op& op, uint32_t nu, const double* diag_in, const typename Op::V* b,
                   typename Op::V* x, uint32_t max_iter, double tol, bool stream, Workspace& w,
                   hipStream_t s, SolveStats* stats) {
    using V = typename Op::V;
    V* g = (V*)w.v64[0];
    V* p = (V*)w.v64[1];
    V* wv = (V*)w.v64[2];
    const PBufs<V> pbuf{{p, (V*)w.v64[6], (V*)w.v64[7], (V*)w.v64[8]}};   // p_j in [j % 4]
    const V* diag = (const V*)diag_in;
    PcgState h{};
    h.tol2 = tol * tol;
    h.max_iter = max_iter;
    NBX_HIP(hipMemcpyAsync(w.st, &h, sizeof h, hipMemcpyHostToDevice, s));
    const unsigned G = red_grid(nu);
    // a workspace without events (the no-allocation entry point) is not timed
    const bool timed = w.ev[0] != nullptr;
    if (timed) NBX_HIP(hipEventRecord(w.ev[0], s));
    hipLaunchKernelGGL(k_pcg_init<Op>, dim3(G), dim3(BLOCK), 0, s, op, b, x, g, p, diag, w.st,
                       w.partials, nu);
    hipLaunchKernelGGL(k_fin_init, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G);
    NBX_HIP(hipGetLastError());
    uint32_t nsamp = 0;   // sampled SpMV launches so far
    // Iteration j's kernels (after the stop they return at once).  They
    // depend on j only through j % 4: the direction buffers rotate and every
    // fourth iteration flushes the x updates.
    auto iteration = [&](uint32_t j, bool samp) {
        j &= 3u;
        const V* pj = pbuf.p[j];
        const bool flush = j == 3u;
        if (samp) (void)hipEventRecord(w.sev[2 * nsamp], s);
        hipLaunchKernelGGL(k_pcg_A<Op>, dim3(G), dim3(BLOCK), 0, s, op, pj, wv, w.st, w.partials, nu);
        if (samp) (void)hipEventRecord(w.sev[2 * nsamp++ + 1], s);
        hipLaunchKernelGGL(k_fin_A, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G);
        if (stream) {
            hipLaunchKernelGGL((k_pcg_B<V, true>), dim3(G), dim3(BLOCK), 0, s, g, wv, diag, w.st,
                               w.partials, nu);
            hipLaunchKernelGGL(k_fin_B, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G);
            if (flush)
                hipLaunchKernelGGL((k_pcg_C<V, true, true>), dim3(G), dim3(BLOCK), 0, s, x, pbuf, j,
                                   g, diag, w.st, nu);
            else
                hipLaunchKernelGGL((k_pcg_C<V, true, false>), dim3(G), dim3(BLOCK), 0, s, x, pbuf, j,
                                   g, diag, w.st, nu);
        } else {
            hipLaunchKernelGGL((k_pcg_B<V, false>), dim3(G), dim3(BLOCK), 0, s, g, wv, diag, w.st,
                               w.partials, nu);
            hipLaunchKernelGGL(k_fin_B, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G);
            if (flush)
                hipLaunchKernelGGL((k_pcg_C<V, false, true>), dim3(G), dim3(BLOCK), 0, s, x, pbuf, j,
                                   g, diag, w.st, nu);
            else
                hipLaunchKernelGGL((k_pcg_C<V, false, false>), dim3(G), dim3(BLOCK), 0, s, x, pbuf,
                                   j, g, diag, w.st, nu);
        }
    };
    // Four iterations (j % 4 = 0..3) captured once and replayed: batches
    // hold multiples of four iterations and start at j % 4 = 0.
    Replay four;
    if (w.replay && s != nullptr)
        NBX_TRY(capture(s, [&] {
            for (uint32_t q = 0; q < 4; ++q) iteration(q, false);
        }, four));
    // 64-bit, so that max_iter near UINT32_MAX ("no limit") cannot wrap the
    // guard below
    uint64_t launched = 0;
    uint32_t batch = 4;
    for (;;) {
        for (uint32_t i = 0; i < batch; i += 4) {
            // iterations j0 .. j0 + 3; a sampled one (j0 % SAMPLE_EVERY = 0)
            // is launched kernel by kernel between its events
            const uint64_t j0 = launched + i;
            const bool samp = timed && j0 % Workspace::SAMPLE_EVERY == 0 &&
                              nsamp < (uint32_t)Workspace::NSAMP;
            if (four.exec && !samp) {
                NBX_HIP(hipGraphLaunch(four.exec, s));
            } else {
                for (uint32_t q = 0; q < 4; ++q) iteration(q, samp && q == 0);
            }
        }
        NBX_HIP(hipGetLastError());
        launched += batch;
        NBX_TRY(poll_state(w, s));
        if (w.h_st->done) break;
        if (launched > (uint64_t)max_iter + 8u) {
            set_last_error("PCG did not report completion after %llu iterations",
                           (unsigned long long)launched);
            return NBX_ERR_BREAKDOWN;
        }
        batch = batch < 64 ? batch * 2 : 64;
    }
    hipLaunchKernelGGL(k_pcg_tail<V>, dim3(G), dim3(BLOCK), 0, s, x, pbuf, w.st, nu);
    NBX_HIP(hipGetLastError());
    if (!timed) {
        NBX_HIP(hipStreamSynchronize(s));
        if (stats) {
            stats->iters = stats->fp64_iters = w.h_st->k;
            stats->res0 = sqrt(w.h_st->gg0);
        }
        return NBX_OK;
    }
    NBX_HIP(hipEventRecord(w.ev[1], s));
    NBX_HIP(hipEventSynchronize(w.ev[1]));
    if (stats) {
        float ms = 0.f;
        NBX_HIP(hipEventElapsedTime(&ms, w.ev[0], w.ev[1]));
        stats->ms = ms;
        stats->iters = w.h_st->k;
        stats->fp64_iters = w.h_st->k;
        stats->res0 = sqrt(w.h_st->gg0);
        // samples of iterations that did run (iteration j * SAMPLE_EVERY < k)
        const uint32_t ran = (w.h_st->k + Workspace::SAMPLE_EVERY - 1) / Workspace::SAMPLE_EVERY;
        NBX_TRY(sampled_ms(w, nsamp < ran ? nsamp : ran, &stats->ms_spmv_avg));
    }
    return NBX_OK;
}

// three lower and three upper blocks a row, every slice alike (an interior
// row of a T3 mesh)
static bool sym_u3(const Sym2& y) {
    return y.u_width && y.u_width <= 3 && y.l_width && y.l_width <= 3;
}

// The iteration in two kernels (k_cg_dir, k_cg_update), with pcg_run's host
// cadence, where one round of workgroups takes all rows: the direction kernel's
// loads ahead are then under way in all of them at once, and it gathers twice
// the bytes of a plain product.  us per iteration, five kernels -> two:
// * rows of up to three lower and three upper blocks (142-149 VGPRs, three
//   workgroups a CU) up to 196,608 nodes: 64x32 cantilever 17.8 -> 9.3, 256x128
//   17 -> 9.1, 400x200 (80k nodes) 17 -> 10.4, 540x270 (147k) 22.3 -> 17.1,
//   600x300 (181k) 23.3 -> 19.5, 640x320 (206k) 24.4 -> 24.7, 1024x512 (525k)
//   40 -> 47;
// * other symmetric rows (174 VGPRs, two a CU) up to 131,072: unstructured
//   triangles 480x270 (130k) 26.8 -> 20.6, 512x256 (132k) 32.2 -> 31.2, 600x300
//   32.9 -> 37.2; the same with nodes in random order 41.4 -> 41.3, 44.7 -> 48.4,
//   57 -> 78; rows of 13 blocks, 125k 31.0 -> 24.4, 150k 33.5 -> 35.8;
// * full rows up to 131,072 as well: 400x200 23 -> 14.6, 510x256 (131k) 25.5 ->
//   20.0, in random order 480x270 28.6 -> 25.4.  (Rows of seven blocks in order
//   gain beyond too: 600x300 27.4 -> 24.1, 640x320 29.4 -> 28.9.)
// Scalar CSR takes it up to 262,144 rows (figures at k_cg_dir_csr; in random
// order 90,000 rows of seven 24.2 -> 17.0, 250,000 34.1 -> 28.7).  All keep the
// partials, which every workgroup sums, at 1,024 a value at most.
constexpr uint32_t CG2_MAX_U3 = 196608, CG2_MAX_NODES = 131072, CG2_MAX_ROWS = 262144;
// ... and the flexible CG's direction, which the launches it saves carry further
// on rows of three and three: up to where its partials allow.
constexpr uint32_t FCG2_MAX_U3 = ALL_PARTS * BLOCK;
// most nodes for the two kernels (u3: where the rows are three and three)
static uint32_t cg2_nodes(const DevMatrix& m, uint32_t u3) {
    return m.has_sym && sym_u3(m.y) ? u3 : CG2_MAX_NODES;
}
template <class Op>
static int pcg2_run(const Op& op, uint32_t nu, const double* diag_in, const typename Op::V* b,
                    typename Op::V* x, uint32_t max_iter, double tol, Workspace& w, hipStream_t s,
                    SolveStats* stats) {
    using V = typename Op::V;
    V* g = (V*)w.v64[0];
    V* wv = (V*)w.v64[8];
    // iteration j reads the pairs (q, p_{j-1}) of buffer j % 2 and leaves
    // (q, p_j) in the other (each takes two consecutive vectors)
    CgPair<V>* const d[2] = {(CgPair<V>*)w.v64[1], (CgPair<V>*)w.v64[6]};
    const V* diag = (const V*)diag_in;
    double* upd = w.partials;                       // of the update: 2 G
    double* dirp = w.partials + 2 * (size_t)MAX_GRID;   // of the direction: G
    PcgState h{};
    h.tol2 = tol * tol;
    h.max_iter = max_iter;
    NBX_HIP(hipMemcpyAsync(w.st, &h, sizeof h, hipMemcpyHostToDevice, s));
    const unsigned G = grid_for(nu);
    const bool timed = w.ev[0] != nullptr;
    if (timed) NBX_HIP(hipEventRecord(w.ev[0], s));
    hipLaunchKernelGGL(k_cg_init<Op>, dim3(G), dim3(BLOCK), 0, s, op, b, x, g, d[0], diag, upd,
                       nu);
    NBX_HIP(hipGetLastError());
    uint32_t nsamp = 0;
    // iteration j's kernels depend on j only through j % 2 (and j = 0)
    auto iteration = [&](uint32_t j, bool first, bool samp) {
        j &= 1u;
        if (samp) (void)hipEventRecord(w.sev[2 * nsamp], s);
        launch_cg_dir(op, G, s, d[j], d[j ^ 1u], wv, w.st + j, w.st + (j ^ 1u), upd, dirp, nu,
                      first);
        if (samp) (void)hipEventRecord(w.sev[2 * nsamp++ + 1], s);
        hipLaunchKernelGGL(k_cg_update<V>, dim3(G), dim3(BLOCK), 0, s, x, g, d[j ^ 1u], wv, diag,
                           w.st + (j ^ 1u), dirp, upd, nu);
    };
    Replay four;
    if (w.replay && s != nullptr)
        NBX_TRY(capture(s, [&] {
            for (uint32_t t = 0; t < 4; ++t) iteration(t, false, false);
        }, four));
    uint64_t launched = 0;   // 64-bit: max_iter near UINT32_MAX cannot wrap the guard
    uint32_t batch = 4;
    for (;;) {
        for (uint32_t i = 0; i < batch; i += 4) {
            const uint64_t j0 = launched + i;
            const bool samp = timed && j0 % Workspace::SAMPLE_EVERY == 0 &&
                              nsamp < (uint32_t)Workspace::NSAMP;
            if (four.exec && !samp && j0 != 0) {
                NBX_HIP(hipGraphLaunch(four.exec, s));
            } else {
                for (uint32_t t = 0; t < 4; ++t) iteration(t, j0 == 0 && t == 0, samp && t == 0);
            }
        }
        NBX_HIP(hipGetLastError());
        launched += batch;
        // (an even number of iterations: the last state is in slot 0)
        NBX_TRY(poll_state(w, s));
        if (w.h_st->done) break;
        if (launched > (uint64_t)max_iter + 8u) {
            set_last_error("PCG did not report completion after %llu iterations",
                           (unsigned long long)launched);
            return NBX_ERR_BREAKDOWN;
        }
        batch = batch < 64 ? batch * 2 : 64;
    }
    if (timed) {
        NBX_HIP(hipEventRecord(w.ev[1], s));
        NBX_HIP(hipEventSynchronize(w.ev[1]));
    }
    if (stats) {
        stats->iters = stats->fp64_iters = w.h_st->k;
        stats->res0 = sqrt(w.h_st->gg0);
        if (timed) {
            float ms = 0.f;
            NBX_HIP(hipEventElapsedTime(&ms, w.ev[0], w.ev[1]));
            stats->ms = ms;
            const uint32_t ran = (w.h_st->k + Workspace::SAMPLE_EVERY - 1) / Workspace::SAMPLE_EVERY;
            NBX_TRY(sampled_ms(w, nsamp < ran ? nsamp : ran, &stats->ms_spmv_avg));
        }
    }
    return NBX_OK;
}

__global__ void k_fill_one(double* __restrict__ v, uint32_t n) {
    const uint32_t i = blockIdx.x * BLOCK + threadIdx.x;
    if (i < n) v[i] = 1.0;
}

int pcg_jacobi(const DevMatrix& m, const double* b, double* x, uint32_t max_iter, double tol,
               uint32_t* niter, double* tol_reached, Workspace& w, hipStream_t s,
               SolveStats* stats, bool unpreconditioned) {
    if (m.n == 0) {
        // empty system: no iteration, ||g|| = 0 (cg_precond_jacobi.c:44-89,
        // conjugate_gradient.c:38-76)
        if (niter) *niter = 0;
        if (tol_reached) *tol_reached = 0.0;
        return 0;
    }
    int rc = ws_alloc(w, m.n);
    if (rc) return -rc;
    const double* diag = m.diag;
    if (unpreconditioned) {
        // v64[5] is free during a PCG run (pcg_run uses v64[0..2] and the
        // direction buffers v64[6..8])
        hipLaunchKernelGGL(k_fill_one, dim3(grid_for(m.n)), dim3(BLOCK), 0, s, w.v64[5], m.n);
        if (hipGetLastError() != hipSuccess) return -NBX_ERR_HIP;
        diag = w.v64[5];
    }
    // Stream the update kernels' vectors past the caches when the
    // iteration's working set (matrix + five vectors) exceeds the 256 MiB
    // Infinity Cache; below that, caching them is faster.
    const double mat_bytes = !m.blocked ? 12.0 * (double)m.c.nnz
                             : m.has_sym ? 24.0 * (double)m.y.n_nodes + 36.0 * (double)m.y.n_upper +
                                               8.0 * (double)m.y.n_lower
                                         : 36.0 * (double)m.s.n_blocks;
    const bool stream = mat_bytes + 40.0 * (double)m.n > (double)INFINITY_CACHE_BYTES;
    const bool two = m.blocked && m.s.n_nodes <= cg2_nodes(m, CG2_MAX_U3);
    if (two && m.has_sym)
        rc = sym_u3(m.y)
                 ? pcg2_run(OpSymU<3>{{m.y}}, m.s.n_nodes, diag, (const double2*)b, (double2*)x,
                            max_iter, tol, w, s, stats)
                 : pcg2_run(OpSymU<4>{{m.y}}, m.s.n_nodes, diag, (const double2*)b, (double2*)x,
                            max_iter, tol, w, s, stats);
    else if (two)
        rc = pcg2_run(OpS2{m.s}, m.s.n_nodes, diag, (const double2*)b, (double2*)x, max_iter, tol,
                      w, s, stats);
    else if (m.blocked && m.has_sym && stream)
        rc = pcg_run(OpSym{m.y}, m.s.n_nodes, diag, (const double2*)b, (double2*)x, max_iter, tol,
                     stream, w, s, stats);
    else if (m.blocked && m.has_sym)
        rc = pcg_run(OpSymC{m.y}, m.s.n_nodes, diag, (const double2*)b, (double2*)x, max_iter, tol,
                     stream, w, s, stats);
    else if (m.blocked)
        rc = pcg_run(OpS2{m.s}, m.s.n_nodes, diag, (const double2*)b, (double2*)x, max_iter, tol,
                     stream, w, s, stats);
    else if (!m.blocked && m.c.n <= CG2_MAX_ROWS)
        rc = pcg2_run(OpCsr{m.c}, m.c.n, diag, b, x, max_iter, tol, w, s, stats);
    else
        rc = pcg_run(OpCsr{m.c}, m.c.n, diag, b, x, max_iter, tol, stream, w, s, stats);
    if (rc) return -rc;
    if (stats) stats->layout = m.blocked && m.has_sym ? 1 : 0;
    if (niter) *niter = w.h_st->k;
    if (tol_reached) *tol_reached = w.h_st->tol_reached;
    return (int)w.h_st->status;
}

int pcg_jacobi_csr_view(const DevCsr& c, const double* diag, const double* b, double* x,
                        uint32_t max_iter, double tol, uint32_t* niter, double* tol_reached,
                        Workspace& w, hipStream_t s) {
    if (c.n == 0) {
        if (niter) *niter = 0;
        if (tol_reached) *tol_reached = 0.0;
        return 0;
    }
    if (c.n > CG2_MAX_ROWS) {
        set_last_error("%u rows exceed the two-kernel PCG's %u", c.n, CG2_MAX_ROWS);
        return -NBX_ERR_ARG;
    }
    const int rc = pcg2_run(OpCsr{c}, c.n, diag, b, x, max_iter, tol, w, s, nullptr);
    if (rc) return -rc;
    if (niter) *niter = w.h_st->k;
    if (tol_reached) *tol_reached = w.h_st->tol_reached;
    return (int)w.h_st->status;
}

// Relative-tolerance solves stop on the true residual.  When the
// recursion's stop test fires, the solver restarts from its iterate; the
// restart's first step computes ||b - A x|| afresh, and a restart that
// finds it within the tolerance ends the solve with no further iteration.
// On ill-conditioned K the recursively updated residual drifts from the
// true one (at 4.2M DOF the reference algorithm's 1e-8 leaves 3.5e-8).
// A restart that finds the residual less than 10 % below the previous
// restart's has met the attainable accuracy: the solve then reports
// NBX_NOT_CONVERGED with that residual.
constexpr int SOLVE_PASSES = 8;

static bool stagnated(int pass, double res0, double prev_res0) {
    return pass > 0 && res0 >= 0.9 * prev_res0;
}

// The relative-tolerance solves refuse a right-hand side with a non-finite
// entry, and report a non-finite final residual (a non-finite matrix value
// or initial guess, or an iteration that broke down) as a breakdown rather
// than as convergence: their stop tests compare with `>`, which a NaN fails.
static int finite_rhs(double bb) {
    if (std::isfinite(bb)) return NBX_OK;
    set_last_error("the right-hand side has a non-finite entry (||b||^2 = %g)", bb);
    return NBX_ERR_BREAKDOWN;
}
static int finite_result(double rel_res) {
    if (std::isfinite(rel_res)) return NBX_OK;
    set_last_error("non-finite residual (%g): a matrix value or the initial guess is not "
                   "finite, or the iteration broke down", rel_res);
    return NBX_ERR_BREAKDOWN;
}

static void add_pass(SolveStats& tot, const SolveStats& p, int pass) {
    tot.ms += p.ms;
    tot.iters += p.iters;
    tot.outer += p.outer;
    tot.fp64_iters += p.fp64_iters;
    tot.fallback += p.fallback;
    tot.layout = p.layout;
    tot.rel_res = p.rel_res;
    if (pass == 0) tot.ms_spmv_avg = p.ms_spmv_avg;
}

int solve_fp64(const DevMatrix& m, const double* b, double* x, double rtol, bool true_residual,
               uint32_t max_iter, Workspace& w, hipStream_t s, SolveStats* stats) {
    int rc = ws_alloc(w, m.n);
    if (rc) return rc;
    const double bb = device_norm2(m.n, b, w, s, &rc);
    if (rc) return rc;
    NBX_TRY(finite_rhs(bb));
    SolveStats tot{};
    int status = NBX_NOT_CONVERGED;
    uint32_t used = 0;
    double prev = 0.0;
    const int passes = true_residual ? SOLVE_PASSES : 1;
    for (int pass = 0; pass < passes; ++pass) {
        SolveStats ps{};
        uint32_t it = 0;
        double tr = 0.0;
        const int st = pcg_jacobi(m, b, x, max_iter - used, rtol * sqrt(bb), &it, &tr, w, s, &ps);
        if (st < 0) return -st;
        used += it;
        ps.rel_res = bb > 0 ? tr / sqrt(bb) : 0.0;
        add_pass(tot, ps, pass);
        if (st != 0) break;          // out of iterations
        if (it == 0 || !true_residual) {   // the fresh residual meets the tolerance,
            status = NBX_OK;               // or the recursion's test is the stop
            break;
        }
        if (stagnated(pass, ps.res0, prev)) {
            tot.rel_res = bb > 0 ? ps.res0 / sqrt(bb) : 0.0;
            break;
        }
        prev = ps.res0;
    }
    if (stats) *stats = tot;
    NBX_TRY(finite_result(tot.rel_res));
    return status;
}

static int solve_mixed_cg(const DevMatrix& m, const double* b, double* x, double rtol,
                          const MixedOpts& opt, uint32_t max_iter, Workspace& w, hipStream_t s,
                          SolveStats* stats) {
    int rc = NBX_OK;
    const uint32_t nu = m.s.n_nodes;
    const double bb = device_norm2(m.n, b, w, s, &rc);
    if (rc) return rc;
    NBX_TRY(finite_rhs(bb));
    PcgState h{};
    h.tol2 = rtol * rtol * bb;
    h.max_iter = max_iter;
    NBX_HIP(hipMemcpyAsync(w.st, &h, sizeof h, hipMemcpyHostToDevice, s));
    float2* r32 = (float2*)w.v32[0];
    float2* p32 = (float2*)w.v32[1];
    float2* w32 = (float2*)w.v32[2];
    float2* y32 = (float2*)w.v32[3];
    const double2* dis = (const double2*)m.dis;
    const unsigned G = red_grid(nu);
    const double delta2 = opt.delta * opt.delta;
    const bool restart = opt.variant == CG_RESTART;
    const double inner_stop = restart ? opt.inner_rtol * opt.inner_rtol : 0.0;
    uint32_t nsamp = 0, samp_valid = 0, updates = 0;
    double prev_res = -1.0;
    int stalled = 0;
    NBX_HIP(hipEventRecord(w.ev[0], s));
    hipLaunchKernelGGL(k_mix_residual, dim3(G), dim3(BLOCK), 0, s, m.s, (const double2*)b,
                       (const double2*)x, dis, r32, p32, y32, w.st, w.partials, nu, 1);
    hipLaunchKernelGGL(k_fin_residual, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G, 1);
    NBX_HIP(hipGetLastError());
    NBX_TRY(poll_state(w, s));
    prev_res = w.h_st->tol_reached;
    uint32_t batch = 8;
    bool first_batch = true;
    while (!w.h_st->done) {
        for (uint32_t i = 0; i < batch; ++i) {
            const bool samp = first_batch && nsamp < (uint32_t)Workspace::NSAMP;
            if (samp) NBX_HIP(hipEventRecord(w.sev[2 * nsamp], s));
            hipLaunchKernelGGL(k_mix_A, dim3(G), dim3(BLOCK), 0, s, m.s, p32, w32, w.st,
                               w.partials32, nu);
            if (samp) NBX_HIP(hipEventRecord(w.sev[2 * nsamp++ + 1], s));
            hipLaunchKernelGGL(k_fin_mixA, dim3(1), dim3(FIN), 0, s, w.st, w.partials32, G);
            hipLaunchKernelGGL(k_mix_B, dim3(G), dim3(BLOCK), 0, s, y32, r32, p32, w32, w.st,
                               w.partials32, nu);
            hipLaunchKernelGGL(k_fin_mixB, dim3(1), dim3(FIN), 0, s, w.st, w.partials32, G, delta2,
                               inner_stop);
            hipLaunchKernelGGL(k_mix_C, dim3(G), dim3(BLOCK), 0, s, p32, r32, w.st, nu);
        }
        NBX_HIP(hipGetLastError());
        NBX_TRY(poll_state(w, s));
        if (first_batch) samp_valid = w.h_st->k;
        first_batch = false;
        if (w.h_st->done) break;
        if (w.h_st->hold) {
            if (w.h_st->breakdown) {
                stalled = 1;
                break;
            }
            // reliable update (or the end of a restarted sweep): fold y into
            // u and recompute the true residual with the FP64 matrix
            const int first = restart ? 1 : 0;
            hipLaunchKernelGGL(k_mix_update, dim3(G), dim3(BLOCK), 0, s, (double2*)x, dis, y32, w.st,
                               nu);
            hipLaunchKernelGGL(k_mix_residual, dim3(G), dim3(BLOCK), 0, s, m.s, (const double2*)b,
                               (const double2*)x, dis, r32, p32, y32, w.st, w.partials, nu, first);
            hipLaunchKernelGGL(k_fin_residual, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G, first);
            if (!first)
                hipLaunchKernelGGL(k_mix_C, dim3(G), dim3(BLOCK), 0, s, p32, r32, w.st, nu);
            NBX_HIP(hipGetLastError());
            ++updates;
            NBX_TRY(poll_state(w, s));
            const double res = w.h_st->tol_reached;
            if (!w.h_st->done && restart && res > 0.5 * prev_res) {
                stalled = 1;   // a sweep that no longer reduces the FP64 residual
                break;
            }
            prev_res = res;
            batch = 8;
            continue;
        }
        batch = batch < 64 ? batch * 2 : 64;
    }
    NBX_HIP(hipEventRecord(w.ev[1], s));
    NBX_HIP(hipEventSynchronize(w.ev[1]));
    float ms = 0.f;
    NBX_HIP(hipEventElapsedTime(&ms, w.ev[0], w.ev[1]));
    const uint32_t inner = w.h_st->k;
    int status = w.h_st->status ? NBX_NOT_CONVERGED : NBX_OK;
    double rel = bb > 0 ? w.h_st->tol_reached / sqrt(bb) : 0.0;
    double spmv_avg = 0.0;
    NBX_TRY(sampled_ms(w, nsamp < samp_valid ? nsamp : samp_valid, &spmv_avg));
    SolveStats fb{};
    if (stalled) {
        // the FP32 iteration broke down or stopped reducing the residual:
        // FP64 PCG finishes from the current iterate
        rc = solve_fp64(m, b, x, rtol, opt.true_residual, max_iter, w, s, &fb);
        if (rc != NBX_OK && rc != NBX_NOT_CONVERGED) return rc;
        status = rc;
        rel = fb.rel_res;
        ms += (float)fb.ms;
    }
    if (stats) {
        stats->ms_spmv_avg = spmv_avg;
        stats->iters = inner;
        stats->outer = updates;
        stats->fp64_iters = fb.fp64_iters;
        stats->rel_res = rel;
        stats->ms = ms;
        stats->fallback = stalled;
    }
    NBX_TRY(finite_result(rel));
    return status;
}


// FP64 flexible CG with the FP32 Chebyshev-Jacobi preconditioner.
static int fcg_cheb_pass(const DevMatrix& m, const double* b, double* x, double rtol,
                         const MixedOpts& opt, uint32_t max_iter, uint32_t hint, Workspace& w,
                         hipStream_t s, SolveStats* stats) {
    const uint32_t nu = m.s.n_nodes;
    int rc = NBX_OK;
    const double bb = device_norm2(m.n, b, w, s, &rc);
    if (rc) return rc;
    PcgState h{};
    h.tol2 = rtol * rtol * bb;
    h.max_iter = max_iter;
    const PcgState h2[2] = {h, h};
    NBX_HIP(hipMemcpyAsync(w.st, h2, sizeof h2, hipMemcpyHostToDevice, s));
    // Chebyshev coefficients on [lmax/ratio, lmax] (Saad, Alg. 12.1)
    const uint32_t deg = opt.cheb_degree < 1 ? 1 : opt.cheb_degree;
    const double lmax = m.lambda_max, lmin = lmax / opt.cheb_ratio;
    const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin), sigma = theta / delta;
    std::vector<float> c1(deg), c2(deg);
    std::vector<double> c1d(deg), c2d(deg);
    double rho = 1.0 / sigma;
    for (uint32_t k = 1; k < deg; ++k) {
        const double rn = 1.0 / (2.0 * sigma - rho);
        c1d[k] = rn * rho;
        c2d[k] = 2.0 * rn / delta;
        c1[k] = (float)c1d[k];
        c2[k] = (float)c2d[k];
        rho = rn;
    }
    const double inv_theta = 1.0 / theta;
    double2* r = (double2*)w.v64[0];
    double2* p = (double2*)w.v64[1];
    double2* wv = (double2*)w.v64[2];
    float2* res = (float2*)w.v32[0];
    float2* da = (float2*)w.v32[1];
    float2* db = (float2*)w.v32[2];
    float2* z = (float2*)w.v32[3];
    // the all-FP64 preconditioner's vectors (free during a flexible CG)
    double2* res64 = (double2*)w.v64[5];
    double2* da64 = (double2*)w.v64[6];
    double2* db64 = (double2*)w.v64[7];
    double2* z64 = (double2*)w.v64[8];
    const bool p64 = opt.precond_bits == 64;
    const double2* dis = (const double2*)m.dis;
    const double2* bv = (const double2*)b;
    double2* xv = (double2*)x;
    const unsigned G = red_grid(nu);
    OpS2 op{m.s};
    OpSym ops{m.y};
    // three kernels around the preconditioner (k_fcg2_update) or seven; the
    // preconditioner's kernels test `done` in stp
    const bool fold = !p64 && nu <= cg2_nodes(m, FCG2_MAX_U3);
    PcgState* const stp = fold ? w.st + 1 : w.st;
    CgPair<double2>* const pair[2] = {(CgPair<double2>*)w.v64[1], (CgPair<double2>*)w.v64[6]};
    if (fold) wv = (double2*)w.v64[8];
    double* const dots = w.partials;                             // 2 G
    double* const dirp = w.partials + 2 * (size_t)MAX_GRID;      // G
    double* const rrp = w.partials + 3 * (size_t)MAX_GRID;       // G
    // The fp16 preconditioner's working set (matrix + four FP32 vectors) is
    // read by each of the degree - 1 steps in a row: when it fits in the
    // Infinity Cache, cached loads keep it there between steps (at 4.2M DOF,
    // 243 MB: 1.48 -> 1.32 s per solve); otherwise the matrix streams.  The
    // FP64 preconditioner reads the FP64 matrix the same way, cached when
    // its working set (matrix + five FP64 vectors) fits.
    const bool off16 = opt.precond_bits == 16 && m.has_off16;
    const bool packed = off16 && m.off_packed;
    const double sym_mat = 24.0 * (double)m.y.n_nodes + 36.0 * (double)m.y.n_upper +
                           8.0 * (double)m.y.n_lower;
    const double cheb_mat = p64     ? (m.has_sym ? sym_mat : 36.0 * (double)m.s.n_blocks)
                            : packed ? 8.0 * (double)m.o.n_blocks + 4.0 * (double)m.o.n_pairs +
                                           4.0 * (double)nu
                            : off16 ? 12.0 * (double)m.o.n_blocks + 4.0 * (double)nu
                                    : 12.0 * (double)m.s.n_blocks;
    const bool cheb_cached =
        cheb_mat + (p64 ? 80.0 : 33.0) * (double)nu <= (double)INFINITY_CACHE_BYTES;
    const bool tiled = off16 && m.t.n;
    const bool amg = opt.variant == AMG_FCG;
    const double2* ones = amg ? (const double2*)amg_ones(m.amg) : nullptr;
    const AmgFine fine = amg ? amg_fine(m.amg) : AmgFine{};
    // the fp16 copy's working set, as above, for the multigrid's finest level
    const double fine_mat = m.off_packed ? 8.0 * (double)m.o.n_blocks +
                                               4.0 * (double)m.o.n_pairs + 4.0 * (double)nu
                                         : 12.0 * (double)m.o.n_blocks + 4.0 * (double)nu;
    const bool fine_cached = fine_mat + 41.0 * (double)nu <= (double)INFINITY_CACHE_BYTES;
    // What precedes and follows the preconditioner in the step that leaves
    // z_j (first: z_0); dscale: the diagonal scaling (ones: none).
    // d0, z0: where the preconditioner's first direction goes, or null.
    auto before = [&](int first, uint32_t j, const double2* dscale, double theta_inv, float2* d0,
                      float2* z0) {
        if (!fold) {
            hipLaunchKernelGGL(k_fcg_update<float2>, dim3(G), dim3(BLOCK), 0, s, m.s, bv, xv, r, p,
                               wv, dscale, res, d0, z0, w.st, w.partials, nu, first, theta_inv);
            hipLaunchKernelGGL(k_fin_fcg_update, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G,
                               first);
        } else if (first) {
            hipLaunchKernelGGL(k_fcg2_update<true>, dim3(G), dim3(BLOCK), 0, s, m.s, bv, xv, r,
                               pair[j & 1], wv, dscale, res, d0, z0, w.st, stp, dirp, rrp, nu,
                               theta_inv);
        } else {
            hipLaunchKernelGGL(k_fcg2_update<false>, dim3(G), dim3(BLOCK), 0, s, m.s, bv, xv, r,
                               pair[j & 1], wv, dscale, res, d0, z0, w.st, stp, dirp, rrp, nu,
                               theta_inv);
        }
    };
    auto after = [&](int first, uint32_t j, const double2* dscale) {
        if (fold) {
            hipLaunchKernelGGL(k_fcg2_dots, dim3(G), dim3(BLOCK), 0, s, z, dscale, wv, r,
                               pair[j & 1], w.st, stp, rrp, dots, nu, first != 0);
            return;
        }
        hipLaunchKernelGGL(k_fcg_dots<float2>, dim3(G), dim3(BLOCK), 0, s, z, dscale, wv, r, w.st,
                           w.partials, nu, first);
        hipLaunchKernelGGL(k_fin_fcg_dots, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G, first);
        hipLaunchKernelGGL(k_fcg_p<float2>, dim3(G), dim3(BLOCK), 0, s, z, dscale, p, w.st, nu,
                           first);
    };
    auto precondition_amg16 = [&](int first, uint32_t j) {
        before(first, j, dis, fine.inv_theta, nullptr, nullptr);
        auto cycle = [&](auto nt, const auto& K) {
            constexpr bool NT = decltype(nt)::value;
            using M = std::decay_t<decltype(K)>;
            hipLaunchKernelGGL((k_amg_residual<NT, M>), dim3(G), dim3(BLOCK), 0, s, K, res, da,
                               (float)fine.inv_theta, stp, nu);
            (void)amg_coarse_correction(m.amg, (const float*)da, fine.c, stp, s);
            const float2* cc = (const float2*)fine.c;
            if (fold) {
                hipLaunchKernelGGL((k_amg_post2<NT, M>), dim3(G), dim3(BLOCK), 0, s, K, cc, res, da,
                                   dis, wv, r, pair[j & 1], w.st, stp, rrp, dots, nu, first != 0,
                                   fine.inv_theta);
                return;
            }
            hipLaunchKernelGGL((k_amg_post<NT, M>), dim3(G), dim3(BLOCK), 0, s, K, cc, res, da, z,
                               stp, nu, fine.inv_theta);
            after(first, j, dis);
        };
        auto layout = [&](auto nt) {
            if (m.off_packed && m.o.width)
                cycle(nt, Off16U{m.o});
            else if (m.off_packed)
                cycle(nt, Off16P{m.o});
            else
                cycle(nt, m.o);
        };
        if (fine_cached)
            layout(std::false_type{});
        else
            layout(std::true_type{});
    };
    auto precondition_amg = [&](int first, uint32_t j) {
        // a one-level hierarchy: the update with a unit scaling writes r in
        // FP32 (res), the dense solve z = C^-1 r, the dot products and
        // direction read z unscaled
        before(first, j, ones, 1.0, nullptr, nullptr);
        (void)amg_vcycle(m.amg, (const float*)res, (float*)z, stp, s);
        after(first, j, ones);
    };
    auto precondition = [&](int first, uint32_t j) {
        if (amg && fine.scaled16) {
            precondition_amg16(first, j);
            return;
        }
        if (amg) {
            precondition_amg(first, j);
            return;
        }
        if (p64) {
            hipLaunchKernelGGL(k_fcg_update<double2>, dim3(G), dim3(BLOCK), 0, s, m.s, bv, xv, r, p,
                               wv, dis, res64, da64, z64, w.st, w.partials, nu, first, inv_theta);
            hipLaunchKernelGGL(k_fin_fcg_update, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G,
                               first);
        } else {
            before(first, j, dis, inv_theta, da, z);
        }
        float2* din = da;
        float2* dout = db;
        if (tiled) {
            float2 *rin = res, *rout = (float2*)w.v64[5];
            ChebSteps cs;
            cs.last = deg - 1;
            for (uint32_t k = 1; k < deg; k += cs.steps) {
                cs.k0 = k;
                cs.steps = std::min(m.t.rings, deg - k);
                for (uint32_t t = 0; t < cs.steps; ++t) {
                    cs.c1[t] = c1d[k + t];
                    cs.c2[t] = c2d[k + t];
                }
                launch_cheb_tiles(m.o, m.t, cs, din, dout, rin, rout, z, stp, s);
                std::swap(din, dout);
                std::swap(rin, rout);
            }
        }
        double2* din64 = da64;
        double2* dout64 = db64;
        for (uint32_t k = 1; k < deg && !tiled; ++k) {
            auto step = [&](const auto& K) {
                if (cheb_cached)
                    launch_cheb_step64<false>(k, deg - 1, G, s, K, din, dout, res, z, stp, nu,
                                              c1d[k], c2d[k]);
                else
                    launch_cheb_step64<true>(k, deg - 1, G, s, K, din, dout, res, z, stp, nu,
                                             c1d[k], c2d[k]);
            };
            if (p64 && m.has_sym && cheb_cached)
                launch_cheb_step_f64(k, deg - 1, G, s, OpSymC{m.y}, din64, dout64, res64, z64, dis,
                                     w.st, nu, c1d[k], c2d[k]);
            else if (p64 && m.has_sym)
                launch_cheb_step_f64(k, deg - 1, G, s, ops, din64, dout64, res64, z64, dis, w.st,
                                     nu, c1d[k], c2d[k]);
            else if (p64)
                launch_cheb_step_f64(k, deg - 1, G, s, op, din64, dout64, res64, z64, dis, w.st,
                                     nu, c1d[k], c2d[k]);
            else if (packed && m.o.width)
                step(Off16U{m.o});
            else if (packed)
                step(Off16P{m.o});
            else if (off16)
                step(m.o);
            else if (opt.precond_bits == 16)
                step(m.s);
            else
                hipLaunchKernelGGL(k_cheb_step<32>, dim3(G), dim3(BLOCK), 0, s, m.s, din, dout, res, z,
                                   stp, nu, c1[k], c2[k]);
            std::swap(din, dout);
            std::swap(din64, dout64);
        }
        if (!p64) {
            after(first, j, dis);
            return;
        }
        hipLaunchKernelGGL(k_fcg_dots<double2>, dim3(G), dim3(BLOCK), 0, s, z64, dis, wv, r, w.st,
                           w.partials, nu, first);
        hipLaunchKernelGGL(k_fin_fcg_dots, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G, first);
        hipLaunchKernelGGL(k_fcg_p<double2>, dim3(G), dim3(BLOCK), 0, s, z64, dis, p, w.st, nu,
                           first);
    };
    NBX_HIP(hipEventRecord(w.ev[0], s));
    precondition(1, 0);
    NBX_HIP(hipGetLastError());
    NBX_TRY(poll_state(w, s));
    // Iterations launched between polls of the device state.  Kernels
    // launched after the stop test fired return at once but still cost a
    // launch each (about 2.5 us; some 50 per outer iteration with the
    // multigrid preconditioner), so the batches end near the expected count:
    // with a hint (the iterations of a similar earlier solve) the first
    // batch runs to 7/8 of it and the next ones take 4, 4, 8, 16, 32; without
    // one they take 4, 8, 16, 32.
    uint32_t batch = 4, nsamp = 0;
    int fours = 0;   // batches of 4 still to come before the doubling
    if (hint >= 16) {
        batch = hint - hint / 8;
        if (batch > max_iter) batch = max_iter > 4 ? max_iter : 4u;
        fours = 2;
    }
    uint64_t launched = 0;   // 64-bit: max_iter near UINT32_MAX cannot wrap the guard
    constexpr uint32_t every = 8;   // sample one outer iteration in eight
    // Outer iteration j: the FP64 product, then the preconditioner and the
    // flexible-CG updates; the same kernels and arguments every second time
    // (but for j = 0).
    auto outer = [&](uint32_t j, bool head, bool samp) {
        if (samp) (void)hipEventRecord(w.sev[2 * nsamp], s);
        auto dir = [&](const auto& o) {
            using Op = std::decay_t<decltype(o)>;
            hipLaunchKernelGGL((k_cg_dir<Op, FcgDir>), dim3(G), dim3(BLOCK), 0, s, o, pair[j & 1],
                               pair[(j + 1) & 1], wv, w.st, stp, dots, dirp, nu, head);
        };
        if (fold && m.has_sym && sym_u3(m.y))
            dir(OpSymU<3>{{m.y}});
        else if (fold && m.has_sym)
            dir(OpSymU<4>{{m.y}});
        else if (fold)
            dir(op);
        else if (m.has_sym)
            hipLaunchKernelGGL(k_pcg_A<OpSym>, dim3(G), dim3(BLOCK), 0, s, ops,
                               (const double2*)p, wv, w.st, w.partials, nu);
        else
            hipLaunchKernelGGL(k_pcg_A<OpS2>, dim3(G), dim3(BLOCK), 0, s, op,
                               (const double2*)p, wv, w.st, w.partials, nu);
        if (samp) (void)hipEventRecord(w.sev[2 * nsamp++ + 1], s);
        if (!fold)
            hipLaunchKernelGGL(k_fin_A, dim3(1), dim3(FIN), 0, s, w.st, w.partials, G);
        precondition(0, j + 1);
    };
    Replay two[2];
    if (w.replay && s != nullptr && !w.h_st->done)
        for (uint32_t j = 0; j < 2; ++j)
            NBX_TRY(capture(s, [&] { outer(j, false, false); }, two[j]));
    while (!w.h_st->done) {
        for (uint32_t i = 0; i < batch; ++i) {
            const bool samp = (launched + i) % every == 0 && nsamp < (uint32_t)Workspace::NSAMP;
            const uint64_t j = launched + i;
            if (two[j & 1].exec && !samp && j != 0)
                NBX_HIP(hipGraphLaunch(two[j & 1].exec, s));
            else
                outer((uint32_t)(j & 1), j == 0, samp);
        }
        NBX_HIP(hipGetLastError());
        launched += batch;
        NBX_TRY(poll_state(w, s));
        if (launched > (uint64_t)max_iter + 8u && !w.h_st->done) {
            set_last_error("flexible CG did not report completion");
            return NBX_ERR_BREAKDOWN;
        }
        if (fours > 0) {
            batch = 4;
            --fours;
        } else {
            batch = batch < 32 ? batch * 2 : 32;
        }
    }
    NBX_HIP(hipEventRecord(w.ev[1], s));
    NBX_HIP(hipEventSynchronize(w.ev[1]));
    if (stats) {
        float ms = 0.f;
        NBX_HIP(hipEventElapsedTime(&ms, w.ev[0], w.ev[1]));
        stats->ms = ms;
        stats->iters = w.h_st->k;
        // SpMVs in the preconditioner (Chebyshev), V-cycles (AMG)
        stats->outer = amg ? w.h_st->k : w.h_st->k * (deg - 1);
        stats->fp64_iters = w.h_st->k;
        stats->rel_res = bb > 0 ? w.h_st->tol_reached / sqrt(bb) : 0.0;
        stats->fallback = (int)w.h_st->breakdown;
        // bits 2, 4, 8: the fp16 copy (packed columns, uniform width) that
        // the Chebyshev preconditioner or the multigrid's finest level read
        const bool o16 = amg ? fine.scaled16 : off16;
        const bool pk = amg ? fine.scaled16 && m.off_packed : packed;
        stats->layout = (m.has_sym ? 1 : 0) | (o16 ? 2 : 0) | (pk ? 4 : 0) |
                        (pk && m.o.width ? 8 : 0) | (amg ? 16 : 0);
        stats->res0 = sqrt(w.h_st->gg0);
        const uint32_t ran = (w.h_st->k + every - 1) / every;
        NBX_TRY(sampled_ms(w, nsamp < ran ? nsamp : ran, &stats->ms_spmv_avg));
    }
    return w.h_st->status ? NBX_NOT_CONVERGED : NBX_OK;
}

// Flexible CG passes until a restart's fresh residual meets the tolerance.
static int solve_fcg_cheb(const DevMatrix& m, const double* b, double* x, double rtol,
                          const MixedOpts& opt, uint32_t max_iter, Workspace& w, hipStream_t s,
                          SolveStats* stats) {
    int rc = NBX_OK;
    const double bn = sqrt(device_norm2(m.n, b, w, s, &rc));
    if (rc) return rc;
    NBX_TRY(finite_rhs(bn * bn));
    SolveStats tot{};
    int status = NBX_NOT_CONVERGED;
    uint32_t used = 0;
    // per preconditioner: a Chebyshev adjoint solve's 147 iterations are no
    // guess for the multigrid state solve's 39 (6 ms of launched kernels that
    // returned at once, of 16, at 256x128)
    uint32_t& hint = w.fcg_hint[opt.variant == AMG_FCG];
    double prev = 0.0;
    const int passes = opt.true_residual ? SOLVE_PASSES : 1;
    for (int pass = 0; pass < passes; ++pass) {
        SolveStats ps{};
        rc = fcg_cheb_pass(m, b, x, rtol, opt, max_iter - used, pass == 0 ? hint : 0u, w, s, &ps);
        if (pass == 0) hint = rc == NBX_OK ? ps.iters : 0u;
        if (rc != NBX_OK && rc != NBX_NOT_CONVERGED) return rc;
        used += ps.iters;
        add_pass(tot, ps, pass);
        if (rc == NBX_NOT_CONVERGED) break;
        if (ps.iters == 0 || !opt.true_residual) {
            status = NBX_OK;
            break;
        }
        if (stagnated(pass, ps.res0, prev)) {
            tot.rel_res = bn > 0 ? ps.res0 / bn : 0.0;
            break;
        }
        prev = ps.res0;
    }
    if (stats) *stats = tot;
    NBX_TRY(finite_result(tot.rel_res));
    return status;
}

int solve_mixed(const DevMatrix& m, const double* b, double* x, double rtol, const MixedOpts& opt,
                uint32_t max_iter, Workspace& w, hipStream_t s, SolveStats* stats) {
    const bool cheb = opt.variant == CHEB_FCG;
    const bool fp16 = cheb && opt.precond_bits == 16;
    const bool fp64 = cheb && opt.precond_bits == 64;
    if (opt.variant == AMG_FCG) {
        if (!m.blocked || !m.amg || !m.amg_current) {
            set_last_error("solve_mixed: no current AMG hierarchy (the AMG preconditioner is "
                           "built for nbx_fem systems, whose node coordinates it needs)");
            return NBX_ERR_ARG;
        }
        int rc = ws_alloc(w, m.n);
        if (rc) return rc;
        return solve_fcg_cheb(m, b, x, rtol, opt, max_iter, w, s, stats);
    }
    if (!m.blocked || !m.has_scale ||
        !(fp64 || (fp16 ? m.has_off16 || m.has_val16 : m.has_val32))) {
        set_last_error("solve_mixed: matrix has no scaled %d-bit copy", fp16 ? 16 : 32);
        return NBX_ERR_ARG;
    }
    int rc = ws_alloc(w, m.n);
    if (rc) return rc;
    if (opt.variant == CHEB_FCG) return solve_fcg_cheb(m, b, x, rtol, opt, max_iter, w, s, stats);
    return solve_mixed_cg(m, b, x, rtol, opt, max_iter, w, s, stats);
}

}  // namespace nbx
