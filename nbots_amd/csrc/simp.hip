// SIMP topology optimisation on the device: density filter, sensitivity
// filter and optimality-criteria update around the device T3 system.
//
// The reference has no topology-optimisation code.  The algorithm is the
// density-filter variant of Andreassen, Clausen, Schevenels, Lazarov and
// Sigmund, "Efficient topology optimization in MATLAB using 88 lines of
// code", Struct. Multidisc. Optim. 43 (2011) 1-16:
//   H_ej = max(0, rmin - |c_e - c_j|) over element centroids c,
//   xPhys = (H x) ./ Hs,  dc <- H (dc ./ Hs),  dv <- H (dv ./ Hs),
//   OC: x_new = clamp(x sqrt(-dc / dv / lmid), x - move, x + move, 0, 1),
//   bisection on lmid from (l1, l2) = (0, 1e9) while (l2-l1)/(l1+l2) > 1e-3,
//   l1 = lmid when the filtered volume exceeds the target, else l2 = lmid.
// Triangles of any size: volume V = sum_e a_e xPhys_e (a = element area), so
// dv_e = a_e.  Every filter sum runs over a row's entries in ascending
// column order with separate multiply and add (-ffp-contract=off), so H x
// and H (dc ./ Hs) are bit-identical with a sequential CPU loop.  The
// bisection tests V through the identity V = x_new . H (a ./ Hs) (H is
// symmetric), which needs no filter pass per step; only the final design
// is filtered.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <new>

#include "simp.hpp"

namespace nbx {

// ---- kernels ----------------------------------------------------------------
// sum_k H_ek v_k, v = x or x ./ Hs
template <bool DIV_IN>
__device__ __forceinline__ double filt_row(const DevFilter& H, uint32_t e,
                                           const double* __restrict__ x) {
    size_t i = (size_t)H.slice_ptr[e >> 6] + (e & 63);
    const int len = H.rowlen[e];
    double s = 0.0;
    for (int k = 0; k < len; ++k, i += SLICE) {
        const uint32_t j = H.idx[i];
        const double v = DIV_IN ? x[j] / H.Hs[j] : x[j];
        s += H.val[i] * v;
    }
    return s;
}

// out_j = (H (d ./ Hs))_j     (sensitivity filter; H is symmetric)
__global__ void k_filter_sens(DevFilter H, const double* __restrict__ d,
                              double* __restrict__ out) {
    const uint32_t j = blockIdx.x * BLOCK + threadIdx.x;
    if (j >= H.ne) return;
    out[j] = filt_row<true>(H, j, d);
}

__global__ void k_simp_moduli(const double* __restrict__ xphys, double penal, double E0,
                              double Emin, uint32_t ne, double* __restrict__ E) {
    const uint32_t e = blockIdx.x * BLOCK + threadIdx.x;
    if (e >= ne) return;
    E[e] = Emin + pow(xphys[e], penal) * (E0 - Emin);
}

__global__ void k_oc_init(OcState* st, double target) {
    if (threadIdx.x != 0) return;
    OcState s;
    s.l1 = 0.0;
    s.l2 = 1e9;
    s.target = target;
    s.steps = 0;
    s.pad0 = s.pad1 = 0;
    s.done = (s.l2 - s.l1) / (s.l1 + s.l2) > 1e-3 ? 0u : 1u;
    s.lmid = 0.5 * (s.l2 + s.l1);
    *st = s;
}

// the OC candidate of one element for the multiplier lmid, from
// q = -dc / dv (-dc / dv / lmid evaluates as q / lmid)
__device__ __forceinline__ double oc_candidate_q(double xe, double q, double lmid, double move) {
    double v = xe * sqrt(q / lmid);
    if (v > xe + move) v = xe + move;
    if (v > 1.0) v = 1.0;
    if (v < xe - move) v = xe - move;
    if (v < 0.0) v = 0.0;
    return v;
}
__device__ __forceinline__ double oc_candidate(double xe, double dce, double dve, double lmid,
                                               double move) {
    return oc_candidate_q(xe, -dce / dve, lmid, move);
}

// The bisection's next three levels in one pass.  From the bracket (l1, l2)
// and its midpoint c0 the next two steps can test only 0.5 (c0 + l1) or
// 0.5 (l2 + c0), then one of four midpoints; the pass evaluates all seven
// candidates, each multiplier formed exactly as the step that would test it
// forms it (0.5 (l2 + l1) of that step's bracket), and k_oc_fin3 walks the
// tree one step at a time with the sequential test.  Candidate k's volume is
// the filtered volume of its design, sum_e a_e (H x_new)_e / Hs_e =
// x_new . (H (a ./ Hs)) = x_new . dv because H is symmetric, so a pass reads
// x, dc and dv once and filters nothing (per-workgroup partials, seven
// sums each in the order a one-candidate pass would take).
constexpr int OC_CAND = 7;   // c0; c1 = (L, R); c2 = (LL, LR, RL, RR)
__device__ __forceinline__ void oc_candidates(const OcState& s, double (&c)[OC_CAND]) {
    // L: the volume did not exceed the target (l2 = mid); R: it did (l1 = mid)
    c[0] = s.lmid;
    c[1] = 0.5 * (c[0] + s.l1);    // bracket (l1, c0)
    c[2] = 0.5 * (s.l2 + c[0]);    // bracket (c0, l2)
    c[3] = 0.5 * (c[1] + s.l1);    // (l1, c1L)
    c[4] = 0.5 * (c[0] + c[1]);    // (c1L, c0)
    c[5] = 0.5 * (c[2] + c[0]);    // (c0, c1R)
    c[6] = 0.5 * (s.l2 + c[2]);    // (c1R, l2)
}
__global__ __launch_bounds__(BLOCK) void k_oc_step3(const OcState* __restrict__ st,
                                                    const double* __restrict__ x,
                                                    const double* __restrict__ dc,
                                                    const double* __restrict__ dv, double move,
                                                    uint32_t ne, double* partials) {
    const OcState s = *st;
    if (s.done) return;   // uniform over the grid
    double c[OC_CAND];
    oc_candidates(s, c);
    double acc[OC_CAND] = {};
    for (uint32_t e = blockIdx.x * BLOCK + threadIdx.x; e < ne; e += gridDim.x * BLOCK) {
        const double xe = x[e], dve = dv[e], q = -dc[e] / dve;
#pragma unroll
        for (int k = 0; k < OC_CAND; ++k) acc[k] += dve * oc_candidate_q(xe, q, c[k], move);
    }
    __shared__ double red[OC_CAND][BLOCK / WAVE];
    block_sum<OC_CAND>(acc, red);
    put_partials<OC_CAND>(acc, partials);
}

// the design of the last multiplier the bisection tried, and its filtered
// densities
__global__ void k_oc_x(const OcState* __restrict__ st, const double* __restrict__ x,
                       const double* __restrict__ dc, const double* __restrict__ dv,
                       double move, uint32_t ne, double* __restrict__ xnew) {
    const uint32_t e = blockIdx.x * BLOCK + threadIdx.x;
    if (e >= ne) return;
    xnew[e] = oc_candidate(x[e], dc[e], dv[e], st->lmid, move);
}
__global__ void k_oc_phys(DevFilter H, const double* __restrict__ xnew,
                          double* __restrict__ xphys) {
    const uint32_t e = blockIdx.x * BLOCK + threadIdx.x;
    if (e >= H.ne) return;
    xphys[e] = filt_row<false>(H, e, xnew) / H.Hs[e];
}

// up to three bisection steps on the pass's volumes: each the volume test,
// the next bracket and multiplier (or the end of the bisection)
__global__ __launch_bounds__(FIN) void k_oc_fin3(OcState* st, const double* partials,
                                                 unsigned np) {
    if (st->done) return;
    double tot[OC_CAND];
    fin_sum<OC_CAND>(partials, np, tot);
    if (threadIdx.x == 0) {
        OcState s = *st;
        int k = 0;   // the candidate this step tests (s.lmid)
        for (int level = 0; level < 3 && !s.done; ++level) {
            const bool above = tot[k] > s.target;
            if (above)
                s.l1 = s.lmid;
            else
                s.l2 = s.lmid;
            if ((s.l2 - s.l1) / (s.l1 + s.l2) > 1e-3)
                s.lmid = 0.5 * (s.l2 + s.l1);
            else
                s.done = 1;
            s.steps += 1;
            k = 2 * k + (above ? 2 : 1);   // the child candidate
        }
        *st = s;
    }
}

__global__ __launch_bounds__(BLOCK) void k_absdiff_max(const double* __restrict__ a,
                                                       const double* __restrict__ b, uint32_t n,
                                                       double* partials) {
    double m = 0.0;
    for (uint32_t i = blockIdx.x * BLOCK + threadIdx.x; i < n; i += gridDim.x * BLOCK)
        m = fmax(m, fabs(a[i] - b[i]));
    for (int off = WAVE / 2; off > 0; off >>= 1) m = fmax(m, __shfl_down(m, off, WAVE));
    __shared__ double red[BLOCK / WAVE];
    if (threadIdx.x % WAVE == 0) red[threadIdx.x / WAVE] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < BLOCK / WAVE; ++w) m = fmax(m, red[w]);
        partials[blockIdx.x] = m;
    }
}

__global__ __launch_bounds__(FIN) void k_fin_absmax(const double* partials, unsigned np,
                                                    double* out) {
    double m = 0.0;
    for (unsigned b = threadIdx.x; b < np; b += FIN) m = fmax(m, partials[b]);
    for (int off = WAVE / 2; off > 0; off >>= 1) m = fmax(m, __shfl_down(m, off, WAVE));
    __shared__ double red[FIN / WAVE];
    if (threadIdx.x % WAVE == 0) red[threadIdx.x / WAVE] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < FIN / WAVE; ++w) m = fmax(m, red[w]);
        *out = m;
    }
}

// ---- building H -------------------------------------------------------------
// Bins of edge >= rmin over the centroid bounding box: the entries of a row
// are in the 3x3 bins around its element's.  Each bin lists its elements in
// ascending order, so a row in ascending columns is a merge of nine lists:
// one thread per row, no sorting and no limit on a row's length.  The host
// loop with a sort per row, the layout and the upload took 54-77 ms at
// 512x256 (262,144 elements, a radius of 1.5 edges), this takes 1.9 ms with
// the allocations (96x48: 1.5 -> 0.3): bound by the gathers of the candidates'
// centroids.  The arithmetic is the host's, so is every bit of H.
struct Bins {
    double x0, y0, edge;
    uint32_t nx, ny;
    __host__ __device__ size_t count() const { return (size_t)nx * ny; }
};

// Centroids, areas, and each workgroup's bounding box of the centroids
__global__ __launch_bounds__(BLOCK) void k_simp_geom(const double2* __restrict__ nod,
                                                     const uint32_t* __restrict__ conn,
                                                     uint32_t ne, double2* __restrict__ c,
                                                     double* __restrict__ area,
                                                     double* __restrict__ box) {
    const size_t e = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    double b[4] = {INFINITY, INFINITY, INFINITY, INFINITY};   // min of x, y, -x, -y
    if (e < ne) {
        const double2 p = nod[conn[3 * e]], q = nod[conn[3 * e + 1]], r = nod[conn[3 * e + 2]];
        const double2 m = make_double2((p.x + q.x + r.x) / 3.0, (p.y + q.y + r.y) / 3.0);
        c[e] = m;
        area[e] = 0.5 * ((q.x - p.x) * (r.y - p.y) - (r.x - p.x) * (q.y - p.y));
        b[0] = m.x;
        b[1] = m.y;
        b[2] = -m.x;
        b[3] = -m.y;
    }
    __shared__ double red[4][BLOCK / WAVE];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        for (int off = WAVE / 2; off > 0; off >>= 1) b[i] = fmin(b[i], __shfl_xor(b[i], off));
        if (threadIdx.x % WAVE == 0) red[i][threadIdx.x / WAVE] = b[i];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double v = red[threadIdx.x][0];
        for (int w = 1; w < BLOCK / WAVE; ++w) v = fmin(v, red[threadIdx.x][w]);
        box[4 * (size_t)blockIdx.x + threadIdx.x] = v;
    }
}

// Each element's bin and a place in it (in the order of arrival)
__global__ __launch_bounds__(BLOCK) void k_bin_count(const double2* __restrict__ c, uint32_t ne,
                                                     Bins B, uint32_t* __restrict__ bin,
                                                     uint32_t* __restrict__ place, uint32_t* cnt) {
    const size_t e = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    if (e >= ne) return;
    const uint32_t bx = min((uint32_t)((c[e].x - B.x0) / B.edge), B.nx - 1);
    const uint32_t by = min((uint32_t)((c[e].y - B.y0) / B.edge), B.ny - 1);
    const uint32_t b = by * B.nx + bx;
    bin[e] = b;
    place[e] = atomicAdd(&cnt[b], 1u);
}
__global__ __launch_bounds__(BLOCK) void k_bin_fill(const uint32_t* __restrict__ bin,
                                                    const uint32_t* __restrict__ place,
                                                    uint32_t ne, const uint32_t* __restrict__ ptr,
                                                    uint32_t* __restrict__ list) {
    const size_t e = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    if (e < ne) list[ptr[bin[e]] + place[e]] = (uint32_t)e;
}
// An element's place in ascending order: how many of its bin come before it
__global__ __launch_bounds__(BLOCK) void k_bin_order(const uint32_t* __restrict__ bin, uint32_t ne,
                                                     const uint32_t* __restrict__ ptr,
                                                     const uint32_t* __restrict__ list,
                                                     uint32_t* __restrict__ out) {
    const size_t e = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    if (e >= ne) return;
    const uint32_t beg = ptr[bin[e]], end = ptr[bin[e] + 1];
    uint32_t r = 0;
    for (uint32_t t = beg; t < end; ++t) r += list[t] < (uint32_t)e;
    out[beg + r] = (uint32_t)e;
}

// rmin - |c_e - c_j|
__device__ __forceinline__ double filt_weight(double2 ce, double2 cj, double rmin) {
    const double dx = ce.x - cj.x, dy = ce.y - cj.y;
    return rmin - sqrt(dx * dx + dy * dy);
}

// Row lengths, and each slice's (a wavefront's) longest row and entries
__global__ __launch_bounds__(BLOCK) void k_filt_count(const double2* __restrict__ c, uint32_t ne,
                                                      Bins B, const uint32_t* __restrict__ bin,
                                                      const uint32_t* __restrict__ ptr,
                                                      const uint32_t* __restrict__ list,
                                                      double rmin, uint32_t* __restrict__ width,
                                                      uint32_t* __restrict__ entries) {
    const size_t e = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    uint32_t len = 0;
    if (e < ne) {
        const double2 ce = c[e];
        const uint32_t bx = bin[e] % B.nx, by = bin[e] / B.nx;
        // the bins of one row of bins lie side by side
        for (uint32_t jy = by ? by - 1 : 0; jy <= min(by + 1, B.ny - 1); ++jy) {
            const uint32_t end = ptr[(size_t)jy * B.nx + min(bx + 1, B.nx - 1) + 1];
            for (uint32_t t = ptr[(size_t)jy * B.nx + (bx ? bx - 1 : 0)]; t < end; ++t)
                len += filt_weight(ce, c[list[t]], rmin) > 0.0;
        }
    }
    uint32_t w = len, n = len;
    for (int off = WAVE / 2; off > 0; off >>= 1) {
        w = max(w, __shfl_xor(w, off));
        n += __shfl_xor(n, off);
    }
    if (threadIdx.x % WAVE == 0 && e < ne) {
        width[e / SLICE] = w;
        entries[e / SLICE] = n;
    }
}

// Rows of H (columns ascending, padded with weight 0), their lengths and sums
__global__ __launch_bounds__(BLOCK) void k_filt_rows(const double2* __restrict__ c, DevFilter H,
                                                     Bins B, const uint32_t* __restrict__ bin,
                                                     const uint32_t* __restrict__ ptr,
                                                     const uint32_t* __restrict__ list,
                                                     double rmin) {
    const size_t e = (size_t)blockIdx.x * BLOCK + threadIdx.x;
    if (e >= H.ne) return;
    constexpr uint32_t NONE = 0xffffffffu;
    const double2 ce = c[e];
    const uint32_t bx = bin[e] % B.nx, by = bin[e] / B.nx;
    uint32_t cur[9], end[9], head[9];
    auto next = [&](int q) {   // the list's next element within rmin
        head[q] = NONE;
        for (; cur[q] < end[q]; ++cur[q]) {
            const uint32_t j = list[cur[q]];
            if (filt_weight(ce, c[j], rmin) > 0.0) {
                head[q] = j;
                break;
            }
        }
    };
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const int64_t jx = (int64_t)bx + q % 3 - 1, jy = (int64_t)by + q / 3 - 1;
        cur[q] = end[q] = 0;
        if (jx >= 0 && jx < B.nx && jy >= 0 && jy < B.ny) {
            cur[q] = ptr[(size_t)jy * B.nx + jx];
            end[q] = ptr[(size_t)jy * B.nx + jx + 1];
        }
        next(q);
    }
    const size_t beg = (size_t)H.slice_ptr[e / SLICE] + e % SLICE;
    const size_t stop = H.slice_ptr[e / SLICE + 1];
    size_t i = beg;
    double sum = 0.0;
    for (;;) {
        uint32_t j = NONE;
#pragma unroll
        for (int q = 0; q < 9; ++q) j = min(j, head[q]);
        if (j == NONE || i >= stop) break;   // (a row never has more than its slice's width)
        const double h = filt_weight(ce, c[j], rmin);
        H.idx[i] = j;
        H.val[i] = h;
        sum += h;
        i += SLICE;
#pragma unroll
        for (int q = 0; q < 9; ++q)
            if (head[q] == j) {
                ++cur[q];
                next(q);
            }
    }
    H.rowlen[e] = (uint16_t)((i - beg) / SLICE);
    H.Hs[e] = sum;
    for (; i < stop; i += SLICE) {
        H.idx[i] = (uint32_t)e;
        H.val[i] = 0.0;
    }
}

// ---- host -------------------------------------------------------------------
namespace {

struct DevBuf {   // device scratch of one call
    void* p = nullptr;
    ~DevBuf() { if (p) (void)hipFree(p); }
    template <class T>
    T* at(size_t byte) const { return (T*)((char*)p + byte); }
};

template <class T>
int upload(T** d, const std::vector<T>& h, hipStream_t s) {
    NBX_HIP(hipMalloc(d, h.size() * sizeof(T) + 8));
    if (!h.empty()) NBX_HIP(hipMemcpyAsync(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, s));
    return NBX_OK;
}

// H, Hs, the element areas and their sum (in element order)
int build_filter(Simp& o, FemSys& S) {
    const uint32_t ne = S.ne;
    const hipStream_t s = S.s;
    const unsigned g = grid_for(ne);
    const uint32_t ns = (ne + SLICE - 1) / SLICE;
    // scratch: centroids, boxes, bins, places, two lists, widths, entries
    DevBuf t, u;
    const size_t at_box = (size_t)ne * 16, at_bin = at_box + (size_t)g * 32, n4 = (size_t)ne * 4;
    const size_t at_width = at_bin + 4 * n4;
    NBX_HIP(hipMalloc(&t.p, at_width + 2 * (size_t)ns * 4));
    double2* c = t.at<double2>(0);
    double* box = t.at<double>(at_box);
    uint32_t *bin = t.at<uint32_t>(at_bin), *place = bin + ne, *list0 = place + ne,
             *list = list0 + ne, *width = list + ne;
    NBX_HIP(hipMalloc(&o.area, (size_t)ne * 8 + 8));
    hipLaunchKernelGGL(k_simp_geom, dim3(g), dim3(BLOCK), 0, s, S.nod, S.conn, ne, c, o.area, box);
    NBX_HIP(hipGetLastError());
    std::vector<double> area(ne), hb(4 * (size_t)g);
    NBX_HIP(hipMemcpyAsync(area.data(), o.area, area.size() * 8, hipMemcpyDeviceToHost, s));
    NBX_HIP(copy_on(hb.data(), box, hb.size() * 8, hipMemcpyDeviceToHost, s));
    double b[4] = {hb[0], hb[1], hb[2], hb[3]};
    for (size_t i = 4; i < hb.size(); ++i) b[i % 4] = std::min(b[i % 4], hb[i]);
    // At most about 20 ne bins, however small rmin is.  (On a mesh of uneven
    // density a bin of the mean element's size holds hundreds of elements, each
    // of which scans nine such bins: with four fifths of the nodes in a 400th of
    // the area 96x48 took 1.95 ms to create, 1.18 in the host loop, and takes 0.35.)
    const double lx = -b[2] - b[0], ly = -b[3] - b[1];
    Bins B{b[0], b[1], o.rmin, 1, 1};
    if (std::isfinite(lx) && std::isfinite(ly)) {
        B.edge = std::max({o.rmin, std::sqrt(lx * ly / (16.0 * ne)), (lx + ly) / (4.0 * ne)});
        B.nx = (uint32_t)(lx / B.edge) + 1;
        B.ny = (uint32_t)(ly / B.edge) + 1;
    }
    const size_t nb = B.count();
    NBX_HIP(hipMalloc(&u.p, (2 * nb + 1) * sizeof(uint32_t)));
    uint32_t *cnt = u.at<uint32_t>(0), *ptr = cnt + nb;
    NBX_HIP(hipMemsetAsync(cnt, 0, nb * sizeof(uint32_t), s));
    hipLaunchKernelGGL(k_bin_count, dim3(g), dim3(BLOCK), 0, s, c, ne, B, bin, place, cnt);
    NBX_TRY(scan_u32(cnt, ptr, nb, s));
    hipLaunchKernelGGL(k_bin_fill, dim3(g), dim3(BLOCK), 0, s, bin, place, ne, ptr, list0);
    hipLaunchKernelGGL(k_bin_order, dim3(g), dim3(BLOCK), 0, s, bin, ne, ptr, list0, list);
    hipLaunchKernelGGL(k_filt_count, dim3(g), dim3(BLOCK), 0, s, c, ne, B, bin, ptr, list, o.rmin,
                       width, width + ns);
    NBX_HIP(hipGetLastError());
    std::vector<uint32_t> we(2 * (size_t)ns), sptr(ns + 1, 0);
    NBX_HIP(hipMemcpyAsync(we.data(), width, we.size() * 4, hipMemcpyDeviceToHost, s));
    // (the sum while the device counts)
    double atot = 0.0;
    for (uint32_t e = 0; e < ne; ++e) atot += area[e];
    o.atot = atot;
    NBX_HIP(hipStreamSynchronize(s));
    DevFilter& H = o.H;
    H.ne = ne;
    H.n_slices = ns;
    H.n_ent = 0;
    size_t tot = 0;
    for (uint32_t sl = 0; sl < ns; ++sl) {
        if (we[sl] > 0xffffu) {
            set_last_error("simp: filter row of %u entries (rmin too large)", we[sl]);
            return NBX_ERR_ARG;
        }
        H.n_ent += we[ns + sl];
        tot += (size_t)we[sl] * SLICE;
        if (tot > 0xffffffffull) {
            set_last_error("simp: filter too large");
            return NBX_ERR_ARG;
        }
        sptr[sl + 1] = (uint32_t)tot;
    }
    H.n_stored = tot;
    NBX_TRY(upload(&H.slice_ptr, sptr, s));
    NBX_HIP(hipMalloc(&H.rowlen, (size_t)ne * 2 + 8));
    NBX_HIP(hipMalloc(&H.idx, tot * 4 + 8));
    NBX_HIP(hipMalloc(&H.val, tot * 8 + 8));
    NBX_HIP(hipMalloc(&H.Hs, (size_t)ne * 8 + 8));
    hipLaunchKernelGGL(k_filt_rows, dim3(g), dim3(BLOCK), 0, s, c, H, B, bin, ptr, list, o.rmin);
    NBX_HIP(hipGetLastError());
    NBX_HIP(hipStreamSynchronize(s));
    return NBX_OK;
}

}  // namespace

// H and Hs as host CSR.  On a stream of its own: the copies wait neither for
// another handle's work (a plain hipMemcpy would, and would end a graph capture
// of another thread) nor for the system's, which need not exist any more.
int simp_filter_csr(const Simp& o, uint32_t* ptr, uint32_t* idx, double* val, double* Hs) {
    const DevFilter& H = o.H;
    const bool rows = ptr || idx || val;
    if (!rows && !Hs) return NBX_OK;
    std::vector<uint32_t> sptr(rows ? H.n_slices + 1 : 0), ei(idx ? H.n_stored : 0);
    std::vector<uint16_t> len(rows ? H.ne : 0);
    std::vector<double> ev(val ? H.n_stored : 0);
    struct Own {
        hipStream_t s = nullptr;
        ~Own() { if (s) (void)hipStreamDestroy(s); }
    } own;
    NBX_HIP(hipStreamCreateWithFlags(&own.s, hipStreamNonBlocking));
    auto get = [&](void* to, const void* from, size_t bytes) {
        return bytes ? hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToHost, own.s) : hipSuccess;
    };
    hipError_t e = Hs ? get(Hs, H.Hs, (size_t)H.ne * 8) : hipSuccess;
    if (e == hipSuccess) e = get(sptr.data(), H.slice_ptr, sptr.size() * 4);
    if (e == hipSuccess) e = get(len.data(), H.rowlen, len.size() * 2);
    if (e == hipSuccess) e = get(ei.data(), H.idx, ei.size() * 4);
    if (e == hipSuccess) e = get(ev.data(), H.val, ev.size() * 8);
    const hipError_t done = hipStreamSynchronize(own.s);   // (before the arrays go, also after an error)
    NBX_HIP(e);
    NBX_HIP(done);
    if (!rows) return NBX_OK;
    size_t at = 0;
    for (uint32_t r = 0; r < H.ne; ++r) {
        if (ptr) ptr[r] = (uint32_t)at;
        size_t i = (size_t)sptr[r / SLICE] + r % SLICE;
        for (uint32_t k = 0; k < len[r]; ++k, ++at, i += SLICE) {
            if (idx) idx[at] = ei[i];
            if (val) val[at] = ev[i];
        }
    }
    if (ptr) ptr[H.ne] = (uint32_t)at;
    return NBX_OK;
}

int simp_create(Simp& o, FemSys& S, double rmin, double volfrac, double penal, double E0,
                double Emin, double move, const double* x0_host) {
    const uint32_t ne = S.ne;
    const hipStream_t s = S.s;
    if (ne == 0 || !(rmin > 0.0) || !(volfrac > 0.0 && volfrac <= 1.0) || !(move > 0.0)) {
        set_last_error("simp: need elements, rmin > 0, 0 < volfrac <= 1, move > 0");
        return NBX_ERR_ARG;
    }
    if (!S.F_load) {
        set_last_error("simp: set the boundary conditions of the system first");
        return NBX_ERR_ARG;
    }
    o.rmin = rmin;
    o.volfrac = volfrac;
    o.penal = penal;
    o.E0 = E0;
    o.Emin = Emin;
    o.move = move;
    NBX_TRY(build_filter(o, S));
    const DevFilter& H = o.H;
    // design, filtered densities (xPhys = x at the start), sensitivities
    std::vector<double> x0(ne, volfrac);
    if (x0_host) std::copy(x0_host, x0_host + ne, x0.begin());
    NBX_TRY(upload(&o.x, x0, s));
    NBX_TRY(upload(&o.xphys, x0, s));
    NBX_HIP(hipMalloc(&o.xnew, (size_t)ne * 8 + 8));
    NBX_HIP(hipMalloc(&o.dvf, (size_t)ne * 8 + 8));
    NBX_HIP(hipMalloc(&o.dcf, (size_t)ne * 8 + 8));
    NBX_HIP(hipMalloc(&o.st, sizeof(OcState)));
    NBX_HIP(hipMalloc(&o.scal, 64));
    hipLaunchKernelGGL(k_filter_sens, dim3(grid_for(ne)), dim3(BLOCK), 0, s, H, o.area, o.dvf);
    // system buffers the loop writes
    if (!S.elemE) NBX_HIP(hipMalloc(&S.elemE, (size_t)(ne + 1) * sizeof(double)));
    if (!S.dc) NBX_HIP(hipMalloc(&S.dc, (size_t)ne * 8 + 8));
    if (!S.ce) NBX_HIP(hipMalloc(&S.ce, (size_t)ne * 8 + 8));
    NBX_HIP(hipMemsetAsync(S.u, 0, 2 * (size_t)S.nn * 8, s));
    NBX_HIP(hipGetLastError());
    NBX_HIP(hipStreamSynchronize(s));
    o.iter = 0;
    return NBX_OK;
}

void simp_free(Simp& o) {
    void* ps[] = {o.H.slice_ptr, o.H.rowlen, o.H.idx, o.H.val, o.H.Hs, o.x, o.xnew, o.xphys,
                  o.area, o.dvf, o.dcf, o.st, o.scal};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    o = Simp();
}

int simp_moduli(Simp& o, FemSys& S) {
    hipLaunchKernelGGL(k_simp_moduli, dim3(grid_for(S.ne)), dim3(BLOCK), 0, S.s, o.xphys, o.penal,
                       o.E0, o.Emin, S.ne, S.elemE);
    NBX_HIP(hipGetLastError());
    S.P.elemE = S.elemE;
    return NBX_OK;
}

int simp_update(Simp& o, FemSys& S, double* change) {
    const hipStream_t s = S.s;
    const uint32_t ne = S.ne;
    const DevFilter& H = o.H;
    hipLaunchKernelGGL(k_filter_sens, dim3(grid_for(ne)), dim3(BLOCK), 0, s, H, S.dc, o.dcf);
    hipLaunchKernelGGL(k_oc_init, dim3(1), dim3(WAVE), 0, s, o.st, o.volfrac * o.atot);
    unsigned g = grid_for(ne);
    if (g > (unsigned)MAX_GRID) g = MAX_GRID;
    // Bisection passes (three steps each) are launched in batches, the
    // first as long as the previous update's bisection; kernels of a
    // finished bisection return at once.  From (0, 1e9) the bracket reaches
    // any multiplier above 1e-300 within about 1050 halvings.
    constexpr int MAX_STEPS = 2048;
    int batch = o.last_oc_steps ? (int)(o.last_oc_steps + 2) / 3 : 16;
    OcState h{};
    // (seven partials per workgroup in the workspace's 4 MAX_GRID)
    const unsigned g3 = std::min(g, (unsigned)(4 * MAX_GRID / OC_CAND));
    for (int done_steps = 0;; done_steps += 3 * batch, batch = 4) {
        if (done_steps >= MAX_STEPS) {
            set_last_error("simp: OC bisection did not close in %d steps", MAX_STEPS);
            return NBX_ERR_BREAKDOWN;
        }
        for (int k = 0; k < batch; ++k) {
            hipLaunchKernelGGL(k_oc_step3, dim3(g3), dim3(BLOCK), 0, s, o.st, o.x, o.dcf, o.dvf,
                               o.move, ne, S.ws.partials);
            hipLaunchKernelGGL(k_oc_fin3, dim3(1), dim3(FIN), 0, s, o.st, S.ws.partials, g3);
        }
        NBX_HIP(hipGetLastError());
        NBX_HIP(hipMemcpyAsync(&h, o.st, sizeof h, hipMemcpyDeviceToHost, s));
        NBX_HIP(hipStreamSynchronize(s));
        if (h.done) break;
    }
    o.last_oc_steps = h.steps;
    hipLaunchKernelGGL(k_oc_x, dim3(grid_for(ne)), dim3(BLOCK), 0, s, o.st, o.x, o.dcf, o.dvf,
                       o.move, ne, o.xnew);
    hipLaunchKernelGGL(k_oc_phys, dim3(grid_for(ne)), dim3(BLOCK), 0, s, H, o.xnew, o.xphys);
    hipLaunchKernelGGL(k_absdiff_max, dim3(g), dim3(BLOCK), 0, s, o.xnew, o.x, ne, S.ws.partials);
    hipLaunchKernelGGL(k_fin_absmax, dim3(1), dim3(FIN), 0, s, S.ws.partials, g, o.scal);
    NBX_HIP(hipGetLastError());
    double ch = 0.0;
    NBX_HIP(hipMemcpyAsync(&ch, o.scal, sizeof ch, hipMemcpyDeviceToHost, s));
    NBX_HIP(hipStreamSynchronize(s));
    std::swap(o.x, o.xnew);
    o.iter += 1;
    if (change) *change = ch;
    return NBX_OK;
}

}  // namespace nbx
