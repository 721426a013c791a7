// Node tiles with halo rings, for kernels that take several dependent
// row-product steps of one matrix in a single launch (k_cheb_tiles,
// solve.hip).
//
// A tile owns the nodes of one cell of a uniform grid over the mesh's
// bounding box (about `own` nodes), so its boundary is short whatever the
// node numbering: S rings around 256 owned nodes of a triangle mesh hold
// (16 + 2 S)^2 nodes, where S bandwidths around 256 consecutive ones hold
// thousands.  The tile lists its nodes ring by ring (the owned ones, then the
// neighbours of the ring before), ascending within a ring so that reads by
// node stay nearly coalesced, and each row's columns as positions in that
// list.  Built on the device, once per pattern.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <vector>

#include "rows.hpp"

namespace nbx {

namespace {

constexpr int TILE_TB = 1024;       // threads of the ring kernel = most rows of a tile
constexpr uint32_t TILE_HASH = 4096;
constexpr uint32_t NONE = 0xffffffffu;
constexpr unsigned TOO_MANY = 0xffffffffu;
constexpr uint32_t RINGS_MAX = 8;
constexpr uint32_t RUNS = RINGS_MAX + 1, INFO = RUNS + 1;   // words of k_tile_rings's info

// per workgroup: smallest and largest x and y
__global__ __launch_bounds__(BLOCK) void k_tile_bbox(const double2* __restrict__ xy, uint32_t n,
                                                     double* __restrict__ out) {
    double v[4] = {INFINITY, INFINITY, INFINITY, INFINITY};   // x, y, -x, -y
    for (uint32_t i = blockIdx.x * BLOCK + threadIdx.x; i < n; i += gridDim.x * BLOCK) {
        const double2 p = xy[i];
        v[0] = fmin(v[0], p.x);
        v[1] = fmin(v[1], p.y);
        v[2] = fmin(v[2], -p.x);
        v[3] = fmin(v[3], -p.y);
    }
    __shared__ double red[4][BLOCK / WAVE];
    for (int m = 0; m < 4; ++m) {
        for (int off = WAVE / 2; off > 0; off >>= 1) v[m] = fmin(v[m], __shfl_down(v[m], off, WAVE));
        if (threadIdx.x % WAVE == 0) red[m][threadIdx.x / WAVE] = v[m];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double m = red[threadIdx.x][0];
        for (int w = 1; w < BLOCK / WAVE; ++w) m = fmin(m, red[threadIdx.x][w]);
        out[4 * (size_t)blockIdx.x + threadIdx.x] = m;
    }
}

// a node's grid cell
struct TileGrid {
    double x0, y0, ix, iy;   // origin, cells per unit length
    uint32_t nx, ny;
};
__device__ __forceinline__ uint32_t tile_cell(const TileGrid& g, double2 p) {
    // (fmax and fmin return the bound for a NaN)
    const uint32_t cx = (uint32_t)fmin(fmax((p.x - g.x0) * g.ix, 0.0), (double)(g.nx - 1));
    const uint32_t cy = (uint32_t)fmin(fmax((p.y - g.y0) * g.iy, 0.0), (double)(g.ny - 1));
    return cy * g.nx + cx;
}
// A wavefront's lanes in runs of equal cells: one atomic a run instead of one a
// lane, all on one address where a cell holds most of the mesh.
struct CellRun {
    unsigned first, len;   // the run's first lane and lanes
};
__device__ __forceinline__ CellRun cell_run(uint32_t cell) {
    const unsigned lane = threadIdx.x % WAVE;
    const uint32_t before = (uint32_t)__shfl_up((int)cell, 1, WAVE);
    const uint64_t heads = __ballot(lane == 0 || cell != before);
    const uint64_t upto = heads & ((2ull << lane) - 1), after = heads & ~((2ull << lane) - 1);
    const unsigned first = WAVE - 1 - (unsigned)__clzll((long long)upto);
    return {first, (after ? (unsigned)__ffsll((long long)after) - 1 : WAVE) - first};
}
__global__ void k_tile_count(TileGrid g, const double2* __restrict__ xy, uint32_t n,
                             uint32_t* __restrict__ cell, uint32_t* cnt) {
    const uint32_t v = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t c = v < n ? tile_cell(g, xy[v]) : NONE;
    if (v < n) cell[v] = c;
    const CellRun run = cell_run(c);
    if (threadIdx.x % WAVE == run.first && c != NONE) atomicAdd(&cnt[c], run.len);
}
__global__ void k_tile_zero(uint32_t* p, uint32_t n) {
    const uint32_t i = blockIdx.x * BLOCK + threadIdx.x;
    if (i < n) p[i] = 0u;
}
// Each cell's nodes, in any order (the ring kernel sorts them); info[0]: a cell
// has more than `limit`.
__global__ void k_tile_fill(const uint32_t* __restrict__ cell, uint32_t n,
                            const uint32_t* __restrict__ ptr, uint32_t* pos,
                            uint32_t* __restrict__ own, uint32_t limit, unsigned* info) {
    const uint32_t v = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t c = v < n ? cell[v] : NONE;
    const CellRun run = cell_run(c);
    uint32_t at = 0;
    if (threadIdx.x % WAVE == run.first && c != NONE) {
        at = atomicAdd(&pos[c], run.len);
        if (at + run.len > limit) info[0] = 1u;
    }
    at = (uint32_t)__shfl((int)at, (int)run.first, WAVE) + threadIdx.x % WAVE - run.first;
    if (c != NONE) own[ptr[c] + at] = v;
}

__device__ __forceinline__ uint32_t tile_hash(uint32_t id) {
    return (id * 2654435761u) >> 20;   // 12 bits
}
// the table position of id; NONE when it is absent and the table is full
__device__ uint32_t tile_find(const uint32_t* keys, uint32_t id) {
    uint32_t h = tile_hash(id);
    for (uint32_t k = 0; k < TILE_HASH; ++k, h = (h + 1) % TILE_HASH)
        if (keys[h] == id) return h;
    return NONE;
}
// true when this call put id into the table (bounded probes: a full table
// takes nothing and the caller's count has overflowed by then)
__device__ bool tile_insert(uint32_t* keys, uint32_t id) {
    uint32_t h = tile_hash(id);
    for (uint32_t k = 0; k < TILE_HASH; ++k, h = (h + 1) % TILE_HASH) {
        const uint32_t old = atomicCAS(&keys[h], NONE, id);
        if (old == NONE) return true;
        if (old == id) return false;
    }
    return false;
}
// list[b..e) ascending (distinct values): each value to its rank
__device__ void tile_sort(uint32_t* list, uint32_t* tmp, uint32_t b, uint32_t e) {
    const uint32_t i = b + threadIdx.x;
    uint32_t key = 0, rank = 0;
    if (i < e) {
        key = list[i];
        for (uint32_t j = b; j < e; ++j) rank += list[j] < key;
        tmp[b + rank] = key;
    }
    __syncthreads();
    if (i < e) list[i] = tmp[i];
    __syncthreads();
}

// One workgroup per tile.  ext = 0: only info[r], r = 1 .. rings, the rows of
// the largest tile of r rings (TOO_MANY: more than `limit`), and info[RUNS], the
// groups of 8 consecutive ids that the tiles' owned rows touch.  Otherwise the
// tile's list, ring offsets and columns (row i's block 2 q + h in half h of word
// lcol[(t W2 + q) ext + i]; padding names the row itself).
template <class Len>
__global__ __launch_bounds__(TILE_TB) void k_tile_rings(TileRows<Len> O,
                                                        const uint32_t* __restrict__ ptr,
                                                        const uint32_t* __restrict__ own,
                                                        uint32_t limit, uint32_t rings,
                                                        uint32_t wmax, uint32_t W2, uint32_t ext,
                                                        uint32_t* __restrict__ ids,
                                                        uint32_t* __restrict__ lcol,
                                                        uint32_t* __restrict__ roff,
                                                        unsigned* info) {
    __shared__ uint32_t keys[TILE_HASH], list[TILE_TB], tmp[TILE_TB];
    __shared__ uint16_t slot[TILE_HASH];
    __shared__ uint32_t cnt;
    const uint32_t t = blockIdx.x, tid = threadIdx.x;
    if (info[0]) return;   // a cell has more than `limit` (set by the kernel before this one)
    const uint32_t o0 = ptr[t], c0 = ptr[t + 1] - o0;
    for (uint32_t i = tid; i < TILE_HASH; i += TILE_TB) keys[i] = NONE;
    __syncthreads();
    if (tid < c0) {
        const uint32_t id = own[o0 + tid];
        list[tid] = id;
        tile_insert(keys, id);
    }
    __syncthreads();
    tile_sort(list, tmp, 0, c0);
    if (!ext) {
        const bool head = tid < c0 && (tid == 0 || list[tid] / 8 != list[tid - 1] / 8);
        const uint64_t heads = __ballot(head);
        if (tid % WAVE == 0 && heads) atomicAdd(&info[RUNS], (unsigned)__popcll(heads));
    }
    if (ext && tid == 0) roff[(size_t)t * (rings + 1)] = c0;
    uint32_t beg = 0, end = c0;
    for (uint32_t r = 1; r <= rings; ++r) {
        if (tid == 0) cnt = end;
        __syncthreads();
        for (uint32_t f = tid; f < (end - beg) * wmax; f += TILE_TB) {
            const uint32_t v = list[beg + f / wmax], k = f % wmax;
            if (k >= O.rowlen[v]) continue;
            const uint32_t w = O.bcol[(size_t)O.slice_ptr[v >> 6] + (v & 63) + (size_t)k * SLICE];
            if (tile_insert(keys, w)) {
                const uint32_t at = atomicAdd(&cnt, 1u);
                if (at < limit) list[at] = w;
            }
        }
        __syncthreads();
        const uint32_t now = cnt;
        __syncthreads();
        if (now > limit) {
            if (tid == 0)
                for (uint32_t q = r; q <= rings; ++q) atomicMax(&info[q], TOO_MANY);
            return;
        }
        if (!ext && tid == 0) atomicMax(&info[r], now);
        tile_sort(list, tmp, end, now);
        beg = end;
        end = now;
        if (ext && tid == 0) roff[(size_t)t * (rings + 1) + r] = end;
    }
    if (!ext) return;
    if (tid < end) slot[tile_find(keys, list[tid])] = (uint16_t)tid;
    __syncthreads();
    if (tid < end) {
        const uint32_t v = list[tid];
        ids[(size_t)t * ext + tid] = v;
        if (tid < beg) {   // a row whose columns are all in the list
            const uint32_t len = O.rowlen[v];
            const size_t g = (size_t)O.slice_ptr[v >> 6] + (v & 63);
            for (uint32_t q = 0; q < W2; ++q) {
                uint32_t word = 0;
                for (uint32_t h = 0; h < 2; ++h) {
                    const uint32_t k = 2 * q + h;
                    const uint32_t s = k < len ? slot[tile_find(keys, O.bcol[g + (size_t)k * SLICE])]
                                               : tid;
                    word |= s << (16 * h);
                }
                lcol[((size_t)t * W2 + q) * ext + tid] = word;
            }
        }
    }
}

}  // namespace

void tiles_free(Tiles& T) {
    void* ps[] = {T.ids, T.lcol, T.roff};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    T = Tiles();
}

// Cuts the n rows at positions xy into the first of `attempts` whose tiles have
// at most `limit` rows with `least` rings or more (as many of its `rings` as
// fit) and whose owned rows touch at most `most_runs` groups of 8 consecutive
// ids.  Leaves T.n = 0 (nothing allocated) when none has, or
// without device memory for them: the kernels that take one step per launch
// then run.
template <class Len>
static int tiles_cut(Tiles& T, const TileRows<Len>& O, uint32_t n, uint32_t wmax, const double2* xy,
                     const std::vector<TileAttempt>& attempts, uint32_t limit, uint32_t most_runs,
                     hipStream_t s) {
    uint32_t *cell = nullptr, *cnt = nullptr, *ptr = nullptr, *own = nullptr;
    unsigned* info = nullptr;
    double* bb = nullptr;
    auto done = [&](int rc) {
        void* ps[] = {cell, cnt, ptr, own, info, bb};
        for (void* p : ps)
            if (p) (void)hipFree(p);
        if (rc != NBX_OK) tiles_free(T);
        return rc;
    };
    auto no_memory = [&]() {
        (void)hipGetLastError();
        tiles_free(T);
        return done(NBX_OK);
    };
    const unsigned gb = std::min(grid_for(n), 256u);
    if (hipMalloc(&bb, 4 * (size_t)gb * sizeof(double)) != hipSuccess) return no_memory();
    hipLaunchKernelGGL(k_tile_bbox, dim3(gb), dim3(BLOCK), 0, s, xy, n, bb);
    std::vector<double> hb(4 * (size_t)gb);
    if (copy_on(hb.data(), bb, hb.size() * sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess) {
        set_last_error("tiles: bounding box");
        return done(NBX_ERR_HIP);
    }
    double lo[4] = {INFINITY, INFINITY, INFINITY, INFINITY};
    for (size_t i = 0; i < hb.size(); ++i) lo[i % 4] = std::min(lo[i % 4], hb[i]);
    const double Lx = -lo[2] - lo[0], Ly = -lo[3] - lo[1];
    if (!(Lx >= 0.0) || !(Ly >= 0.0) || !std::isfinite(Lx) || !std::isfinite(Ly) ||
        !(Lx + Ly > 0.0))
        return done(NBX_OK);
    if (hipMalloc(&cell, (size_t)n * 4) != hipSuccess ||
        hipMalloc(&own, (size_t)n * 4) != hipSuccess ||
        hipMalloc(&info, INFO * sizeof(unsigned)) != hipSuccess)
        return no_memory();
    const uint32_t W2 = (wmax + 1) / 2;
    for (const auto& at : attempts) {
        const uint32_t rings = std::min(at.rings, RINGS_MAX);
        // at most so many cells, about square
        const double cells = (double)at.cells;
        const double fx = Lx > 0.0 && Ly > 0.0
                              ? std::min(std::max(1.0, std::round(sqrt(cells * Lx / Ly))), cells)
                              : (Lx > 0.0 ? cells : 1.0);
        const double fy = Ly > 0.0 ? std::max(1.0, std::floor(cells / fx)) : 1.0;
        TileGrid g{lo[0], lo[1], Lx > 0.0 ? fx / Lx : 0.0, Ly > 0.0 ? fy / Ly : 0.0,
                   (uint32_t)fx, (uint32_t)fy};
        const uint32_t nt = g.nx * g.ny;
        if (cnt) (void)hipFree(cnt);
        if (ptr) (void)hipFree(ptr);
        cnt = ptr = nullptr;
        if (hipMalloc(&cnt, (size_t)nt * 4) != hipSuccess ||
            hipMalloc(&ptr, ((size_t)nt + 1) * 4) != hipSuccess)
            return no_memory();
        hipLaunchKernelGGL(k_tile_zero, dim3(grid_for(nt)), dim3(BLOCK), 0, s, cnt, nt);
        hipLaunchKernelGGL(k_tile_zero, dim3(1), dim3(BLOCK), 0, s, (uint32_t*)info, INFO);
        hipLaunchKernelGGL(k_tile_count, dim3(grid_for(n)), dim3(BLOCK), 0, s, g, xy, n, cell, cnt);
        const int rc = scan_u32(cnt, ptr, nt, s);
        if (rc) return done(rc);
        hipLaunchKernelGGL(k_tile_zero, dim3(grid_for(nt)), dim3(BLOCK), 0, s, cnt, nt);
        hipLaunchKernelGGL(k_tile_fill, dim3(grid_for(n)), dim3(BLOCK), 0, s, cell, n, ptr, cnt, own,
                           limit, info);
        hipLaunchKernelGGL(k_tile_rings<Len>, dim3(nt), dim3(TILE_TB), 0, s, O, ptr, own, limit, rings,
                           wmax, W2, 0u, (uint32_t*)nullptr, (uint32_t*)nullptr, (uint32_t*)nullptr, info);
        unsigned hi[INFO];
        if (hipGetLastError() != hipSuccess ||
            copy_on(hi, info, sizeof hi, hipMemcpyDeviceToHost, s) != hipSuccess) {
            set_last_error("tiles: halo rings");
            return done(NBX_ERR_HIP);
        }
        if (hi[RUNS] > most_runs) return done(NBX_OK);
        uint32_t fit = hi[0] ? 0 : rings;
        while (fit && hi[fit] > limit) --fit;
        if (fit < at.least) continue;
        T.n = nt;
        T.most = hi[fit];
        T.ext = (T.most + WAVE - 1) / WAVE * WAVE;
        T.rings = fit;
        T.W2 = W2;
        break;
    }
    if (T.n == 0) return done(NBX_OK);
    if (hipMalloc(&T.ids, (size_t)T.n * T.ext * 4) != hipSuccess ||
        hipMalloc(&T.lcol, (size_t)T.n * T.ext * W2 * 4) != hipSuccess ||
        hipMalloc(&T.roff, (size_t)T.n * (T.rings + 1) * 4) != hipSuccess)
        return no_memory();
    hipLaunchKernelGGL(k_tile_rings<Len>, dim3(T.n), dim3(TILE_TB), 0, s, O, ptr, own, limit, T.rings, wmax, W2,
                       T.ext, T.ids, T.lcol, T.roff, info);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
        set_last_error("tiles: lists");
        return done(NBX_ERR_HIP);
    }
    return done(NBX_OK);
}

int tiles_build(Tiles& T, const Off16& O, uint32_t wmax, const double2* xy, hipStream_t s) {
    const uint32_t n = O.n_nodes;
    tiles_free(T);
    if (!xy || n == 0 || wmax == 0 || wmax > TILE_WMAX) return NBX_OK;
    // Tiles and rings (= steps per launch).  A launch takes as long as its
    // fullest CU, so the tiles are as many as run at once, or twice that, with
    // as many rings as a tile's TILE_TB rows leave room for; from 540k nodes
    // bytes bound a step, and 256 nodes with three rings read least per node.
    // At once: 256 tiles (one a CU: a row's values in FP64 registers, or the
    // rows of up to TILE_WMAX blocks), or 512 (two a CU, values in FP32).
    // us per outer iteration of the default solve (39 steps), with about 160 or
    // 256 owned nodes and 8, 5 or 3 rings before -> now.  Rows of six blocks,
    // 256 tiles: 64x32 54.9 -> 43.5, 150x75 56.7 -> 46.0, 256x128 58.9 -> 52.9,
    // 300x150 71.3 -> 55.8, 400x200 89.6 -> 73.4 (78.0 with 512 tiles); 512
    // tiles: 450x225 93.2 -> 85.6, 501x247 97.4 -> 93.9 (95 with 256), 570x285
    // 128 -> 104, 700x350 158 -> 131, 800x400 196 -> 180; 1,024: 900x450 271 ->
    // 249, 1024x512 279 -> 268; 2048x1024 937 (979 in rounds of 512).  Longer
    // rows: 33k nodes 74.5 -> 73.8, 80k 151 -> 97, 136k 230 -> 127, 193k 325 ->
    // 207; 263k 320 against 437 with a step per launch; beyond, with three rings,
    // 526k 878 against 657: a step per launch there.
    const bool six = O.width == 6;
    if (!six && n > 512 * 528u) return NBX_OK;
    uint32_t tiles = 256;
    if (six && n > 98304) tiles = n <= 512 * 640 ? 512 : 1024;
    if (!six && n > 256 * 640) tiles = 512;
    uint32_t own0 = std::max((n + tiles - 1) / tiles, 16u), rings0 = 3, least = 3;
    uint32_t limit = TILE_TB;
    if (n > 1024 * 528u) {
        own0 = 256;
        tiles = (n + own0 - 1) / own0;
        limit = 704;
    } else {
        // the rows of r rings around a square of own0 nodes of a triangle mesh
        auto rows = [&](uint32_t r) { return own0 + 4.0 * r * sqrt((double)own0) + 3.0 * r * r; };
        while (rings0 < 8 && rows(rings0 + 1) <= TILE_TB) ++rings0;
        least = std::max(rings0 / 2, six || tiles <= 256 ? 2u : 3u);
    }
    const uint32_t cells0 = std::max(std::min(tiles, n / own0), 1u);
    // A mesh of uneven density, or with wider rows, can outgrow a tile in a few
    // cells: fewer rings then, or (rows of six blocks, eight rings) twice the
    // cells with four.  Every tile takes the threads of the fullest and most
    // then own little, so more cells with fewer rings lose to a step per launch;
    // us per outer iteration of 1024x512 (541), spacing growing to three, five
    // times the first in x and y: 579, 904 with 2 and 4 times the cells and two
    // rings; 512x256 (275-318), growing ten times: 429.  In the three rings of
    // the largest meshes tiles of more than 704 rows do (1430x720, 834: of 664
    // 741, of 747 832, of 829 877).
    std::vector<TileAttempt> attempts{{cells0, rings0, least}};
    if (six && rings0 == 8) attempts.push_back({2 * cells0, 4, 4});
    // A tile reads its rows' blocks where the rows lie.  Where the matrix exceeds
    // the caches and the numbering scatters a tile's rows, each block is a line of
    // its own and the overlap costs more than the launches: nodes in random order,
    // single steps -> tiles: 620x310 524 -> 486, 724x362 705 -> 675, 850x425 907 ->
    // 948, 1024x512 1,332 -> 1,552, 1430x720 3,403 -> 4,227.  (In order 256 owned
    // rows touch about 50 groups of 8, scattered ones 256.)
    const uint32_t most_runs = n > 512 * 640 ? n / 2 : n;
    return tiles_cut(T, TileRows<uint8_t>{O.slice_ptr, O.rowlen, O.bcol}, n, wmax, xy, attempts,
                     limit, most_runs, s);
}

int tiles_build(Tiles& T, const TileRows<uint16_t>& O, uint32_t n, uint32_t wmax, const double2* xy,
                const std::vector<TileAttempt>& attempts, uint32_t limit, hipStream_t s) {
    tiles_free(T);
    if (!xy || n == 0 || wmax == 0) return NBX_OK;
    return tiles_cut(T, O, n, wmax, xy, attempts, std::min(limit, (uint32_t)TILE_TB), n, s);
}

}  // namespace nbx
