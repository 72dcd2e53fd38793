// batch.hip — many independent FP32 simulations advanced by one persistent
// kernel launch per step, optionally replayed from a hipGraph.
//
// The reference can run exactly one compile-time configuration per binary
// (src/params.h, src/device_solver.cu:123-125); here every simulation of a
// batch has its own grid, boundary tags and constants. Each simulation is an
// ordinary FP32 handle (own HBM buffers, slot table, diagnostics); the batch
// adds a device array of per-simulation descriptors and a work list of
// (simulation, tile) items that a persistent grid of blocks walks each step.
// A descriptor holds both ping-pong views of the simulation's buffers, so two
// consecutive steps differ only in a parity argument and can be captured once
// as a graph and replayed.
//
// Simulations with walls in x and y only (z periodic, no anchoring, no
// moving wall; the slit and channel presets) run the third pipeline's
// wall-aware form, which computes every cell in the one launch. Other
// simulations with walls take the split of the single-simulation path: the
// periodic specialisation over every tile is exact for the cells two or more
// cells from every open face, and two one-thread-per-cell passes with the
// full wall handling then overwrite their wall shells.
#define LBM_FUSED_BODY_ONLY
#include "step_kernels.hpp"
#include "fused_step.hpp"
#include "batch_split.hpp"
#include "solver_state.hpp"

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

using namespace lbm;

namespace {

struct SimDesc {
    Fields<float> f[2];   // [parity]: parity 1 swaps Q/Q', u/u', g/g'
    BCDesc<float> bc;
    Phys<float> k;
    int periodic;
    int ntx, nty, nzc;
    int tile_x, tile_y;   // columns of a tile (third pipeline)
    int tile_begin;       // first work item of this simulation
    int pull;             // 0 until the first step after an upload
    int aux_always;       // moving walls read rho every step
    int walls;            // third pipeline with its wall handling (no shell passes)
    ShellRegion r3, r2;   // shell and halo (Q pass), shell alone (force pass); empty if periodic or walls
    int sq_begin;         // first item of this simulation in the shell Q pass
    int sf_begin;         // first item of this simulation in the shell force pass
};

// Last simulation whose range starts at or before item w (ranges ascending;
// empty ranges share their start with the next simulation).
template <typename Get>
__device__ __forceinline__ int find_sim(int nsims, int w, Get begin_of) {
    int lo = 0, hi = nsims - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (begin_of(mid) <= w) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Tile shapes of the batched kernel: kind 0 runs the first fused pipeline
// over every tile (cells of the wall shells excluded, the shell passes write
// them), kind 1 the third pipeline (one barrier per plane; simulations with
// walls in x and y only are computed whole by its wall-aware form, others
// with walls have their shells rewritten by the shell passes, as on a single
// simulation).
struct BatchTile {
    int kind, tx, ty, zc;
    const char* name;
};
constexpr BatchTile kBatchTiles[] = {
    {0, 32, 8, 32, "32x8x32"},       {0, 16, 16, 32, "16x16x32"},     {0, 32, 8, 16, "32x8x16"},
    {0, 16, 16, 16, "16x16x16"},     {0, 16, 16, 8, "16x16x8"},       {0, 32, 8, 8, "32x8x8"},
    {1, 32, 8, 64, "p2:32x8x64"},    {1, 32, 8, 32, "p2:32x8x32"},    {1, 32, 8, 16, "p2:32x8x16"},
    {1, 64, 4, 32, "p2:64x4x32"},    {1, 0, 0, 64, "p2:rows:64"},
};
constexpr int kNumBatchTiles = sizeof(kBatchTiles) / sizeof(kBatchTiles[0]);

template <int TX, int TY, int ZC>
__global__ void __launch_bounds__(TX * TY)
batch_step_kernel(const SimDesc* __restrict__ descs, int nsims, int total, int parity, int aux) {
    using G = TileGeom<TX, TY>;
    __shared__ float sIn[kNumIn][G::NI];
    __shared__ float sA[2][kNumA][G::NA];
    __shared__ float sRing[3][kNumIn][G::NR];
    // Persistent blocks: every block walks the work list with a grid stride;
    // the exit condition (w >= total) is reached by every block.
    for (int w = blockIdx.x; w < total; w += gridDim.x) {
        const SimDesc& d = descs[find_sim(nsims, w, [&](int i) { return descs[i].tile_begin; })];
        const int local = w - d.tile_begin;
        const int tx = local % d.ntx, ty = (local / d.ntx) % d.nty, tz = local / (d.ntx * d.nty);
        const int a = aux | d.aux_always;
        fused_body<TX, TY, ZC, true>(d.f[parity], d.bc, d.k, d.pull, a, tx, ty, tz, sIn, sA, sRing,
                                     d.periodic ? 0 : 1);
        __syncthreads();
    }
}

// The work list on the third pipeline: block b runs the items
// [ranges[b].x, ranges[b].y), which the host has cut so that every block has
// the same work (see build_items). A simulation's advection scheme and walls
// pick the instantiation per work item (uniform over the block); its tile
// shape is a run-time value, which costs 2-3 % of a sweep of equal boxes,
// but one set of bodies for both shapes is what a mixed sweep's blocks share
// in the instruction cache (64 mixed boxes 313 us, compile-time shapes 316).
__global__ void __launch_bounds__(RowGeom::NT) __attribute__((amdgpu_waves_per_eu(2, 2)))
batch_step_kernel_p2(const SimDesc* __restrict__ descs, const BatchItem* __restrict__ items,
                     const int2* __restrict__ ranges, int parity, int aux) {
    using G = RowGeom;
    __shared__ float sIn[2][kNumIn][G::LI];
    __shared__ float sP[2][6][G::LA];
    __shared__ float sRing[4][kNumIn][G::LR];
    const int2 range = ranges[blockIdx.x];
    for (int w = range.x; w < range.y; ++w) {
        const BatchItem it = items[w];
        const SimDesc& d = descs[it.sim];
        const int tx = it.txy % d.ntx, ty = it.txy / d.ntx;
        const int a = aux | d.aux_always;
        const G geo(d.tile_x, d.tile_y);
        if (d.walls) {
            if (d.k.advection != 0)
                p2_range<false, true, true, false, true>(geo, d.f[parity], d.bc, d.k, d.pull, a, tx, ty, it.z0, it.z1,
                                                         sIn, sP, sRing);
            else
                p2_range<false, false, true, false, true>(geo, d.f[parity], d.bc, d.k, d.pull, a, tx, ty, it.z0, it.z1,
                                                          sIn, sP, sRing);
        } else if (d.k.advection != 0) {
            p2_range<true, true, true>(geo, d.f[parity], d.bc, d.k, d.pull, a, tx, ty, it.z0, it.z1, sIn, sP, sRing);
        } else {
            p2_range<true, false, true>(geo, d.f[parity], d.bc, d.k, d.pull, a, tx, ty, it.z0, it.z1, sIn, sP, sRing);
        }
        __syncthreads();
    }
}

// Wall shells of every simulation with walls, one thread per cell, in the
// two passes of the single-simulation path: the Q update over each shell and
// its one-cell halo, then body force and collide-stream of the shell cells.
__global__ void __launch_bounds__(kBlock)
batch_shell_q_kernel(const SimDesc* __restrict__ descs, int nsims, int total, int parity) {
    const int w = blockIdx.x * kBlock + threadIdx.x;
    if (w >= total) return;
    const SimDesc& d = descs[find_sim(nsims, w, [&](int i) { return descs[i].sq_begin; })];
    int q[3];
    region_cell(d.r3, d.bc.n, w - d.sq_begin, q);
    qstep_cell<true, false>(d.f[parity], d.bc, d.k, shell_node(q, d.bc.n), !cell_mask(d.bc, 1, q[0], q[1]).writes(q[2]));
}

__global__ void __launch_bounds__(kBlock)
batch_shell_force_kernel(const SimDesc* __restrict__ descs, int nsims, int total, int parity, int aux) {
    const int w = blockIdx.x * kBlock + threadIdx.x;
    if (w >= total) return;
    const SimDesc& d = descs[find_sim(nsims, w, [&](int i) { return descs[i].sf_begin; })];
    int q[3];
    region_cell(d.r2, d.bc.n, w - d.sf_begin, q);
    Fields<float> fq = d.f[parity];
    for (int m = 0; m < 5; ++m) fq.q[m] = fq.qn[m];   // the force reads Q^{n+1}
    const int flags = FL_FORCE | FL_LBM | ((aux | d.aux_always) ? (FL_STORE_F | FL_STORE_RHO) : 0);
    force_lbm_cell<float, true, true, true, true, false>(fq, d.bc, d.k, shell_node(q, d.bc.n), flags, d.pull);
}

template <int KIND, int TX, int TY, int ZC>
int occupancy_blocks() {
    int nb = 0;
    hipError_t e;
    if constexpr (KIND == 0)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, batch_step_kernel<TX, TY, ZC>, TX * TY, 0);
    else
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, batch_step_kernel_p2, RowGeom::NT, 0);
    return e == hipSuccess ? std::max(1, nb) : 1;
}

template <int KIND, int TX, int TY, int ZC>
void launch_batch(const SimDesc* d, int nsims, int total, const BatchItem* items, const int2* ranges, int parity,
                  int aux, int grid, hipStream_t s) {
    if constexpr (KIND == 0)
        hipLaunchKernelGGL((batch_step_kernel<TX, TY, ZC>), dim3(grid), dim3(TX * TY), 0, s, d, nsims, total,
                           parity, aux);
    else
        hipLaunchKernelGGL(batch_step_kernel_p2, dim3(grid), dim3(RowGeom::NT), 0, s, d, items, ranges, parity, aux);
}

// Every batch tile shape, in catalogue order: fn(TileTag<KIND, TX, TY, ZC>{}).
static_assert(kNumBatchTiles == 11, "the dispatch below lists every catalogue entry");
template <int K, int X, int Y, int Z>
struct TileTag {
    static constexpr int kind = K, tx = X, ty = Y, zc = Z;
};
template <typename F>
auto with_batch_tile(int tile, F&& fn) {
    switch (tile) {
        case 0: return fn(TileTag<0, 32, 8, 32>{});
        case 1: return fn(TileTag<0, 16, 16, 32>{});
        case 2: return fn(TileTag<0, 32, 8, 16>{});
        case 3: return fn(TileTag<0, 16, 16, 16>{});
        case 4: return fn(TileTag<0, 16, 16, 8>{});
        case 5: return fn(TileTag<0, 32, 8, 8>{});
        default: return fn(TileTag<1, 0, 0, 0>{});
    }
}

}  // namespace

struct lbm_batch {
    std::vector<lbm_handle> sims;
    std::vector<SimDesc> desc;
    SimDesc* d_desc = nullptr;
    // Third-pipeline tiles only: the items, and behind them each block's range of them.
    char* d_items = nullptr;
    size_t items_cap = 0;          // bytes
    std::vector<BatchItem> items;  // host copies (the upload reads them asynchronously)
    std::vector<int2> ranges;
    hipStream_t stream = nullptr;
    int total = 0;
    int sq_total = 0;      // cells of the shell Q pass (simulations with walls)
    int sf_total = 0;      // cells of the shell force pass
    int parity = 0;        // how far the buffers have ping-ponged since the handles were synced
    int tile = 0;
    int grid = 0;
    int grid_limit = 0;    // cap on the persistent grid (0: as many blocks as fit at once)
    bool desc_dirty = true;
    hipGraphExec_t graph[2] = {nullptr, nullptr};   // two steps starting at parity 0 / 1
};

namespace {

void drop_graphs(lbm_batch* b) {
    for (auto& g : b->graph)
        if (g) {
            (void)hipGraphExecDestroy(g);
            g = nullptr;
        }
}

int tiles_up(int n, int tile) { return (n + tile - 1) / tile; }

// Columns of a tile of simulation c: the catalogue's, or the shape of 64 x 4
// and 32 x 8 that covers the nx x ny columns with fewer tiles; 64 x 4 for as
// many (whole rows: 24 boxes of 48 x 64 x 64 take 258 us with it, 327 us with
// 32 x 8, whose tiles then begin inside cache lines; 18 boxes of 64^3 take
// 226 and 241 us). Tiles that fit the columns exactly but begin inside a line
// (24 x 10, 48 x 5) fetch up to three times the bytes: 698 and 406 us.
void tile_shape(const BatchTile& t, const lbm_config& c, int& tx, int& ty) {
    tx = t.tx;
    ty = t.ty;
    if (tx) return;
    long best = 0;
    for (int w = 64; w >= 32; w /= 2) {
        const int h = 256 / w;
        const long cost = (long)tiles_up(c.nx, w) * tiles_up(c.ny, h);
        if (tx == 0 || cost < best) {
            best = cost;
            tx = w;
            ty = h;
        }
    }
}

int tiles_of(const lbm_batch* b, int i, SimDesc& d) {
    const BatchTile& t = kBatchTiles[b->tile];
    const lbm_config& c = b->sims[i]->cfg;
    tile_shape(t, c, d.tile_x, d.tile_y);
    d.ntx = tiles_up(c.nx, d.tile_x);
    d.nty = tiles_up(c.ny, d.tile_y);
    d.nzc = tiles_up(c.nz, t.zc);
    return d.ntx * d.nty * d.nzc;
}

int grid_for_tile(int tile, int total, int limit) {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) {
        hipDeviceProp_t p;
        if (hipGetDeviceProperties(&p, dev) == hipSuccess) cus = p.multiProcessorCount;
    }
    const int occ = with_batch_tile(tile, [](auto t) {
        using T = decltype(t);
        return occupancy_blocks<T::kind, T::tx, T::ty, T::zc>();
    });
    const int grid = std::max(1, std::min(total, cus * occ));
    return limit > 0 ? std::min(grid, limit) : grid;
}

// Items and block ranges of the third-pipeline kernel (batch_split.hpp): one
// range of equal cost per resident block. Before, blocks drew chunks of 16, 32
// or 64 planes from a queue, longest first, so a sweep with fewer chunks than
// a few rounds of blocks waited for the last ones: 6 boxes of 24 to 64 per
// side 95 -> 40 us, 20 boxes 127 -> 97 us, 64 boxes 335 -> 308 us, 80 boxes
// 377 -> 357 us (with the tile shapes above and one loop body).
// Simulations of one form are neighbours in the order, so that a compute
// unit's blocks run the same body (18 boxes of 64^3, half of them slits: 256
// -> 240 us), and neighbouring ranges run on the same XCD (block b runs on
// XCD b mod 8), whose L2 then holds their shared halo columns.
int build_items(lbm_batch* b) {
    const int zc = kBatchTiles[b->tile].zc;
    int planes = 0;
    for (const SimDesc& d : b->desc) planes += d.ntx * d.nty * d.bc.n[2];
    const int slots = grid_for_tile(b->tile, planes, b->grid_limit);
    std::vector<BatchColumns> sims;
    for (size_t i = 0; i < b->desc.size(); ++i) {
        const SimDesc& d = b->desc[i];
        sims.push_back({(int)i, d.ntx * d.nty, d.bc.n[2], d.walls != 0});
    }
    auto form = [&](const BatchColumns& c) {
        const SimDesc& d = b->desc[c.sim];
        return 4 * (d.tile_x > 32) + 2 * d.walls + (d.k.advection != 0);
    };
    std::stable_sort(sims.begin(), sims.end(),
                     [&](const BatchColumns& x, const BatchColumns& y) { return form(x) < form(y); });
    BatchSplit split = split_columns(sims, zc, slots);
    const int n = split.ranges();
    b->items = std::move(split.items);
    b->ranges.resize(n);
    for (int r = 0, q = n / 8, m = n % 8; r < n; ++r) {
        const int xcd = r % 8, at = xcd * q + std::min(xcd, m) + r / 8;
        b->ranges[r] = int2{split.first[at], split.first[at + 1]};
    }
    const size_t item_bytes = b->items.size() * sizeof(BatchItem), range_bytes = n * sizeof(int2);
    if (item_bytes + range_bytes > b->items_cap) {
        if (b->d_items) (void)hipFree(b->d_items);
        b->d_items = nullptr;
        b->items_cap = 0;
        if (hipMalloc(&b->d_items, item_bytes + range_bytes) != hipSuccess)
            return fail(LBM_ERR_HIP, "hipMalloc(batch items) failed");
        b->items_cap = item_bytes + range_bytes;
    }
    if (hipMemcpyAsync(b->d_items, b->items.data(), item_bytes, hipMemcpyHostToDevice, b->stream) != hipSuccess ||
        hipMemcpyAsync(b->d_items + item_bytes, b->ranges.data(), range_bytes, hipMemcpyHostToDevice, b->stream) !=
            hipSuccess)
        return fail(LBM_ERR_HIP, "batch item upload failed");
    b->total = (int)b->items.size();
    b->grid = n;
    return LBM_OK;
}

// Build the descriptors from the handles' current buffers (parity 0 view).
int rebuild(lbm_batch* b) {
    b->desc.resize(b->sims.size());
    int begin = 0, sq_begin = 0, sf_begin = 0;
    for (size_t i = 0; i < b->sims.size(); ++i) {
        lbm_solver* s = b->sims[i];
        SimDesc& d = b->desc[i];
        d.f[0] = s->d32;
        d.f[1] = s->d32;
        for (int m = 0; m < 5; ++m) std::swap(d.f[1].q[m], d.f[1].qn[m]);
        for (int m = 0; m < 3; ++m) std::swap(d.f[1].u[m], d.f[1].un[m]);
        std::swap(d.f[1].g, d.f[1].gn);
        d.bc = s->bc32;
        d.k = s->k32;
        d.periodic = 1;
        for (int f = 0; f < 6; ++f)
            if (s->cfg.walls[f].qbc != LBM_Q_PERIODIC || s->cfg.walls[f].ubc != LBM_U_PERIODIC) d.periodic = 0;
        d.tile_begin = begin;
        begin += tiles_of(b, (int)i, d);
        d.pull = s->pulled;
        d.aux_always = s->moving ? 1 : 0;
        d.walls = (!d.periodic && kBatchTiles[b->tile].kind == 1 && p2_walls_ok(d.bc)) ? 1 : 0;
        d.r3 = d.walls ? ShellRegion{} : make_shell_region(d.bc, 3);
        d.r2 = d.walls ? ShellRegion{} : make_shell_region(d.bc, 2);
        d.sq_begin = sq_begin;
        d.sf_begin = sf_begin;
        sq_begin += (int)region_cells(d.r3);
        sf_begin += (int)region_cells(d.r2);
    }
    b->total = begin;
    b->grid = grid_for_tile(b->tile, b->total, b->grid_limit);
    if (kBatchTiles[b->tile].kind == 1)
        if (int r = build_items(b)) return r;
    b->sq_total = sq_begin;
    b->sf_total = sf_begin;
    if (hipMemcpyAsync(b->d_desc, b->desc.data(), b->desc.size() * sizeof(SimDesc), hipMemcpyHostToDevice,
                       b->stream) != hipSuccess)
        return fail(LBM_ERR_HIP, "descriptor upload failed");
    if (hipStreamSynchronize(b->stream) != hipSuccess) return fail(LBM_ERR_HIP, "descriptor upload failed");
    b->desc_dirty = false;
    drop_graphs(b);
    return LBM_OK;
}

// Bring every handle's buffer pointers in line with the batch parity so
// per-simulation calls (upload, download, diagnostics) see the current state.
int sync_handles(lbm_batch* b) {
    if (hipStreamSynchronize(b->stream) != hipSuccess) return fail(LBM_ERR_HIP, "batch synchronize failed");
    if (b->parity) {
        for (lbm_solver* s : b->sims) {
            for (int m = 0; m < 5; ++m) std::swap(s->d32.q[m], s->d32.qn[m]);
            for (int m = 0; m < 3; ++m) std::swap(s->d32.u[m], s->d32.un[m]);
            std::swap(s->d32.g, s->d32.gn);
        }
        b->parity = 0;
        b->desc_dirty = true;
    }
    return LBM_OK;
}

void launch_step(lbm_batch* b, int aux) {
    const int n = (int)b->sims.size();
    with_batch_tile(b->tile, [&](auto t) {
        using T = decltype(t);
        launch_batch<T::kind, T::tx, T::ty, T::zc>(b->d_desc, n, b->total, (const BatchItem*)b->d_items,
                                                   (const int2*)(b->d_items + b->items.size() * sizeof(BatchItem)),
                                                   b->parity, aux, b->grid, b->stream);
    });
    if (b->sf_total > 0) {
        hipLaunchKernelGGL(batch_shell_q_kernel, dim3(grid_for(b->sq_total)), dim3(kBlock), 0, b->stream, b->d_desc,
                           n, b->sq_total, b->parity);
        hipLaunchKernelGGL(batch_shell_force_kernel, dim3(grid_for(b->sf_total)), dim3(kBlock), 0, b->stream,
                           b->d_desc, n, b->sf_total, b->parity, aux);
    }
}

// One step outside any graph; afterwards every simulation pulls.
int plain_step(lbm_batch* b, int aux) {
    if (b->desc_dirty)
        if (int r = rebuild(b)) return r;
    launch_step(b, aux);
    if (hipGetLastError() != hipSuccess) return fail(LBM_ERR_HIP, "batch step launch failed");
    b->parity ^= 1;
    bool any_fresh = false;
    for (auto& d : b->desc) any_fresh = any_fresh || d.pull == 0;
    if (any_fresh) {
        for (lbm_solver* s : b->sims) s->pulled = 1;
        for (auto& d : b->desc) d.pull = 1;
        if (hipMemcpyAsync(b->d_desc, b->desc.data(), b->desc.size() * sizeof(SimDesc), hipMemcpyHostToDevice,
                           b->stream) != hipSuccess)
            return fail(LBM_ERR_HIP, "descriptor upload failed");
        drop_graphs(b);
    }
    return LBM_OK;
}

int graph_pair(lbm_batch* b) {
    hipGraphExec_t& ge = b->graph[b->parity];
    if (!ge) {
        hipGraph_t g = nullptr;
        if (hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal) != hipSuccess)
            return fail(LBM_ERR_HIP, "graph capture failed to start");
        launch_step(b, 0);
        b->parity ^= 1;
        launch_step(b, 0);
        b->parity ^= 1;
        if (hipStreamEndCapture(b->stream, &g) != hipSuccess) return fail(LBM_ERR_HIP, "graph capture failed");
        const hipError_t e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
            ge = nullptr;
            return fail(LBM_ERR_HIP, "graph instantiate failed");
        }
    }
    if (hipGraphLaunch(ge, b->stream) != hipSuccess) return fail(LBM_ERR_HIP, "graph launch failed");
    return LBM_OK;   // two steps: parity unchanged
}

int batch_steps(lbm_batch* b, int n, int use_graph) {
    if (n <= 0) return LBM_OK;
    int done = 0;
    if (b->desc_dirty)
        if (int r = rebuild(b)) return r;
    bool fresh = false;
    for (auto& d : b->desc) fresh = fresh || d.pull == 0;
    if (fresh) {
        if (int r = plain_step(b, n == 1)) return r;
        done = 1;
    }
    if (use_graph) {
        while (n - done > 2) {
            if (int r = graph_pair(b)) return r;
            done += 2;
        }
    }
    while (done < n) {
        if (int r = plain_step(b, done == n - 1)) return r;
        ++done;
    }
    return LBM_OK;
}

}  // namespace

extern "C" {

int lbm_batch_create(const lbm_config* cfgs, int32_t count, lbm_batch_handle* out) {
    if (!cfgs || !out || count < 1) return fail(LBM_ERR_INVALID, "bad argument");
    *out = nullptr;
    for (int i = 0; i < count; ++i)
        if (cfgs[i].precision != LBM_FP32_SHIFTED)
            return fail(LBM_ERR_UNSUPPORTED, "batched simulations must use LBM_FP32_SHIFTED");
    lbm_batch* b = new lbm_batch();
    auto bail = [&](int r) {
        lbm_batch_destroy(b);
        return r;
    };
    for (int i = 0; i < count; ++i) {
        lbm_handle h = nullptr;
        if (int r = lbm_create(&cfgs[i], &h)) return bail(r);
        b->sims.push_back(h);
        if (!h->fused_ok) return bail(fail(LBM_ERR_UNSUPPORTED, "simulation too large for the batched kernel"));
    }
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(LBM_ERR_HIP, "hipStreamCreate failed"));
    if (hipMalloc(&b->d_desc, count * sizeof(SimDesc)) != hipSuccess)
        return bail(fail(LBM_ERR_HIP, "hipMalloc(descriptors) failed"));
    if (int r = rebuild(b)) return bail(r);
    *out = b;
    return LBM_OK;
}

int lbm_batch_destroy(lbm_batch_handle b) {
    if (!b) return LBM_OK;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    drop_graphs(b);
    for (lbm_handle h : b->sims) lbm_destroy(h);
    if (b->d_desc) (void)hipFree(b->d_desc);
    if (b->d_items) (void)hipFree(b->d_items);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
    return LBM_OK;
}

int lbm_batch_upload_state(lbm_batch_handle b, int32_t sim, const double* rho, const double* ux, const double* uy,
                           const double* uz, const double* q) {
    if (!b || sim < 0 || sim >= (int)b->sims.size()) return fail(LBM_ERR_INVALID, "bad simulation index");
    if (int r = sync_handles(b)) return r;
    if (int r = lbm_upload_state(b->sims[sim], rho, ux, uy, uz, q)) return r;
    b->desc_dirty = true;
    return LBM_OK;
}

int lbm_batch_download_state(lbm_batch_handle b, int32_t sim, double* rho, double* ux, double* uy, double* uz,
                             double* q) {
    if (!b || sim < 0 || sim >= (int)b->sims.size()) return fail(LBM_ERR_INVALID, "bad simulation index");
    if (int r = sync_handles(b)) return r;
    return lbm_download_state(b->sims[sim], rho, ux, uy, uz, q);
}

int lbm_batch_diagnostics(lbm_batch_handle b, int32_t sim, lbm_diag* out) {
    if (!b || sim < 0 || sim >= (int)b->sims.size()) return fail(LBM_ERR_INVALID, "bad simulation index");
    if (int r = sync_handles(b)) return r;
    return lbm_diagnostics(b->sims[sim], out);
}

int lbm_batch_step(lbm_batch_handle b, int32_t n, int32_t use_graph) {
    if (!b || n < 0) return fail(LBM_ERR_INVALID, "bad argument");
    return batch_steps(b, n, use_graph);
}

int lbm_batch_time_steps(lbm_batch_handle b, int32_t n, int32_t use_graph, double* ms) {
    if (!b || !ms || n < 1) return fail(LBM_ERR_INVALID, "bad argument");
    if (b->desc_dirty)
        if (int r = rebuild(b)) return r;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        if (e0) (void)hipEventDestroy(e0);
        return fail(LBM_ERR_HIP, "hipEventCreate failed");
    }
    (void)hipEventRecord(e0, b->stream);
    int r = batch_steps(b, n, use_graph);
    (void)hipEventRecord(e1, b->stream);
    (void)hipEventSynchronize(e1);
    float f = 0.0f;
    (void)hipEventElapsedTime(&f, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = f;
    return r;
}

int lbm_batch_tile_count(void) { return kNumBatchTiles; }

int lbm_batch_tile_name(int32_t tile, char* buf, size_t len) {
    if (!buf || !len) return fail(LBM_ERR_INVALID, "null buffer");
    if (tile < 0 || tile >= kNumBatchTiles) return fail(LBM_ERR_INVALID, "tile out of range");
    std::strncpy(buf, kBatchTiles[tile].name, len - 1);
    buf[len - 1] = 0;
    return LBM_OK;
}

int lbm_batch_set_tile(lbm_batch_handle b, int32_t tile) {
    if (!b || tile < 0 || tile >= kNumBatchTiles) return fail(LBM_ERR_INVALID, "tile out of range");
    if (int r = sync_handles(b)) return r;
    b->tile = tile;
    b->desc_dirty = true;
    return LBM_OK;
}

int lbm_batch_autotune(lbm_batch_handle b, int32_t n, double* ms_out, int32_t max, int32_t* count) {
    if (!b || n < 1) return fail(LBM_ERR_INVALID, "bad argument");
    if (count) *count = 0;
    if (int r = sync_handles(b)) return r;
    // Tune on scratch copies of every simulation's state, then restore.
    std::vector<std::vector<double>> saved(b->sims.size());
    for (size_t i = 0; i < b->sims.size(); ++i) {
        lbm_solver* s = b->sims[i];
        const long V = s->V;
        saved[i].resize(9 * V + 15 * V);
        double* p = saved[i].data();
        if (int r = lbm_download_state(s, p, p + V, p + 2 * V, p + 3 * V, p + 4 * V)) return r;
        if (int r = lbm_download_populations(s, p + 9 * V)) return r;
    }
    double best = 1e300;
    int best_t = 0;
    for (int t = 0; t < kNumBatchTiles; ++t) {
        if (int r = lbm_batch_set_tile(b, t)) return r;
        double ms = 0.0;
        if (int r = batch_steps(b, 2, 0)) return r;
        if (int r = lbm_batch_time_steps(b, n, 1, &ms)) return r;
        if (ms_out && t < max) ms_out[t] = ms / n;
        if (ms < best) {
            best = ms;
            best_t = t;
        }
    }
    if (int r = lbm_batch_set_tile(b, best_t)) return r;
    for (size_t i = 0; i < b->sims.size(); ++i) {
        lbm_solver* s = b->sims[i];
        const long V = s->V;
        double* p = saved[i].data();
        if (int r = lbm_upload_state(s, p, p + V, p + 2 * V, p + 3 * V, p + 4 * V)) return r;
        if (int r = lbm_upload_populations(s, p + 9 * V)) return r;
        s->pulled = 0;
    }
    b->desc_dirty = true;
    if (count) *count = std::min(kNumBatchTiles, (int)max);
    return LBM_OK;
}

int lbm_batch_set_grid_limit(lbm_batch_handle b, int32_t max_blocks) {
    if (!b || max_blocks < 0) return fail(LBM_ERR_INVALID, "bad argument");
    if (int r = sync_handles(b)) return r;
    b->grid_limit = max_blocks;
    b->desc_dirty = true;
    return LBM_OK;
}

int lbm_batch_get_tile(lbm_batch_handle b, int32_t* tile) {
    if (!b || !tile) return fail(LBM_ERR_INVALID, "null argument");
    *tile = b->tile;
    return LBM_OK;
}

}  // extern "C"
