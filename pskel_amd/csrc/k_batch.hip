// Batched persistent sweeps: many uneven 2D grids advanced together.
//
// The reference runs one Stencil at a time, one launch + sync per sweep
// (include/PSkelStencil.hpp:1078-1082, 1790-1791); a workload of hundreds of
// small grids is then launch-bound.  Here one persistent kernel per launch
// covers every tile of every grid: a fixed set of blocks walks a work list of
// (grid, tile) items round-robin (static order: deterministic, every block exits
// after its last item), each item running the body of the standalone kernels
// with the grid's kernel family (Jacobi f32, 3x3 weighted f32, life u8) and
// tile shape.  The sequence of launches is captured once in a hipGraph and
// replayed; each family's kernels run on a stream of their own, side by side
// with the other families' (no grid belongs to two).
//
// Temporal depth.  Each grid fuses K sweeps per launch (K odd: 1 or 3 for the
// f32 stencils, on register tiles (k_rtile2d.hpp) or, where those do not run
// or are slower, the LDS temporal tile; 1, 3, 5 or 7 for life, on bit-packed tiles
// (k_ltile.hpp); K = 1 runs the one-sweep tiles of k_tiles2d.hpp).  A grid of
// a family that holds its tiles in registers (bit-packed life, the f32 register
// tiles) fuses as many sweeps as pay for the whole family, at least the depths
// its grids ask for: plan_batch picks it for each run length.  An odd number of
// sweeps per launch moves the state to the other buffer, so grid g's launch l reads
// buffer l & 1 and writes the other, with no third buffer.  N sweeps of grid g
// run as N / K launches of K, then the rest r = N mod K as one launch of r
// (odd) or two of r - 1 and 1 (even r): n_g launches.  Where launches of the depth
// asked for end in a single sweep, so do these (N - 1 sweeps as above, then 1): the
// other buffer then holds the state before it.  Work items are ordered by
// n_g, longest first, so launch l's items are a prefix of the list.
#include <algorithm>
#include <cstring>
#include <numeric>
#include <vector>

#include "k_tiles2d.hpp"
#include "k_march2d.hpp"
#define PSKEL_RTILE_INSTANTIATE
#include "k_rtile2d.hpp"
#define PSKEL_LTILE_INSTANTIATE
#include "k_ltile.hpp"

using namespace pskel;

namespace {

enum BatchKind : int { BK_J5 = 0, BK_BOX9 = 1, BK_LIFE = 2 };

// One grid of the batch (device table entry).
struct BatchEntry {
    void* buf[2];     // launch l reads buf[l & 1] and writes buf[(l & 1) ^ 1]
    int W, H;
    int pitch;
    int radius;
    int kind;
    int ry;           // K = 1: rows per lane; LDS tiles: tile rows
    int rtile;        // f32 at K = 3 on register tiles (choose_f32_tiles)
    int depth;        // K, sweeps fused per launch (odd); of a tile family: the tiles' halo
    int full;         // launches of K sweeps
    int tail0, tail1, tail2;  // sweeps of the launches after them (odd; 0: none)
    int tiles_x;      // tiles along w
    int ntiles;       // tiles of the grid
    int item0;        // first work item of this grid
    float coeff;
    float wt[9];
};

constexpr int kBatchWaves = 4;  // block = (64, 4)
constexpr int kTTileCX = 120;   // columns of an f32 temporal tile
constexpr int kTTileK = 3;      // depth of the f32 temporal tiles
// register and bit-packed life tiles: 8 waves of 8 rows (a 64-row tile keeps 58
// rows of its own at 3 sweeps, 50 at 7 generations)
constexpr int kBatchTileWaves = 8;
constexpr int kBatchTileRows = 8;
constexpr int kBatchTileH = kBatchTileWaves * kBatchTileRows;
constexpr int kBatchLds = ttile_lds<kTTileK, kTTileCX, 32>();  // floats per LDS buffer (the largest tile)

__device__ __forceinline__ int sweeps_of(const BatchEntry& E, int launch)
{
    if (launch < E.full) return E.depth;
    if (launch == E.full) return E.tail0;
    if (launch == E.full + 1) return E.tail1;
    if (launch == E.full + 2) return E.tail2;
    return 0;
}

template <int RY>
__device__ __forceinline__ void run_item(const BatchEntry& E, const Sweep2D& s, int t)
{
    const int tx = t % E.tiles_x, ty = t / E.tiles_x;
    if (E.kind == BK_LIFE) {
        tile_life<RY>(s, tx, ty);
    } else if (E.kind == BK_J5) {
        tile_f32<PAT_J5, RY>(s, E, tx, ty);
    } else {
        tile_f32<PAT_BOX9, RY>(s, E, tx, ty);
    }
}

template <int PAT>
__device__ __forceinline__ void run_ttile(const BatchEntry& E, const Sweep2D& s, int t, int k, float* A, float* B)
{
    const int tid = (int)threadIdx.y * kWave + (int)threadIdx.x;
    const int tx = t % E.tiles_x, ty = t / E.tiles_x;
    if (E.ry == 16) ttile_body<PAT, kTTileK, kTTileCX, 16>(s, E, tx, ty, k, tid, A, B);
    else ttile_body<PAT, kTTileK, kTTileCX, 32>(s, E, tx, ty, k, tid, A, B);
}

// Work families, one kernel each so each keeps the registers its body needs
// (one-sweep tiles, f32 LDS temporal tiles, bit-packed life tiles, f32 register
// tiles of the 5-point and the 3x3 stencil, which need 76 and 88 registers, and
// 130 in one kernel).
enum BatchFamily : int { BF_REG = 0, BF_TTILE = 1, BF_BITS = 2, BF_J5 = 3, BF_BOX9 = 4, BF_COUNT = 5 };

// waves per block
constexpr int fam_waves(int fam) { return fam >= BF_BITS ? kBatchTileWaves : kBatchWaves; }

template <int FAM>
struct FamLds {
    float lds[FAM == BF_TTILE ? 2 * kBatchLds : 1];
};
template <>
struct FamLds<BF_BITS> : LtLds<kBatchTileRows, kBatchTileWaves> {};
template <>
struct FamLds<BF_J5> : RtLds<kBatchTileRows, kBatchTileWaves> {};
template <>
struct FamLds<BF_BOX9> : RtLds<kBatchTileRows, kBatchTileWaves> {};

// (the life tiles fit 64 registers, four blocks per CU)
template <int FAM>
__global__ __launch_bounds__(fam_waves(FAM) * kWave, FAM == BF_BITS ? 8 : 1) void k_batch(
    const BatchEntry* __restrict__ tab, const int* __restrict__ item_grid, int nitems, int launch)
{
    __shared__ FamLds<FAM> L;
    const int parity = launch & 1;
    for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
        const int g = item_grid[item];
        const BatchEntry& E = tab[g];
        const int k = sweeps_of(E, launch);  // uniform across the block
        if (k == 0) continue;
        const int t = item - E.item0;
        Sweep2D s;
        s.src = E.buf[parity];
        s.dst = E.buf[parity ^ 1];
        s.ring_other = E.buf[parity ^ 1];
        s.W = E.W;
        s.H = E.H;
        s.pitch = (size_t)E.pitch;
        s.radius = E.radius;
        if constexpr (FAM == BF_REG) {
            switch (E.ry) {
            case 1: run_item<1>(E, s, t); break;
            case 2: run_item<2>(E, s, t); break;
            case 4: run_item<4>(E, s, t); break;
            default: run_item<8>(E, s, t); break;
            }
        } else if constexpr (FAM >= BF_BITS) {
            const int lane = (int)threadIdx.x, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
            const int tx = t % E.tiles_x, ty = t / E.tiles_x;
            if constexpr (FAM == BF_BITS) {
                life_tile<kBatchTileRows, kBatchTileWaves, false>(s, tx, ty, E.depth, k, lane, wave, L);
            } else {
                RtParams p;
                p.coeff = E.coeff;
#pragma unroll
                for (int i = 0; i < 9; ++i) p.wt[i] = E.wt[i];
                rt_tile<FAM == BF_J5 ? PAT_J5 : PAT_BOX9, kBatchTileRows, kBatchTileWaves, false, false>(
                    s, p, tx, ty, E.depth, k, lane, wave, L);
            }
            __syncthreads();  // the next item's first rows go where this one's last may still be read
        } else {
            if (E.kind == BK_J5) run_ttile<PAT_J5>(E, s, t, k, L.lds, L.lds + kBatchLds);
            else run_ttile<PAT_BOX9>(E, s, t, k, L.lds, L.lds + kBatchLds);
        }
    }
}

int family_of(const BatchEntry& e)
{
    if (e.depth == 1) return BF_REG;
    if (e.kind == BK_LIFE) return BF_BITS;
    if (e.rtile) return e.kind == BK_J5 ? BF_J5 : BF_BOX9;
    return BF_TTILE;
}

// the schedule of N sweeps at depth K: full launches of K, then the tail; it ends in
// a single sweep where the schedule at depth `asked` does
void schedule(BatchEntry& e, size_t n, int asked)
{
    const int K = e.depth;
    auto split = [&](size_t m) {
        e.full = (int)(m / K);
        const int r = (int)(m % K);
        e.tail0 = e.tail1 = e.tail2 = 0;
        if (r % 2 == 1) e.tail0 = r;
        else if (r > 0) {
            e.tail0 = r - 1;
            e.tail1 = 1;
        }
    };
    split(n);
    const size_t rest = n % (size_t)asked;
    const bool single = asked == 1 || rest == 1 || (rest > 0 && rest % 2 == 0);
    if (!single || (e.tail1 ? e.tail1 : e.tail0 ? e.tail0 : K) == 1) return;
    split(n - 1);
    (e.tail0 == 0 ? e.tail0 : e.tail1 == 0 ? e.tail1 : e.tail2) = 1;
}

// tiles of a grid of a register-tile family at depth K
void tile_grid(BatchEntry& e, int K)
{
    e.depth = K;
    if (e.kind == BK_LIFE) {
        e.tiles_x = lt_tiles(e.W, kLtCols, 32);
    } else {
        e.tiles_x = rt_tiles(e.W, kRtCols, rt_halo_cols(K));
    }
    e.ntiles = e.tiles_x * rt_tiles(e.H, kBatchTileH, K);
}

// LDS tiles of a grid: 3 sweeps, e.ry rows
void lds_grid(BatchEntry& e)
{
    e.depth = kTTileK;
    e.tiles_x = (e.W + kTTileCX - 1) / kTTileCX;
    e.ntiles = e.tiles_x * ((e.H + e.ry - 1) / e.ry);
}

int launches_of(const BatchEntry& e) { return e.full + (e.tail0 > 0) + (e.tail1 > 0) + (e.tail2 > 0); }

}  // namespace

struct pskel_batch {
    std::vector<pskel_grid_t*> grids;
    std::vector<BatchEntry> host_tab;
    BatchEntry* d_tab = nullptr;
    int* d_items = nullptr;          // the work items of each family, one list after the other
    size_t items_cap = 0;
    std::vector<int> asked;          // depth asked for each grid
    // f32 grids that fit the register tiles and the LDS tiles: 1 LDS tiles named, 2 the
    // register march (0: others)
    std::vector<char> either;
    int fam_slots[BF_COUNT] = {};    // blocks of a family's kernel the device holds at once
    int fam_items[BF_COUNT] = {};    // items per family
    int fam_first[BF_COUNT] = {};    // offset of a family's list in d_items
    int fam_blocks[BF_COUNT] = {};   // persistent blocks of a family's kernel
    std::vector<int> launch_items[BF_COUNT];  // items of launch l: a prefix of the family's list
    int nlaunch = 0;
    int nitems = 0;
    int nblocks = 0;
    int device = 0;
    size_t sched_sweeps = 0;        // iteration count the schedule and item order are for
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // one stream per kernel family (default priority): no grid belongs to two
    // families, so the families' launch sequences run side by side, forked
    // from and joined back into the issuing stream by events
    hipStream_t fam_stream[BF_COUNT] = {};
    hipEvent_t fork = nullptr, join[BF_COUNT] = {};
    hipGraphExec_t exec = nullptr;
    size_t graph_sweeps = 0;
};

namespace {

// items per family, their places in the list, and the blocks that walk them: at
// most as many as the device holds at once, so no block waits for a slot with a
// full share of items
void count_items(pskel_batch_t* b)
{
    b->nitems = 0;
    for (int f = 0; f < BF_COUNT; ++f) b->fam_items[f] = 0;
    for (const auto& e : b->host_tab) {
        b->fam_items[family_of(e)] += e.ntiles;
        b->nitems += e.ntiles;
    }
    for (int f = 0; f < BF_COUNT; ++f) {
        b->fam_first[f] = f ? b->fam_first[f - 1] + b->fam_items[f - 1] : 0;
        b->fam_blocks[f] = std::max(1, std::min(b->fam_items[f], b->fam_slots[f]));
    }
}

// The depth of a register-tile family for runs of n sweeps: odd, at least what
// each of its grids asked for and at most n, with the least time for the run's launches
// (the tiles' halo grows with it, the crossings of memory and the launches get
// fewer).  A batched launch costs about 8 us more than one of a single grid (the
// item and table lookups, the graph's steps).  Measured, 105 sweeps of the f32
// half of 16, 48 and 256 grids of 64 to 2048 a side: depth 3 285, 573 and 2061
// us; the picks 21, 13 and 7 185, 332 and 1270; the life half: depth 7 216, 287
// and 600 us; the picks 21, 15 and 7 168, 238 and 600.
constexpr double kBatchLaunchUs = 8.0;

int family_depth(const pskel_batch_t* b, int f, size_t n)
{
    const bool life = f == BF_BITS;
    int lo = 0;
    double cells = 0.0;
    for (size_t i = 0; i < b->host_tab.size(); ++i) {
        const BatchEntry& e = b->host_tab[i];
        if (family_of(e) != f) continue;
        lo = std::max(lo, b->asked[i]);
        cells += (double)e.W * e.H;
    }
    int best = lo;
    double best_t = 0.0;
    for (int K = lo; K <= 21 && (K == lo || (size_t)K <= n); K += 2) {
        int64_t nb = 0;
        for (const BatchEntry& e : b->host_tab) {
            if (family_of(e) != f) continue;
            BatchEntry t = e;
            tile_grid(t, K);
            nb += t.ntiles;
        }
        BatchEntry t{};
        t.depth = K;
        schedule(t, n, lo);
        const int per_cu = std::max(1, b->fam_slots[f] / kRtCus);
        const double one = life ? lt_launch_time(kBatchTileH, per_cu, nb, cells, K)
                                : rt_launch_time(f == BF_J5 ? PAT_J5 : PAT_BOX9, kBatchTileH, per_cu, nb, cells, K);
        const double time = (one + kBatchLaunchUs) * launches_of(t);
        if (K == lo || time < best_t) {
            best = K;
            best_t = time;
        }
    }
    return best;
}

// Register or LDS tiles for the f32 grids that fit both, for runs of n sweeps.  Where
// the launch names LDS tiles: the 3x3 stencil's 64-row register tiles take 2 us a sweep however few
// there are, so they need about one for every second CU (a 700 x 900 grid, 52 tiles,
// 12 sweeps: LDS 37 us, register 48; 24 grids, 325 tiles: 0.87 times the LDS time),
// and grids up to 120 wide leave half their lanes idle (4 grids of 20000 x 30, 105
// sweeps 1197 and 1533; a few among wider ones ride along).  And the LDS tiles run
// both stencils in one kernel: a kernel more costs a run about 20 us, the graph's fork
// and join (4 to 48 mixed grids, 3 sweeps, 2.2 to 2.4 times the LDS time), which the
// register tiles win back at 0.3 (5-point) and 0.5 us (3x3) per million cells and sweep.
void choose_f32_tiles(pskel_batch_t* b, size_t n)
{
    double mj = 0.0, mb = 0.0, narrow = 0.0;  // million cells
    int64_t box_tiles = 0;
    bool march = false;
    for (size_t i = 0; i < b->host_tab.size(); ++i) {
        if (!b->either[i]) continue;
        BatchEntry t = b->host_tab[i];
        tile_grid(t, kTTileK);
        const double m = 1e-6 * t.W * t.H;
        if (t.kind == BK_J5) {
            mj += m;
        } else {
            mb += m;
            if (t.W <= kTTileCX) narrow += m;
            box_tiles += t.ntiles;
            march |= b->either[i] == 2;
        }
    }
    bool box = march || (box_tiles >= (n < 20 ? 200 : 130) && narrow < 0.5 * mb), j5 = true;
    if (mj > 0.0 && mb > 0.0 && (0.3 * mj + (box ? 0.5 * mb : 0.0)) * (double)n <= 20.0) box = j5 = false;
    for (size_t i = 0; i < b->host_tab.size(); ++i) {
        if (!b->either[i]) continue;
        BatchEntry& e = b->host_tab[i];
        e.rtile = e.kind == BK_J5 ? j5 : box;
        if (e.rtile) tile_grid(e, kTTileK);
        else lds_grid(e);
    }
}

// Depths, schedules and item order for `n` sweeps: in each family's list, grids
// with more launches first.
pskel_status_t plan_batch(pskel_batch_t* b, size_t n)
{
    const size_t ng = b->host_tab.size();
    choose_f32_tiles(b, n);
    count_items(b);
    for (int f = BF_BITS; f < BF_COUNT; ++f) {
        if (b->fam_items[f] == 0) continue;
        const int K = family_depth(b, f, n);
        for (auto& e : b->host_tab)
            if (family_of(e) == f) tile_grid(e, K);
    }
    count_items(b);
    if ((size_t)b->nitems > b->items_cap) {
        // the list of the last run length is no longer in use: runs wait for their launches
        if (b->d_items) (void)hipFree(b->d_items);
        b->d_items = nullptr;
        b->items_cap = 0;
        PSKEL_HIP(hipMalloc(&b->d_items, (size_t)b->nitems * sizeof(int)));
        b->items_cap = (size_t)b->nitems;
    }
    for (size_t i = 0; i < ng; ++i) schedule(b->host_tab[i], n, b->asked[i]);
    std::vector<int> order(ng);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(),
                     [&](int x, int y) { return launches_of(b->host_tab[x]) > launches_of(b->host_tab[y]); });
    b->nlaunch = 0;
    for (int g : order) b->nlaunch = std::max(b->nlaunch, launches_of(b->host_tab[g]));
    std::vector<int> items((size_t)b->nitems);
    int fill[BF_COUNT];
    for (int f = 0; f < BF_COUNT; ++f) {
        fill[f] = 0;
        b->launch_items[f].assign((size_t)b->nlaunch, 0);
    }
    for (int g : order) {
        BatchEntry& e = b->host_tab[g];
        const int f = family_of(e);
        e.item0 = fill[f];
        const int ni = e.ntiles;
        for (int t = 0; t < ni; ++t) items[(size_t)(b->fam_first[f] + fill[f]++)] = g;
        for (int l = 0; l < launches_of(e); ++l) b->launch_items[f][l] += ni;
    }
    for (int f = 0; f < BF_COUNT; ++f)
        if (fill[f] != b->fam_items[f]) return fail(PSKEL_ERR_RUNTIME, "batch item count changed");
    PSKEL_HIP(hipMemcpyAsync(b->d_items, items.data(), items.size() * sizeof(int), hipMemcpyHostToDevice, b->stream));
    PSKEL_HIP(hipStreamSynchronize(b->stream));
    b->sched_sweeps = n;
    return PSKEL_OK;
}

// Refresh the per-grid buffer pointers from the grids' current states.
pskel_status_t refresh_table(pskel_batch_t* b)
{
    for (size_t i = 0; i < b->grids.size(); ++i) {
        b->host_tab[i].buf[0] = b->grids[i]->buf[0];
        b->host_tab[i].buf[1] = b->grids[i]->buf[1];
    }
    PSKEL_HIP(hipMemcpyAsync(b->d_tab, b->host_tab.data(), b->host_tab.size() * sizeof(BatchEntry),
                             hipMemcpyHostToDevice, b->stream));
    return PSKEL_OK;
}

// Each family's launches in order on the family's stream, forked from `st`
// and joined back into it (under capture: parallel branches of the graph).
hipError_t issue_batch(pskel_batch_t* b, hipStream_t st)
{
    hipError_t e = hipEventRecord(b->fork, st);
    for (int f = 0; f < BF_COUNT && e == hipSuccess; ++f) {
        if (b->fam_items[f] == 0) continue;
        hipStream_t fs = b->fam_stream[f];
        e = hipStreamWaitEvent(fs, b->fork, 0);
        const int* items = b->d_items + b->fam_first[f];
        for (int l = 0; l < b->nlaunch && e == hipSuccess; ++l) {
            const int n = b->launch_items[f][l];
            if (n == 0) continue;
            const dim3 grid((unsigned)std::min(n, b->fam_blocks[f])), block(kWave, fam_waves(f));
            if (f == BF_REG) hipLaunchKernelGGL(k_batch<BF_REG>, grid, block, 0, fs, b->d_tab, items, n, l);
            else if (f == BF_TTILE) hipLaunchKernelGGL(k_batch<BF_TTILE>, grid, block, 0, fs, b->d_tab, items, n, l);
            else if (f == BF_BITS) hipLaunchKernelGGL(k_batch<BF_BITS>, grid, block, 0, fs, b->d_tab, items, n, l);
            else if (f == BF_J5) hipLaunchKernelGGL(k_batch<BF_J5>, grid, block, 0, fs, b->d_tab, items, n, l);
            else hipLaunchKernelGGL(k_batch<BF_BOX9>, grid, block, 0, fs, b->d_tab, items, n, l);
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipEventRecord(b->join[f], fs);
        if (e == hipSuccess) e = hipStreamWaitEvent(st, b->join[f], 0);
    }
    return e;
}

}  // namespace

extern "C" {

pskel_status_t pskel_batch_create(pskel_grid_t* const* grids, const pskel_stencil_desc_t* descs,
                                  const pskel_launch_cfg_t* cfgs, size_t n, pskel_batch_t** out)
{
    if (!grids || !descs || !out || n == 0 || n > (1u << 20)) return fail(PSKEL_ERR_INVALID_ARGUMENT, "bad batch");
    *out = nullptr;
    for (size_t i = 0; i < n; ++i)
        if (!grids[i]) return fail(PSKEL_ERR_INVALID_ARGUMENT, "batch grid is NULL");
    auto* b = new pskel_batch_t();
    b->device = grids[0]->device;
    for (size_t i = 0; i < n; ++i) {
        pskel_grid_t* g = grids[i];
        auto reject = [&](pskel_status_t st, const char* msg) {
            delete b;
            return fail(st, msg);
        };
        if (g->ndim != 2 || g->device != b->device) return reject(PSKEL_ERR_UNSUPPORTED, "batches hold 2D grids of one device");
        const pskel_stencil_desc_t& d = descs[i];
        const int pat = classify(d, 2);
        BatchEntry e{};
        char either = 0;
        if (pat == PAT_J5 && g->storage == PSKEL_DTYPE_F32) e.kind = BK_J5;
        else if (pat == PAT_BOX9 && g->storage == PSKEL_DTYPE_F32) e.kind = BK_BOX9;
        else if (pat == PAT_LIFE8 && g->storage == PSKEL_DTYPE_U8) e.kind = BK_LIFE;
        else return reject(PSKEL_ERR_UNSUPPORTED, "batched grids run Jacobi 5-point, 3x3 weighted (f32) or life (u8)");
        const int radius = desc_radius(d, 2);
        if (radius < 1) return reject(PSKEL_ERR_INVALID_ARGUMENT, "mask range");
        const int depth = cfgs && cfgs[i].time_tile > 1 ? cfgs[i].time_tile : 1;
        e.depth = depth;
        e.W = (int)g->W;
        e.H = (int)g->H;
        e.pitch = (int)g->pitch;
        e.radius = radius;
        e.coeff = d.coeff;
        for (int k = 0; k < 9; ++k) e.wt[k] = d.weights[k];
        if (depth == 1) {
            const int ry = cfgs && cfgs[i].tile_y > 0 ? cfgs[i].tile_y : 4;
            if (ry != 1 && ry != 2 && ry != 4 && ry != 8)
                return reject(PSKEL_ERR_UNSUPPORTED, "batched rows per lane must be 1, 2, 4 or 8");
            e.ry = ry;
            const int cols = e.kind == BK_LIFE ? 1024 : 256;
            e.tiles_x = (e.W + cols - 1) / cols;
            e.ntiles = e.tiles_x * ((e.H + kBatchWaves * ry - 1) / (kBatchWaves * ry));
        } else if (e.kind == BK_LIFE) {
            // bit-packed tiles, 3, 5 or 7 generations per launch
            if (depth != 3 && depth != 5 && depth != 7)
                return reject(PSKEL_ERR_UNSUPPORTED, "batched life depths are 1, 3, 5 or 7");
            if (radius != 1) return reject(PSKEL_ERR_UNSUPPORTED, "batched life temporal tiles need mask range 1");
            if (lt_fits(g->pitch)) {
                tile_grid(e, depth);
            } else {  // boards of 8M columns: a generation per launch
                e.depth = 1;
                e.ry = 4;
                e.tiles_x = (e.W + 1023) / 1024;
                e.ntiles = e.tiles_x * ((e.H + kBatchWaves * 4 - 1) / (kBatchWaves * 4));
            }
        } else {
            // 3 sweeps per launch: the register tiles; LDS tiles of 120 columns and
            // 16 or 32 rows at a mask range above 1, on grids the register tiles do
            // not take and where they are faster (choose_f32_tiles)
            const bool march = cfgs && cfgs[i].tile_x == kMarch2DVd;
            if (march) {
                if (depth != 3) return reject(PSKEL_ERR_UNSUPPORTED, "the batched register march runs 3 sweeps per launch");
                if (radius != 1 || !march2d_fits(e.W, e.H, g->pitch))
                    return reject(PSKEL_ERR_UNSUPPORTED, "the batched register march needs mask range 1 and a grid over 8 cells wide");
                if (march2d_shape(e.W, e.H, 0).units < 1)
                    return reject(PSKEL_ERR_UNSUPPORTED, "the batched register march needs interior rows");
            }
            if (depth != kTTileK) return reject(PSKEL_ERR_UNSUPPORTED, "batched f32 depths are 1 or 3");
            const int cy = cfgs && cfgs[i].tile_y > 0 && !march ? cfgs[i].tile_y : 16;
            if (cy != 16 && cy != 32) return reject(PSKEL_ERR_UNSUPPORTED, "batched f32 temporal tiles have 16 or 32 rows");
            e.ry = cy;
            if (radius == 1 && rt_fits(e.W, e.H, g->pitch)) {
                e.rtile = 1;
                tile_grid(e, depth);
                either = march ? 2 : 1;
            } else {
                lds_grid(e);
            }
        }
        b->either.push_back(either);
        b->grids.push_back(g);
        b->host_tab.push_back(e);
        b->asked.push_back(depth);
    }
    hipError_t e = hipSetDevice(b->device);
    int cus = 256;
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, b->device);
    const void* fam_kernel[BF_COUNT] = {reinterpret_cast<const void*>(&k_batch<BF_REG>),
                                        reinterpret_cast<const void*>(&k_batch<BF_TTILE>),
                                        reinterpret_cast<const void*>(&k_batch<BF_BITS>),
                                        reinterpret_cast<const void*>(&k_batch<BF_J5>),
                                        reinterpret_cast<const void*>(&k_batch<BF_BOX9>)};
    for (int f = 0; f < BF_COUNT; ++f) {
        int per_cu = 4;
        if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fam_kernel[f], kWave * fam_waves(f), 0);
        b->fam_slots[f] = cus * std::max(1, per_cu);
    }
    count_items(b);
    b->nblocks = std::max(1, std::min(b->nitems, cus * 4));
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreate(&b->ev0);
    if (e == hipSuccess) e = hipEventCreate(&b->ev1);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&b->fork, hipEventDisableTiming);
    for (int f = 0; f < BF_COUNT && e == hipSuccess; ++f) {
        e = hipStreamCreateWithFlags(&b->fam_stream[f], hipStreamNonBlocking);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&b->join[f], hipEventDisableTiming);
    }
    if (e == hipSuccess) e = hipMalloc(&b->d_tab, b->host_tab.size() * sizeof(BatchEntry));
    if (e == hipSuccess) e = hipMalloc(&b->d_items, (size_t)b->nitems * sizeof(int));
    if (e == hipSuccess) b->items_cap = (size_t)b->nitems;
    if (e != hipSuccess) {
        pskel_status_t st = hip_fail(e, "batch setup");
        pskel_batch_destroy(b);
        return st;
    }
    *out = b;
    return PSKEL_OK;
}

pskel_status_t pskel_batch_destroy(pskel_batch_t* b)
{
    if (!b) return PSKEL_OK;
    (void)hipSetDevice(b->device);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->d_tab) (void)hipFree(b->d_tab);
    if (b->d_items) (void)hipFree(b->d_items);
    if (b->ev0) (void)hipEventDestroy(b->ev0);
    if (b->ev1) (void)hipEventDestroy(b->ev1);
    if (b->fork) (void)hipEventDestroy(b->fork);
    for (int f = 0; f < BF_COUNT; ++f) {
        if (b->fam_stream[f]) (void)hipStreamSynchronize(b->fam_stream[f]);
        if (b->fam_stream[f]) (void)hipStreamDestroy(b->fam_stream[f]);
        if (b->join[f]) (void)hipEventDestroy(b->join[f]);
    }
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
    return PSKEL_OK;
}

pskel_status_t pskel_batch_run(pskel_batch_t* b, size_t iterations, int32_t use_graph, pskel_run_stats_t* stats)
{
    if (!b) return fail(PSKEL_ERR_INVALID_ARGUMENT, "batch is NULL");
    if (stats) {
        stats->elapsed_ms = 0.0;
        stats->launches = 0;
        stats->sweeps = (int64_t)iterations;
        stats->residual_count = 0;
    }
    if (iterations == 0) return PSKEL_OK;
    if (iterations > (size_t)0x7fffffff) return fail(PSKEL_ERR_INVALID_ARGUMENT, "too many iterations");
    PSKEL_HIP(hipSetDevice(b->device));
    // the grids' own streams may still be working on their buffers
    for (pskel_grid_t* g : b->grids) PSKEL_HIP(hipStreamSynchronize(g->stream));
    pskel_status_t st;
    if (b->sched_sweeps != iterations) {
        // the captured launches and the schedule go before their item list may
        if (b->exec) (void)hipGraphExecDestroy(b->exec);
        b->exec = nullptr;
        b->sched_sweeps = 0;
        if ((st = plan_batch(b, iterations)) != PSKEL_OK) return st;
    }
    if ((st = refresh_table(b)) != PSKEL_OK) return st;
    if (use_graph && (!b->exec || b->graph_sweeps != iterations)) {
        if (b->exec) (void)hipGraphExecDestroy(b->exec);
        b->exec = nullptr;
        hipStream_t cap;
        PSKEL_HIP(hipStreamCreateWithFlags(&cap, hipStreamNonBlocking));
        hipError_t e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) e = issue_batch(b, cap);
        hipGraph_t graph = nullptr;
        const hipError_t e2 = hipStreamEndCapture(cap, &graph);
        (void)hipStreamDestroy(cap);
        if (e == hipSuccess) e = e2;
        if (e == hipSuccess) e = hipGraphInstantiate(&b->exec, graph, nullptr, nullptr, 0);
        if (graph) (void)hipGraphDestroy(graph);
        if (e != hipSuccess) return hip_fail(e, "batch graph");
        b->graph_sweeps = iterations;
    }
    PSKEL_HIP(hipEventRecord(b->ev0, b->stream));
    if (use_graph) PSKEL_HIP(hipGraphLaunch(b->exec, b->stream));
    else {
        const hipError_t e = issue_batch(b, b->stream);
        if (e != hipSuccess) return hip_fail(e, "batch launch");
    }
    PSKEL_HIP(hipEventRecord(b->ev1, b->stream));
    PSKEL_HIP(hipEventSynchronize(b->ev1));
    float ms = 0.f;
    PSKEL_HIP(hipEventElapsedTime(&ms, b->ev0, b->ev1));
    // every launch of a grid fused an odd number of sweeps: the state moved to
    // the other buffer once per launch
    for (size_t i = 0; i < b->grids.size(); ++i) {
        pskel_grid_t* g = b->grids[i];
        const BatchEntry& e = b->host_tab[i];
        if (launches_of(e) % 2) advance_state(*g, 1, e.radius);
        else g->spare_width = std::min(g->spare_width, e.radius);
        g->sweeps_done += iterations;
    }
    if (stats) {
        stats->elapsed_ms = ms;
        stats->launches = (int64_t)b->nlaunch;
    }
    return PSKEL_OK;
}

pskel_status_t pskel_batch_info(const pskel_batch_t* b, int32_t* nitems, int32_t* nblocks)
{
    if (!b) return fail(PSKEL_ERR_INVALID_ARGUMENT, "batch is NULL");
    if (nitems) *nitems = b->nitems;
    if (nblocks) *nblocks = b->nblocks;
    return PSKEL_OK;
}

}  // extern "C"
