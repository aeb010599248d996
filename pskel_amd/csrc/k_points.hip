// Arbitrary masks (any points, weights and order) in 2D and 3D: the tuned
// variant's kernel for stencils without a specialised one.
//
// Reference contract: stencilTilingCU (include/PSkelStencil.hpp:572-652,
// 685-701) runs the user kernel, which sums Mask::get values in mask order
// (include/PSkelMask.hpp:186-199, 292-305).  Sums here are in mask order, no
// contraction, so results equal the plain kernels' bit for bit.
//
// A block of 512 lanes stages a tile of cells and its halo in LDS as f32 (16-bit
// storage decoded once, cells outside the grid as the halo value), then every
// lane updates 8 cells stacked along w (h in 2D): a point costs one address add
// and eight LDS reads at constant offsets, whatever its place in the mask, and
// 16 products and sums.  The mask travels as LDS offsets, computed on the host,
// in scalar registers.
//
// What bounds it: per cell and point 4 bytes of LDS (128 B per clock and CU) and
// two VALU lane-operations (64 per clock and CU), 0.03 clocks each, after a
// fixed part of staging and storing (a 7-point star takes 22 us where 27 points
// take 32); at 27 points VALU issue runs at 77% of its rate, 88 instructions per
// cell for 53 (staging, idle lanes), with no bank conflicts.  The plain kernel waits for each point's global load in turn (a
// uniform branch per point keeps the loads from overlapping).  Measured, f32,
// 3x3x3 weighted box with HALO faces: 192 x 225 x 260 32 us per sweep (3.5e11
// cell-updates/s; plain 259 us), 256^3 40 us (400 us), 60 x 70 x 50 6.5 us (14 us).
#include <cmath>

#include "k_common.hpp"

namespace pskel {

namespace {

constexpr int kPtThreads = 512;
constexpr int kPtWaves = kPtThreads / kWave;
constexpr int kPtCells = 8;        // cells per lane, along w (2D: h)
constexpr int kPtChunk = 4;        // points whose offsets and weights load at once
constexpr size_t kPtLdsMax = 64 * 1024;

// The mask and the tile as the kernel sees them.  3D: axes (a, b, x) = (h, w,
// d); 2D: (-, h, w).  Lanes run along x.
struct PointsTile {
    int np, radius, boundary;
    float coeff, halo, off, c0;
    int A, B, X;               // grid extents
    int alo, blo;              // halo planes and rows before the tile
    int LA, LB;                // planes and rows staged
    uint32_t magic;            // ceil(2^20 / LB): row index -> plane, by a multiply
    int nta, ntb, ntx;         // tiles along a, b and x
    int rounding;
    uint32_t seed, plane0;
    uint64_t sweep;
    size_t pitch;
    const void* src;
    void* dst;
    double* partials;
    int loff[kMaxPoints];      // LDS offset of each point, in floats
    float wt[kMaxPoints];
};

// halo granules of four cells on each side of the tile along x
template <int TX, int HG>
constexpr int pt_stride()
{
    return TX + 8 * HG;
}

// TX: cells of the tile along x (lanes); a wave covers 64 / TX planes (2D: row
// groups).  HG: halo granules of 4 cells along x on each side.
template <int ST, int KIND, bool IS2D, int TX, int HG>
__global__ __launch_bounds__(kPtThreads) void k_points(PointsTile t)
{
    using Tr = Stor<ST>;
    using T = typename Tr::T;
    constexpr int LS = pt_stride<TX, HG>();
    constexpr int SUB = kWave / TX;
    // 16-bit scaled sums add the stored values (u - off) and fold the offset
    // into one fused multiply-add (scaled_sum_offset_term), as the plain kernel
    constexpr bool DEV = ST != PSKEL_DTYPE_F32 && KIND == PSKEL_KIND_SCALED_SUM;
    extern __shared__ __align__(16) float tile[];
    __shared__ double red[kPtWaves];

    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
    const int tx = (int)(id % t.ntx), tb = (int)(id / t.ntx % t.ntb), ta = (int)(id / t.ntx / t.ntb);
    const int x0 = tx * TX;
    const int a0 = IS2D ? 0 : ta * kPtWaves * SUB;
    const int b0 = tb * (IS2D ? kPtWaves * SUB * kPtCells : kPtCells);
    const T* __restrict__ src = (const T*)t.src;

    // stage: a wave takes whole rows, G granules of four cells each, 64 / G rows
    // at a time
    {
        constexpr int G = LS / 4, RPS = kWave / G;
        const int sub = lane / G, g = lane % G;
        const int rows = t.LA * t.LB;
        const int xg = x0 + 4 * (g - HG);
        const int xc = xg < 0 ? 0 : (xg < t.X ? xg : (t.X - 1) & ~3);
        const bool xin = xg >= 0 && xg < t.X;
        constexpr int NB = 4;  // rows in flight per lane
        if (sub < RPS) {
#pragma unroll 1
            for (int r0 = wave * RPS + sub; r0 < rows; r0 += NB * kPtWaves * RPS) {
                T q[NB][4];
                bool in[NB];
                // every lane loads, from the nearest cell of the grid
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const int r = min(r0 + k * kPtWaves * RPS, rows - 1);
                    const int z = IS2D ? 0 : (int)(((uint32_t)r * t.magic) >> 20);
                    const int a = a0 + z - t.alo, b = b0 + r - z * t.LB - t.blo;
                    const int ac = min(max(a, 0), t.A - 1), bc = min(max(b, 0), t.B - 1);
                    in[k] = xin && a == ac && b == bc;
                    load_vec<T, 4>(src + ((size_t)ac * t.B + bc) * t.pitch + xc, q[k]);
                }
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const int r = r0 + k * kPtWaves * RPS;
                    if (r >= rows) break;
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float u = DEV ? Tr::dec_raw(q[k][j]) : Tr::dec(q[k][j], t.off);
                        v[j] = in[k] && xg + j < t.X ? u : t.halo;
                    }
                    *reinterpret_cast<float4*>(&tile[r * LS + 4 * g]) = make_float4(v[0], v[1], v[2], v[3]);
                }
            }
        }
    }
    __syncthreads();

    const int xl = lane % TX, grp = wave * SUB + lane / TX;
    const int al = IS2D ? 0 : grp, bl = IS2D ? grp * kPtCells : 0;
    const float* base = tile + ((al + t.alo) * t.LB + bl + t.blo) * LS + xl + 4 * HG;
    float acc[kPtCells];
    {
        const float* q = base + t.loff[0];
        const float w0 = t.wt[0];
#pragma unroll
        for (int c = 0; c < kPtCells; ++c) {
            const float v = q[c * LS];
            acc[c] = KIND == PSKEL_KIND_SCALED_SUM ? v : w0 * v;
        }
    }
    auto point = [&](int lo, float wv) __attribute__((always_inline)) {
        const float* q = base + lo;
#pragma unroll
        for (int c = 0; c < kPtCells; ++c) {
            const float v = q[c * LS];
            if constexpr (KIND == PSKEL_KIND_SCALED_SUM) acc[c] = acc[c] + v;
            else acc[c] = acc[c] + wv * v;
        }
    };
    int i = 1;
#pragma unroll 1
    for (; i + kPtChunk <= t.np; i += kPtChunk) {
#pragma unroll
        for (int k = 0; k < kPtChunk; ++k) point(t.loff[i + k], t.wt[i + k]);
    }
#pragma unroll 1
    for (; i < t.np; ++i) point(t.loff[i], t.wt[i]);

    const int x = x0 + xl, a = a0 + al, r = t.radius;
    double rr = 0.0;
    auto finish = [&](float u) __attribute__((always_inline)) -> float {
        if constexpr (DEV) return __builtin_fmaf(t.coeff, u, t.c0);
        else if constexpr (KIND == PSKEL_KIND_SCALED_SUM) return t.coeff * u;
        else return u;
    };
    // a block of f32 cells that all take the sum (uniform): plain stores
    const int bend = b0 + (IS2D ? kPtWaves * SUB : 1) * kPtCells;
    const bool whole = ST == PSKEL_DTYPE_F32 && !t.partials && bend <= t.B &&
                       (IS2D ? b0 >= r && bend <= t.B - r && x0 >= r && x0 + TX <= t.X - r
                             : t.boundary != PSKEL_BOUNDARY_COPY ||
                                   (b0 >= r && bend <= t.B - r && x0 >= r && x0 + TX <= t.X - r && a0 >= r &&
                                    a0 + kPtWaves * SUB <= t.A - r));
    if (whole) {
        if (x < t.X && a < t.A) {
            float* o = (float*)t.dst + ((size_t)a * t.B + b0 + bl) * t.pitch + x;
#pragma unroll
            for (int c = 0; c < kPtCells; ++c) o[c * t.pitch] = finish(acc[c]);
        }
        return;
    }
    if (x < t.X && a < t.A) {
        uint32_t ckey = 0, rb = 0;
        if (ST != PSKEL_DTYPE_F32 && t.rounding == PSKEL_ROUND_STOCHASTIC) {
            ckey = sr_cell_key(t.seed);
            rb = sr_plane_bits(sweep_key(t.seed, t.sweep), t.plane0 + a);
        }
#pragma unroll
        for (int c = 0; c < kPtCells; ++c) {
            const int b = b0 + bl + c;
            if (b >= t.B) break;
            const bool edge = x < r || x >= t.X - r || b < r || b >= t.B - r ||
                              (!IS2D && (a < r || a >= t.A - r));
            if (IS2D && edge) continue;  // 2D sweeps never write the ring
            const size_t idx = ((size_t)a * t.B + b) * t.pitch + x;
            T res;
            if (!IS2D && edge && t.boundary == PSKEL_BOUNDARY_COPY) {
                res = src[idx];
            } else {
                const float u = finish(acc[c]);
                if (ST != PSKEL_DTYPE_F32 && t.rounding == PSKEL_ROUND_STOCHASTIC) {
                    const uint32_t rw = sr_cell_bits(ckey, (uint32_t)b * t.X + x) ^ rb;
                    res = DEV ? Tr::enc_sr_raw(u, rw) : Tr::enc_sr(u, t.off, rw);
                } else {
                    res = DEV ? Tr::enc_raw(u) : Tr::enc(u, t.off);
                }
            }
            ((T*)t.dst)[idx] = res;
            if (t.partials) {
                const double dv = (double)Tr::dec_raw(res) - (double)Tr::dec_raw(src[idx]);
                rr += dv * dv;
            }
        }
    }
    if (t.partials) {
        const double s = block_sum<kPtWaves>(rr, red);
        if (threadIdx.x == 0) t.partials[id] = s;
    }
}

// The tile for a mask on a grid: the lanes' width along x that leaves the
// fewest idle lanes and rows.  false: its halo does not fit (the plain kernels
// run): more than 8 cells along x, or a tile over 64 KB.
struct PtPlan {
    PointsTile t;
    int tx = 0, hg = 0;
    size_t lds = 0, blocks = 0;
};

bool pt_plan(const Points& p, bool is2d, int A, int B, int X, PtPlan* best)
{
    int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
    for (int i = 0; i < p.np; ++i) {
        const int o[3] = {is2d ? 0 : p.dh[i], is2d ? p.dh[i] : p.dw[i], is2d ? p.dw[i] : p.dd[i]};
        for (int k = 0; k < 3; ++k) {
            lo[k] = std::max(lo[k], -o[k]);
            hi[k] = std::max(hi[k], o[k]);
        }
    }
    const int rx = std::max(lo[2], hi[2]);
    if (rx > 8) return false;
    const int hg = rx <= 4 ? 1 : 2;
    double best_cost = 0.0;
    for (int tx : {64, 32, 16}) {
        const int sub = kWave / tx, grps = kPtWaves * sub;
        const int ta = is2d ? 1 : grps, tb = is2d ? grps * kPtCells : kPtCells;
        const int LA = ta + lo[0] + hi[0], LB = tb + lo[1] + hi[1], LS = tx + 8 * hg;
        const size_t lds = (size_t)LA * LB * LS * sizeof(float);
        // rows are split into planes by a multiply, exact below 2^20 / LB rows
        if (lds > kPtLdsMax || (size_t)LA * LB * LB >= (1u << 20)) continue;
        const int64_t na = (A + ta - 1) / ta, nb = (B + tb - 1) / tb, nx = (X + tx - 1) / tx;
        // lane-points that run and cells staged (weighted by what each measured:
        // box27, 13- and 7-point stars at 192 x 225 x 260 and 256^3 pick the
        // fastest width or one within 4%), over the blocks a CU's LDS holds (4
        // at most: 32 waves)
        const double cost = (double)(na * nb * nx) * (1.0 * ta * tb * tx * (p.np + 4) + 6.0 * LA * LB * LS) /
                            (double)std::min<size_t>(4, (160 * 1024) / lds);
        if (na * nb * nx > 0x7fffffff || (best->tx && cost >= best_cost)) continue;
        best_cost = cost;
        best->tx = tx;
        best->hg = hg;
        best->lds = lds;
        best->blocks = (size_t)(na * nb * nx);
        PointsTile& t = best->t;
        t.np = p.np;
        t.radius = p.radius;
        t.boundary = p.boundary;
        t.coeff = p.coeff;
        t.A = A;
        t.B = B;
        t.X = X;
        t.alo = lo[0];
        t.blo = lo[1];
        t.LA = LA;
        t.LB = LB;
        t.magic = ((1u << 20) + LB - 1) / LB;
        t.nta = (int)na;
        t.ntb = (int)nb;
        t.ntx = (int)nx;
        for (int i = 0; i < p.np; ++i) {
            const int a = is2d ? 0 : p.dh[i], b = is2d ? p.dh[i] : p.dw[i], x = is2d ? p.dw[i] : p.dd[i];
            t.loff[i] = (a * LB + b) * LS + x;
            t.wt[i] = p.wt[i];
        }
    }
    return best->tx != 0;
}

template <int ST, int KIND, bool IS2D>
hipError_t pt_launch(const PtPlan& q, hipStream_t st)
{
    const dim3 grid((unsigned)q.blocks), block(kPtThreads);
#define PSKEL_PT(TX, HG) \
    if (q.tx == TX && q.hg == HG) hipLaunchKernelGGL((k_points<ST, KIND, IS2D, TX, HG>), grid, block, q.lds, st, q.t)
    PSKEL_PT(64, 1);
    PSKEL_PT(64, 2);
    PSKEL_PT(32, 1);
    PSKEL_PT(32, 2);
    PSKEL_PT(16, 1);
    PSKEL_PT(16, 2);
#undef PSKEL_PT
    return hipGetLastError();
}

template <int ST>
hipError_t pt_launch3d(const PtPlan& q, int kind, hipStream_t st)
{
    if (kind == PSKEL_KIND_SCALED_SUM) return pt_launch<ST, PSKEL_KIND_SCALED_SUM, false>(q, st);
    return pt_launch<ST, PSKEL_KIND_WEIGHTED_SUM, false>(q, st);
}

bool pt_kind(const Points& p)
{
    return p.kind == PSKEL_KIND_SCALED_SUM || p.kind == PSKEL_KIND_WEIGHTED_SUM;
}

}  // namespace

// The time of a sweep through the tile against the plain kernel's, whose block is bx
// lanes along x by `by` along b.  Both are a launch and the larger of one block's (or
// wave's) latency and the work: tiles stage and sum all their cells, those outside
// the grid too; the plain kernel sums only the cells that take one (a copied face or
// a ring costs it next to nothing), but lanes past a row's end cost it waves, and
// points of HALO faces are checked one by one.  Microseconds, fitted to 1035 pairs
// (31 3D grids from 40^3 to 256^3 and thin in each axis, 13 2D grids, 1 to 64
// points, COPY and HALO, f32 and bf16): 1% behind the faster of the two on average,
// where the tile throughout was 25% behind and up to 11 times slower (1 x 1500 x 1000
// 27 points COPY, plain 4.3, tile 26; 5 x 200000 49 points 3.6 and 41).
bool points_pay(const Points& p, bool is2d, int A, int B, int X, bool half, int bx, int by)
{
    PtPlan q;
    if (!pt_kind(p) || !pt_plan(p, is2d, A, B, X, &q)) return false;
    const bool halo = !is2d && p.boundary == PSKEL_BOUNDARY_HALO;
    auto inner = [&](int n) { return (double)std::max(0, n - 2 * p.radius); };
    const double cells = (double)A * B * X, sums = (is2d ? 1.0 : inner(A)) * inner(B) * inner(X), np = p.np;
    // copies only (rows of a few cells: the plain kernel's waves are nearly empty)
    if (!halo && sums == 0 && (X >= 16 || p.np > 27)) return false;
    const double waves = (double)((X + bx - 1) / bx) * ((B + by - 1) / by) * A * bx * by / kWave;
    const double ms = sums / 1e6, mf = (cells - sums) / 1e6, mw = waves / 1e4;
    const double plain = halo ? 0.85 + std::max(2.35 * mw + (1.0 * ms + 0.527 * mf) * np, 2.05 + 0.356 * np)
                              : 1.81 + std::max(1.24 * mw + ms * (0.184 + 0.635 * np), 1.01 + 0.186 * np);
    const double stage = (double)q.lds / sizeof(float) / 1e3;  // thousands of cells
    const double per_cu = (double)((q.blocks + 255) / 256), at_once = (double)std::min<size_t>(4, (160 * 1024) / q.lds);
    const double rounds = std::ceil(per_cu / at_once);
    const double tile = halo ? 3.08 + std::max((0.0589 * np + 0.311 * stage) * rounds,
                                               per_cu * (0.05 * np + 0.1525 * stage + (half ? 0.544 : 0.0)))
                             : 4.04 + std::max((0.0715 * np + 0.227 * stage) * rounds,
                                               per_cu * (0.0471 * np + 0.199 * stage + (half ? 0.047 : 0.0)));
    // grids a cell or two thick (but along x) lie farthest from the fit
    const bool thin = X >= 16 && cells < 0.25 * kPtCells * kPtThreads * (double)q.blocks;
    return tile < (thin ? 0.75 : 0.95) * plain;
}

size_t points3d_blocks(const Sweep3D& s, const Points& p)
{
    PtPlan q;
    return pt_kind(p) && pt_plan(p, false, s.H, s.W, s.D, &q) ? q.blocks : 0;
}

hipError_t launch_3d_points(const Sweep3D& s, const Points& p, int storage, hipStream_t st)
{
    PtPlan q;
    if (!pt_kind(p) || !pt_plan(p, false, s.H, s.W, s.D, &q)) return hipErrorInvalidValue;
    PointsTile& t = q.t;
    const bool dev = storage != PSKEL_DTYPE_F32 && p.kind == PSKEL_KIND_SCALED_SUM;
    t.halo = dev ? p.halo - s.store_offset : p.halo;
    t.off = s.store_offset;
    t.c0 = s.c0;
    t.rounding = s.rounding;
    t.seed = s.seed;
    t.plane0 = s.plane0;
    t.sweep = s.sweep;
    t.pitch = s.pitch;
    t.src = s.src;
    t.dst = s.dst;
    t.partials = s.partials;
    switch (storage) {
    case PSKEL_DTYPE_F32: return pt_launch3d<PSKEL_DTYPE_F32>(q, p.kind, st);
    case PSKEL_DTYPE_BF16: return pt_launch3d<PSKEL_DTYPE_BF16>(q, p.kind, st);
    case PSKEL_DTYPE_F16: return pt_launch3d<PSKEL_DTYPE_F16>(q, p.kind, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_2d_points_f32(const Sweep2D& s, const Points& p, hipStream_t st)
{
    PtPlan q;
    if (!pt_kind(p) || !pt_plan(p, true, 1, s.H, s.W, &q)) return hipErrorInvalidValue;
    PointsTile& t = q.t;
    t.halo = 0.0f;  // only ring cells reach outside, and they are not written
    t.off = t.c0 = 0.0f;
    t.rounding = PSKEL_ROUND_NEAREST;
    t.seed = t.plane0 = 0;
    t.sweep = 0;
    t.pitch = s.pitch;
    t.src = s.src;
    t.dst = s.dst;
    t.partials = nullptr;
    if (p.kind == PSKEL_KIND_SCALED_SUM) return pt_launch<PSKEL_DTYPE_F32, PSKEL_KIND_SCALED_SUM, true>(q, st);
    return pt_launch<PSKEL_DTYPE_F32, PSKEL_KIND_WEIGHTED_SUM, true>(q, st);
}

}  // namespace pskel
