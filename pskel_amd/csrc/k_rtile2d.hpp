// K fused sweeps per launch of a radius-1 2D stencil on tiles held in registers.
//
// A block of NW waves owns a tile of 256 columns (64 lanes x 4 cells) by R*NW
// rows; a wave keeps its R rows in registers and sweeps them in place.  A lane's
// neighbours along w are its own cells and the lanes beside it (DPP); a wave's
// neighbour rows come from the waves above and below through LDS, two rows per
// wave and sweep, one barrier per sweep.  A grid crosses the memory once per K
// sweeps, and a sweep costs its arithmetic and little else: 4 VALU instructions
// per cell for the 5-point sum (the sums take the neighbour lanes' cells as DPP
// operands).
//
// Rows sit in a[1..R] before an odd sweep and in a[0..R-1] before an even one: the
// loop body is two sweeps, so that no row is copied back.
//
// Tiles.  A tile loses one cell per sweep at each edge that is not the grid's;
// neighbouring tiles overlap by 2K rows and 2*hx columns, hx = K rounded up to
// whole lane vectors.  A wave whose rows no later level needs stops sweeping.
//
// The ring.  2D sweeps never write the grid's ring (rows 0 and H-1, columns 0
// and W-1): level l reads, at a ring cell, the ring of the buffer level l lives
// in (even l: src, odd l: ring_other).  Tiles that hold ring cells put those
// values back after every sweep, from LDS.  Cells past the grid hold zeros or stale values that only
// ever reach ring cells.
//
// Every cell evaluates the same expression in the same order as the other 2D
// kernels, with no contraction: a launch equals K single sweeps bit for bit.
//
// Measured, us per sweep, against the kernels that ran before (4 sweeps per
// launch: LDS tiles or the register march; CLOUDSIM: one): 5-point 2048^2 1.6
// (2.9), 4096^2 4.1 (7.1); 9-point 1021 x 1531 2.3 (3.4); CLOUDSIM 4096^2 14.7
// (52; 14.4 without the state before the last sweep), bound by VALU issue (86% of
// its rate, 31 instructions per cell for the formula's 24) and the 16 bytes per
// cell and launch (69% of a copy's rate).
#pragma once

#include <type_traits>

#include "k_common.hpp"

namespace pskel {

constexpr int kRtCols = 256;  // columns of a tile

// columns of halo on each side for K sweeps
__host__ __device__ constexpr int rt_halo_cols(int K) { return (K + 3) / 4 * 4; }

// tiles along an extent n: t cells each, h of them halo on each side
inline int rt_tiles(int n, int t, int h) { return n <= t ? 1 : 1 + (n - t + (t - 2 * h) - 1) / (t - 2 * h); }

// grids whose buffer (and the rows a tile reads past it) a 32-bit buffer offset
// covers, wider than two lane vectors (a lane holds one ring column at most)
inline bool rt_fits(int W, int H, size_t pitch)
{
    return W > 8 && H >= 3 && (uint64_t)H * pitch * 4 < 0x7fffffffull && (uint64_t)(H + 256) * pitch * 4 < 0xffffffffull;
}

// what the stencils read besides the cells
struct RtParams {
    float coeff;         // 5-point: the scale; CLOUDSIM: the time step
    float wt[9];         // 3x3 weights
    const float* wx;     // CLOUDSIM's fields, rows of xpitch and ypitch
    const float* wy;
    uint32_t xpitch, ypitch;
};

// Time of one launch in microseconds: a launch, then rounds of blocks, each
// sweep of a round at the VALU's rate for the rows a CU holds or, with few, at
// the latency of a barrier and one block's rows; no less than its bytes take.
// The constants are a least-squares fit of 820, 640 and 420 measured launches
// (64^2 to 4096^2, depths 1 to 32): the fastest choice or one within 10% on 25
// of 27 grids, 19% at worst.
struct RtCost {
    double launch, round, row, barrier, bytes;  // us, us, us per wave-row, us, bytes per us
};
constexpr RtCost rt_cost(int pattern)
{
    return pattern == PAT_J5     ? RtCost{3.30, 0.19, 0.0096, 0.272, 7.6e6}
           : pattern == PAT_BOX9 ? RtCost{3.34, 0.00, 0.0269, 0.327, 6.2e6}
                                 : RtCost{2.64, 1.39, 0.0316, 0.282, 7.2e6};
}
constexpr int kRtCus = 256;  // what the fit was measured on

// nb blocks of `rows` rows, per_cu of them on a CU at once, writing `cells` cells
inline double rt_launch_time(int pattern, int rows, int per_cu, int64_t nb, double cells, int k)
{
    const RtCost c = rt_cost(pattern);
    const int64_t slots = (int64_t)kRtCus * per_cu, full = nb / slots, rest = nb % slots;
    auto round = [&](int64_t b) {
        return c.round + k * std::max(c.row * (double)(b * rows), c.barrier + c.row * rows);
    };
    const double t = c.launch + (double)full * round(per_cu) + (rest ? round((rest + kRtCus - 1) / kRtCus) : 0.0);
    const double bytes = 4.0 * ((pattern == PAT_CLOUD ? 3.0 : 1.0) * (double)nb * kRtCols * rows + cells);
    return std::max(t, c.launch + bytes / c.bytes);
}

#ifdef PSKEL_RTILE_INSTANTIATE
namespace {

template <int R, int NW>
struct RtLds {
    float4 x[2][NW][2][kWave];  // first and last row of each wave, two levels
    float4 ring[2][2][kWave];   // rows 0 and H-1 of src and ring_other
    float col[2][2][NW * R];    // columns 0 and W-1 of the tile's rows, of src and ring_other
};

__device__ __forceinline__ void rt_load(const __amdgpu_buffer_rsrc_t& r, uint32_t off, float (&v)[4])
{
    const u32x4_t x = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = __uint_as_float(x[j]);
}

// the cell left of a lane's first and right of its last (a halo at the wave's
// ends); zero where there is no lane, so the move folds into the instruction
// that uses it
__device__ __forceinline__ float rt_left(const float (&v)[4])
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v[3]), kDppWaveShr1, 0xf, 0xf, true));
}

__device__ __forceinline__ float rt_right(const float (&v)[4])
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v[0]), kDppWaveShl1, 0xf, 0xf, true));
}

// one CLOUDSIM cell (PSKEL_KIND_CLOUDSIM's formula and order)
__device__ __forceinline__ float rt_cloud(float c, float n, float e, float w, float s, float xw, float yw, float dt)
{
    const float sum = 4.0f * c - (((n + e) + w) + s);
    const bool xp = xw > 0.f, yp = yw > 0.f;
    const float cx = xp ? xw : -xw, cy = yp ? yw : -yw;  // the sign factor times the wind
    const float tx = xp ? e : w, ty = yp ? s : n;
    const float wind = (-cx * ((c - tx) * 10.0f)) - (cy * ((c - ty) * 10.0f));
    const float cond = (-0.0243f * (sum * 0.25f)) * dt;
    return (c + cond) + wind * dt;
}

// one row: u, c, d are the rows above, at and below; uL .. dR the cells beside
// the lane's vector (3x3 box only: u's and d's)
template <int PAT>
__device__ __forceinline__ void rt_row(const RtParams& p, const float (&u)[4], const float (&c)[4], const float (&d)[4],
                                       float uL, float uR, float cL, float cR, float dL, float dR,
                                       const float (&fx)[4], const float (&fy)[4], float (&o)[4])
{
    float q[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float cm = j > 0 ? c[j - 1] : cL, cp = j < 3 ? c[j + 1] : cR;
        float acc;
        if constexpr (PAT == PAT_J5) {
            acc = u[j] + d[j];
            acc = acc + cm;
            acc = acc + cp;
            acc = p.coeff * acc;
        } else if constexpr (PAT == PAT_BOX9) {
            const float um = j > 0 ? u[j - 1] : uL, up = j < 3 ? u[j + 1] : uR;
            const float dm = j > 0 ? d[j - 1] : dL, dp = j < 3 ? d[j + 1] : dR;
            acc = p.wt[0] * um;
            acc = acc + p.wt[1] * u[j];
            acc = acc + p.wt[2] * up;
            acc = acc + p.wt[3] * cm;
            acc = acc + p.wt[4] * c[j];
            acc = acc + p.wt[5] * cp;
            acc = acc + p.wt[6] * dm;
            acc = acc + p.wt[7] * d[j];
            acc = acc + p.wt[8] * dp;
        } else {
            acc = rt_cloud(c[j], u[j], cp, cm, d[j], fx[j], fy[j], p.coeff);
        }
        q[j] = acc;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = q[j];
}

// Tile (tx, ty) of a grid tiled for K sweeps, by the block's NW waves; k sweeps
// run (1 <= k <= K).  Every wave must call it (it synchronises the block).
// With RES returns this lane's sum of squared changes of the last sweep over the
// tile's own cells, ring cells included.  With KEEP the state before the last sweep
// goes to s.prev, if set (in the loop of every kernel the check would cost the 5-point
// 8-row tiles a wave per SIMD).
template <int PAT, int R, int NW, bool RES, bool KEEP>
__device__ __forceinline__ double rt_tile(const Sweep2D& s, const RtParams& p, int tx, int ty, int K, int k, int lane,
                                          int wave, RtLds<R, NW>& L)
{
    constexpr int TH = R * NW;
    constexpr bool CLOUD = PAT == PAT_CLOUD;
    const int H = s.H, W = s.W;
    const int hx = rt_halo_cols(K);
    const int x0 = tx * (kRtCols - 2 * hx), y0 = ty * (TH - 2 * K);
    const int cx0 = tx == 0 ? 0 : x0 + hx, cx1 = x0 + kRtCols >= W ? W : x0 + kRtCols - hx;
    const int cy0 = ty == 0 ? 0 : y0 + K, cy1 = y0 + TH >= H ? H : y0 + TH - K;
    const int wy = y0 + wave * R;     // this wave's first row
    const int xs = x0 + lane * 4;     // this lane's first column
    const uint32_t pb = (uint32_t)s.pitch * 4u;
    const int bytes = (int)((uint32_t)H * pb);
    const __amdgpu_buffer_rsrc_t rs = plane_rsrc(s.src, bytes);
    const __amdgpu_buffer_rsrc_t ro = plane_rsrc(s.ring_other, bytes);
    // rows past H fall out of range
    auto roff = [&](int y) -> uint32_t { return xs < W ? (uint32_t)y * pb + (uint32_t)xs * 4u : kNoAccess; };

    float a[R + 1][4];
#pragma unroll
    for (int i = 0; i < R; ++i) rt_load(rs, roff(wy + i), a[i + 1]);
    float fx[CLOUD ? R : 1][4], fy[CLOUD ? R : 1][4];
    if constexpr (CLOUD) {
        const uint32_t xb = p.xpitch * 4u, yb = p.ypitch * 4u;
        const __amdgpu_buffer_rsrc_t rx = plane_rsrc(p.wx, (int)((uint32_t)H * xb));
        const __amdgpu_buffer_rsrc_t ry = plane_rsrc(p.wy, (int)((uint32_t)H * yb));
#pragma unroll
        for (int i = 0; i < R; ++i) {
            rt_load(rx, xs < W ? (uint32_t)(wy + i) * xb + (uint32_t)xs * 4u : kNoAccess, fx[i]);
            rt_load(ry, xs < W ? (uint32_t)(wy + i) * yb + (uint32_t)xs * 4u : kNoAccess, fy[i]);
        }
    }

    // ring cells of this wave (uniform): rows itop and ibot, and the columns of a
    // tile at the grid's left or right edge
    const int itop = -wy, ibot = H - 1 - wy;  // row 0 and row H-1 as rows of this wave
    const bool has_top = itop >= 0 && itop < R, has_bot = ibot >= 0 && ibot < R;
    const bool edge_c = x0 == 0 || x0 + kRtCols >= W;
    const bool edge = edge_c || has_top || has_bot;
    int ie = -1;  // the ring column among this lane's cells
    const int side = xs == 0 ? 0 : 1;
    if (edge) {
        if (xs == 0) ie = 0;
        else if (xs <= W - 1 && W - 1 < xs + 4) ie = W - 1 - xs;
        // only this wave reads back what it puts here
        if (ie >= 0) {
            float ea[R], eb[R];
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const uint32_t o = (uint32_t)(wy + i) * pb + (uint32_t)(xs + ie) * 4u;
                ea[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)o, 0, 0));
                eb[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ro, (int)o, 0, 0));
            }
#pragma unroll
            for (int i = 0; i < R; ++i) {
                L.col[side][0][wave * R + i] = ea[i];
                L.col[side][1][wave * R + i] = eb[i];
            }
        }
        auto keep = [&](int which, int y) {
            float va[4], vb[4];
            rt_load(rs, roff(y), va);
            rt_load(ro, roff(y), vb);
            L.ring[which][0][lane] = make_float4(va[0], va[1], va[2], va[3]);
            L.ring[which][1][lane] = make_float4(vb[0], vb[1], vb[2], vb[3]);
        };
        if (has_top) keep(0, 0);
        if (has_bot) keep(1, H - 1);
    }

    double rr = 0.0;
    // the level's ring values over row i
    auto patch = [&](int i, bool odd, float (&v)[4]) __attribute__((always_inline)) {
        if (has_top && i == itop) {
            const float4 q = L.ring[0][odd][lane];
            v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
        } else if (has_bot && i == ibot) {
            const float4 q = L.ring[1][odd][lane];
            v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
        } else if (edge_c) {
            const float e = L.col[side][odd][wave * R + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = ie == j ? e : v[j];
        }
    };
    auto put = [&](float4* q, const float (&v)[4]) __attribute__((always_inline)) {
        q[lane] = make_float4(v[0], v[1], v[2], v[3]);
    };
    auto get = [&](const float4* q, float (&v)[4]) __attribute__((always_inline)) {
        const float4 x = q[lane];
        v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
    };
    const int up = wave > 0 ? wave - 1 : 0, dn = wave < NW - 1 ? wave + 1 : NW - 1;
    // rows [cy0 - left, cy1 + left) are needed once `left` sweeps remain
    auto needed = [&](int left) { return wy < cy1 + left && wy + R > cy0 - left && wy < H; };

    // One sweep: rows a[OLD .. OLD+R) -> a[NEW .. NEW+R).  The wave's end rows come
    // last, so that the neighbour waves' rows have left LDS by then.
    // SUM: with RES, the last sweep.
    auto sweep = [&](auto old_t, bool odd, auto sum_t) __attribute__((always_inline)) {
        constexpr bool SUM = decltype(sum_t)::value;
        constexpr int OLD = decltype(old_t)::value, NEW = 1 - OLD;
        float ab[4], be[4];
        get(L.x[NEW][up][1], ab);
        get(L.x[NEW][dn][0], be);
        float c[R][4], n[R][4], left[R + 2], right[R + 2];
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) c[i][j] = a[OLD + i][j];
        auto row = [&](int i, const float (&u)[4], const float (&d)[4]) __attribute__((always_inline)) {
            if constexpr (PAT == PAT_BOX9) {
                rt_row<PAT>(p, u, c[i], d, left[i], right[i], left[i + 1], right[i + 1], left[i + 2], right[i + 2],
                            fx[0], fy[0], n[i]);
            } else {
                rt_row<PAT>(p, u, c[i], d, 0.f, 0.f, rt_left(c[i]), rt_right(c[i]), 0.f, 0.f, fx[CLOUD ? i : 0],
                            fy[CLOUD ? i : 0], n[i]);
            }
            if constexpr (SUM) {
                __builtin_amdgcn_sched_barrier(0);
                if (edge) patch(i, odd, n[i]);
                if (wy + i >= cy0 && wy + i < cy1) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        __builtin_amdgcn_sched_barrier(0);
                        const double dv = (double)n[i][j] - (double)c[i][j];
                        if (xs + j >= cx0 && xs + j < cx1) rr += dv * dv;
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // a row at a time: the scheduler would hold every row's operands
        };
        auto sides = [&](int i, const float (&v)[4]) __attribute__((always_inline)) {
            if constexpr (PAT == PAT_BOX9) {
                left[i + 1] = rt_left(v);
                right[i + 1] = rt_right(v);
            }
        };
        sides(0, c[0]);
        sides(1, c[1]);
#pragma unroll
        for (int i = 1; i < R - 1; ++i) {
            sides(i + 1, c[i + 1]);
            row(i, c[i - 1], c[i + 1]);
        }
        sides(R, be);
        row(R - 1, c[R - 2], be);
        sides(-1, ab);
        row(0, ab, c[1]);
        if (!SUM && edge) {  // no row reads another's new values: the ring goes back once
#pragma unroll
            for (int i = 0; i < R; ++i) patch(i, odd, n[i]);
        }
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) a[NEW + i][j] = n[i][j];
    };

    const __amdgpu_buffer_rsrc_t rd = plane_rsrc(s.dst, bytes);
    const bool own_x = xs >= cx0 && xs < cx1;
    // the tile's own interior rows (with `ring` the ring's too); a lane vector holding a ring column writes
    // the ring value it holds, which is dst's own.  The padding of a row may be
    // the caller's (not CLOUDSIM's, whose buffers are a grid's): the vector that
    // reaches past W stores its cells as a pair and a single.
    auto store = [&](const __amdgpu_buffer_rsrc_t& r, auto off_t, bool ring) __attribute__((always_inline)) {
        // 5-point and 9-point: recomputed from the lane; hoisted above the sweeps,
        // these would hold registers there (5-point 8-row tiles 81 for 72, two waves
        // per SIMD less)
        int x = xs;
        bool own = own_x;
        if constexpr (!CLOUD) {
            int ln = lane;
            asm volatile("" : "+v"(ln));
            x = x0 + ln * 4;
            own = x >= cx0 && x < cx1;
        }
        const bool ragged = !CLOUD && W % 4 != 0 && x0 + kRtCols >= W;  // uniform
        const int part = ragged && own && x + 4 > W ? W - x : 0;  // cells of such a vector
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int y = wy + i;
            if (y < cy0 || y >= cy1 || (!ring && (y < 1 || y > H - 2))) continue;  // uniform
            const uint32_t o = (uint32_t)y * pb + (uint32_t)x * 4u;
            u32x4_t v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = __float_as_uint(a[i + decltype(off_t)::value][j]);
            __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)(own && !part ? o : kNoAccess), 0, 0);
            if (!ragged) continue;
            const u32x2_t two = {v[0], v[1]};
            __builtin_amdgcn_raw_buffer_store_b64(two, r, (int)(part & 2 ? o : kNoAccess), 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(part & 2 ? v[2] : v[0], r,
                                                  (int)(part & 1 ? o + (part & 2) * 4u : kNoAccess), 0, 0);
        }
    };

    // Level l's rows to the neighbour waves, and a barrier.  False: no later
    // level needs this wave's rows (nor any level after that one), so it only
    // keeps up with the block's barriers, one per sweep, and is done.
    auto exchange = [&](int l, float4 (*x)[2][kWave], const float (&first)[4], const float (&last)[4])
                        __attribute__((always_inline)) -> bool {
        put(x[wave][0], first);
        put(x[wave][1], last);
        if (needed(k - 1 - l)) {
            __syncthreads();
            return true;
        }
#pragma unroll 1
        for (; l < k; ++l) __syncthreads();
        return false;
    };
    constexpr std::integral_constant<int, 0> at0;
    constexpr std::integral_constant<int, 1> at1;
    auto finish = [&](auto off_t) __attribute__((always_inline)) {
        store(rd, off_t, false);
        return rr;
    };
    // before the last sweep: of an even number to the buffer that holds its ring, of an
    // odd one (at least 3) to one that does not
    auto keep_prev = [&](auto off_t) __attribute__((always_inline)) {
        if (!KEEP || !s.prev) return;  // uniform
        store(plane_rsrc(s.prev, bytes), off_t, decltype(off_t)::value == 1);
    };
    int l = 0;
    // with RES the last sweep is another copy of the code: its sums, and the
    // registers they take, stay out of the other sweeps
#pragma unroll 1
    for (;;) {
        if (!exchange(l, L.x[0], a[1], a[R])) return rr;
        if (RES && l + 1 == k) {
            keep_prev(at1);
            sweep(at1, true, std::bool_constant<RES>());
            return finish(at0);
        }
        if (KEEP && l + 1 == k) keep_prev(at1);
        sweep(at1, true, std::false_type());
        if (++l == k) return finish(at0);
        if (!exchange(l, L.x[1], a[0], a[R - 1])) return rr;
        if (RES && l + 1 == k) {
            keep_prev(at0);
            sweep(at0, false, std::bool_constant<RES>());
            return finish(at1);
        }
        if (KEEP && l + 1 == k) keep_prev(at0);
        sweep(at0, false, std::false_type());
        if (++l == k) return finish(at1);
    }
}

// 64 registers (8 waves per SIMD, two blocks of 16 waves per CU) hold 4 rows
template <int PAT, int R, int NW, bool RES, bool KEEP>
__global__ __launch_bounds__(NW * kWave, PAT != PAT_CLOUD && R <= 4 ? 8 : 1) void k2d_rtile(Sweep2D s, RtParams p, int ntx, int K, double* partials)
{
    __shared__ RtLds<R, NW> L;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int t = (int)xcd_remap(blockIdx.x, gridDim.x);
    const double rr = rt_tile<PAT, R, NW, RES, KEEP>(s, p, t % ntx, t / ntx, K, K, lane, wave, L);
    if constexpr (RES) {
        __shared__ double red[NW];
        const double v = block_sum<NW>(rr, red);
        if (threadIdx.x == 0) partials[t] = v;
    }
}

}  // namespace
#endif  // PSKEL_RTILE_INSTANTIATE

}  // namespace pskel
