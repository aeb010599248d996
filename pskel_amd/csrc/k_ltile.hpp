// Several generations of B3/S23 per launch on bit-packed tiles held in registers.
//
// A block of NW waves owns a tile of 64 lanes x 32 columns by R*NW rows: a lane
// keeps its 32 columns of each row as one word (bit b = column x + b), packed
// from the u8 cells on load and unpacked on store, so a board crosses the
// memory as bytes once per launch and lives in registers for all its
// generations.  A generation of a row takes
//   * the words shifted by a column each way, with a bit from the lane beside
//     (two DPP moves, two v_alignbit),
//   * the horizontal sums H = left + centre + right and M = left + right as two
//     bit planes each, once per row,
//   * the count H(y-1) + H(y+1) + M(y) by full adders; alive' = (count is 3) or
//     (count is 2 and alive): 14 instructions per 32 cells.
// A wave's neighbour rows come from the waves above and below through LDS, one
// word per lane, with one barrier per generation.
//
// Tiles lose a cell per generation at each edge that is not the grid's: they
// overlap by 2K rows and two lanes (32 columns each, K < 32).  A wave whose
// rows no later generation needs stops.
//
// The ring (rows 0 and H-1, columns 0 and W-1) is never computed: after each
// generation a ring cell takes the ring of the buffer its level maps to (odd
// levels: ring_other's, even: src's), from LDS, in the tiles that hold ring
// cells.  Cells past the grid only ever reach ring cells.
//
// Measured, us per generation, against the bit tiles that ran before (a wave per
// tile, at most 8 generations per launch): 8194^2 2.8 (9.7), 4096^2 1.6; 1000 x
// 1503 0.83 (3.6, one generation per launch).  The floor of an 8194^2 board is
// 0.75 us of VALU; the rest is the halo (5 tiles of 1984 columns hold 4.1, 96 to
// 104 of 128 rows are a tile's own) and the bytes of load and store.
#pragma once

#include "k_common.hpp"

namespace pskel {

constexpr int kLtCols = 64 * 32;  // columns of a tile
constexpr int kLtMaxDepth = 31;   // a lane's halo

// tiles along an extent n: t cells each, h of them halo on each side
inline int lt_tiles(int n, int t, int h) { return n <= t ? 1 : 1 + (n - t + (t - 2 * h) - 1) / (t - 2 * h); }

// boards whose tiles (up to 256 rows) a 32-bit buffer offset covers
inline bool lt_fits(size_t pitch) { return pitch * 256 < 0x7fffffffull; }

// Time of one launch in microseconds: a launch, then rounds of blocks, each
// packing and unpacking its rows and running its generations at the VALU's rate
// for the rows a CU holds or, with few, at the latency of a barrier and one
// block's rows; no less than its bytes take.  Fitted to 472 measured launches
// (64^2 to 8194^2, 1 to 30 generations): the fastest choice on all 8 boards.
// nb blocks of `rows` rows, per_cu of them on a CU at once, writing `cells` cells.
inline double lt_launch_time(int rows, int per_cu, int64_t nb, double cells, int k)
{
    constexpr double launch = 2.54, pack = 0.0442, row = 0.0093, barrier = 0.342, rate = 6.6e6;
    constexpr int cus = 256;  // what the fit was measured on
    const int64_t slots = (int64_t)cus * per_cu, full = nb / slots, rest = nb % slots;
    auto round = [&](int64_t b) {
        return pack * (double)(b * rows) + k * std::max(row * (double)(b * rows), barrier + row * rows);
    };
    const double t = launch + (double)full * round(per_cu) + (rest ? round((rest + cus - 1) / cus) : 0.0);
    return std::max(t, launch + ((double)nb * kLtCols * rows + cells) / rate);
}

#ifdef PSKEL_LTILE_INSTANTIATE
namespace {

template <int R, int NW>
struct LtLds {
    uint32_t x[2][NW][2][kWave];    // first and last row of each wave, two generations
    uint32_t ring[2][2][kWave];     // rows 0 and H-1 of src and ring_other
    uint32_t col[2][2][NW * R];     // the ring columns' bits in their lanes' words, of src and ring_other
};

// 32 cells (bytes 0 or 1) as bits: a byte dot product places four cells at a time
__device__ __forceinline__ uint32_t lt_pack(const u32x4_t& a, const u32x4_t& b)
{
    constexpr uint32_t lo = 0x08040201u, hi = 0x80402010u;
    auto eight = [](uint32_t x, uint32_t y) {
        return __builtin_amdgcn_udot4(y, hi, __builtin_amdgcn_udot4(x, lo, 0u, false), false);
    };
    return eight(a[0], a[1]) | eight(a[2], a[3]) << 8 | eight(b[0], b[1]) << 16 | eight(b[2], b[3]) << 24;
}

// bits 4q .. 4q+3 as bytes: bit i of the nibble lands on bit 8i of its product
// with 0x204081, with no carries (a 24-bit multiply, full rate)
__device__ __forceinline__ uint32_t lt_unpack(uint32_t w, int q)
{
    return __umul24((w >> (4 * q)) & 0xFu, 0x00204081u) & 0x01010101u;
}

// three-input boolean operations, one instruction each (v_bitop3_b32; the table
// byte is the function of a = 0xF0, b = 0xCC, c = 0xAA).  Written out because
// the optimiser rewrites the plain expressions into half as many more.
__device__ __forceinline__ uint32_t lt_xor3(uint32_t a, uint32_t b, uint32_t c)
{
    return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)c, 0x96);
}
__device__ __forceinline__ uint32_t lt_maj(uint32_t a, uint32_t b, uint32_t c)
{
    return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)c, 0xE8);
}
__device__ __forceinline__ uint32_t lt_xor_andn(uint32_t a, uint32_t b, uint32_t c)  // (a ^ b) & ~c
{
    return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)c, 0x14);
}
__device__ __forceinline__ uint32_t lt_and_or(uint32_t a, uint32_t b, uint32_t c)  // a & (b | c)
{
    return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)c, 0xE0);
}

// horizontal sums of a row's word: h = left + centre + right, m = left + right
__device__ __forceinline__ void lt_sums(uint32_t x, uint32_t& h0, uint32_t& h1, uint32_t& m0, uint32_t& m1)
{
    const uint32_t up = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppWaveShr1, 0xf, 0xf, true);
    const uint32_t dn = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppWaveShl1, 0xf, 0xf, true);
    const uint32_t l = __builtin_amdgcn_alignbit(x, up, 31), r = __builtin_amdgcn_alignbit(dn, x, 1);
    h0 = lt_xor3(l, x, r);
    h1 = lt_maj(l, x, r);
    m0 = l ^ r;
    m1 = l & r;
}

// Tile (tx, ty) of a board tiled for K generations, by the block's NW waves; k
// run (1 <= k <= K).  Every wave must call it (it synchronises the block).  With KEEP
// the state before the last generation goes to s.prev, if set.
template <int R, int NW, bool KEEP>
__device__ __forceinline__ void life_tile(const Sweep2D& s, int tx, int ty, int K, int k, int lane, int wave,
                                          LtLds<R, NW>& L)
{
    constexpr int TH = R * NW;
    const int H = s.H, W = s.W;
    const int x0 = tx * (kLtCols - 64), y0 = ty * (TH - 2 * K);
    const int cx0 = tx == 0 ? 0 : x0 + 32, cx1 = x0 + kLtCols >= W ? W : x0 + kLtCols - 32;
    const int cy0 = ty == 0 ? 0 : y0 + K, cy1 = y0 + TH >= H ? H : y0 + TH - K;
    const int wy = y0 + wave * R;
    const int xs = x0 + lane * 32;  // rows are padded to whole 1 KiB: a lane's 32 bytes stay inside
    const size_t pitch = s.pitch;
    const uint32_t p = (uint32_t)pitch;
    // resources from the tile's first row; rows past the grid fall out of range
    const int rows = min(H - y0, TH);
    const int bytes = (int)((uint32_t)rows * p);
    const uint8_t* oth = (const uint8_t*)s.ring_other + (size_t)y0 * pitch;
    const __amdgpu_buffer_rsrc_t rs = plane_rsrc((const uint8_t*)s.src + (size_t)y0 * pitch, bytes);
    const __amdgpu_buffer_rsrc_t ro = plane_rsrc(oth, bytes);
    auto off = [&](int i) -> uint32_t {  // row i of this wave
        return xs < W ? (uint32_t)(wave * R + i) * p + (uint32_t)xs : kNoAccess;
    };

    uint32_t c[R];
    constexpr int BR = R < 4 ? R : 4;  // rows in flight
#pragma unroll
    for (int b = 0; b < R; b += BR) {
        u32x4_t v[BR][2];
#pragma unroll
        for (int i = 0; i < BR; ++i) {
            v[i][0] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off(b + i), 0, 0);
            v[i][1] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off(b + i) + 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < BR; ++i) c[b + i] = lt_pack(v[i][0], v[i][1]);
    }

    // ring cells of this wave (uniform) and the ring columns in this lane's words
    const int itop = -wy, ibot = H - 1 - wy;
    const bool has_top = itop >= 0 && itop < R, has_bot = ibot >= 0 && ibot < R;
    const bool edge_c = x0 == 0 || x0 + kLtCols >= W;
    const bool edge = edge_c || has_top || has_bot;
    const int bw = W - 1 - xs;
    const uint32_t cm = (xs == 0 ? 1u : 0u) | (bw >= 0 && bw < 32 ? 1u << bw : 0u);
    const int side = xs == 0 ? 0 : 1;
    if (edge) {
        // only this wave reads back what it puts here
        auto keep = [&](int which, int i, uint32_t w) {
            const u32x4_t a = __builtin_amdgcn_raw_buffer_load_b128(ro, (int)off(i), 0, 0);
            const u32x4_t b = __builtin_amdgcn_raw_buffer_load_b128(ro, (int)off(i) + 16, 0, 0);
            L.ring[which][0][lane] = w;
            L.ring[which][1][lane] = lt_pack(a, b);
        };
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if (has_top && i == itop) keep(0, i, c[i]);
            if (has_bot && i == ibot) keep(1, i, c[i]);
        }
        if (cm) {
            uint32_t a[R], b[R];
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const uint32_t o = (uint32_t)(wave * R + i) * p;
                a[i] = __builtin_amdgcn_raw_buffer_load_b8(ro, (int)(xs == 0 ? o : kNoAccess), 0, 0);
                b[i] = __builtin_amdgcn_raw_buffer_load_b8(ro, (int)(bw < 32 ? o + (uint32_t)(W - 1) : kNoAccess), 0, 0);
            }
#pragma unroll
            for (int i = 0; i < R; ++i) {
                L.col[side][0][wave * R + i] = c[i] & cm;
                L.col[side][1][wave * R + i] = a[i] | (bw < 32 ? b[i] << bw : 0u);
            }
        }
    }

    const int up = wave > 0 ? wave - 1 : 0, dn = wave < NW - 1 ? wave + 1 : NW - 1;
    // rows [cy0 - left, cy1 + left) are needed once `left` generations remain
    auto needed = [&](int left) { return wy < cy1 + left && wy + R > cy0 - left && wy < H; };

    // the tile's own interior rows (with `ring` the ring's too); a lane holding a ring
    // column writes the ring value it holds, which is dst's own.  The padding of a row may be the caller's:
    // a 16-byte half that reaches past W is stored in pieces of 8, 4, 2 and 1 cells.
    auto store = [&](void* to, bool ring) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rd = plane_rsrc((uint8_t*)to + (size_t)y0 * pitch, bytes);
        // recomputed from the lane: hoisted above the generations, these would hold
        // registers there
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int xl = x0 + ln * 32;
        const int cells = xl >= cx0 && xl < cx1 ? min(W - xl, 32) : 0;  // this lane's cells on the board
        const bool ragged = W % 16 != 0 && x0 + kLtCols >= W;           // uniform
        const int part = ragged ? cells & 15 : 0;                       // cells of such a half
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int y = wy + i;
            if (y < cy0 || y >= cy1 || (!ring && (y < 1 || y > H - 2))) continue;  // uniform
            u32x4_t a, b;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                a[q] = lt_unpack(c[i], q);
                b[q] = lt_unpack(c[i], q + 4);
            }
            const uint32_t o = (uint32_t)(wave * R + i) * p + (uint32_t)xl;
            __builtin_amdgcn_raw_buffer_store_b128(a, rd, (int)(cells >= 16 ? o : kNoAccess), 0, 0);
            __builtin_amdgcn_raw_buffer_store_b128(b, rd, (int)(cells == 32 ? o + 16 : kNoAccess), 0, 0);
            if (!ragged) continue;
            const uint32_t h = o + (cells & 16);
#pragma unroll
            for (int q = 0; q < 4; ++q) a[q] = cells & 16 ? b[q] : a[q];
            const u32x2_t two = {a[0], a[1]};
            __builtin_amdgcn_raw_buffer_store_b64(two, rd, (int)(part & 8 ? h : kNoAccess), 0, 0);
            const uint32_t w4 = part & 8 ? a[2] : a[0];
            __builtin_amdgcn_raw_buffer_store_b32(w4, rd, (int)(part & 4 ? h + (part & 8) : kNoAccess), 0, 0);
            const uint32_t w2 = part & 8 ? (part & 4 ? a[3] : a[2]) : (part & 4 ? a[1] : a[0]);
            __builtin_amdgcn_raw_buffer_store_b16((uint16_t)w2, rd, (int)(part & 2 ? h + (part & 12) : kNoAccess), 0,
                                                  0);
            __builtin_amdgcn_raw_buffer_store_b8((uint8_t)(part & 2 ? w2 >> 16 : w2), rd,
                                                 (int)(part & 1 ? h + (part & 14) : kNoAccess), 0, 0);
        }
    };

    int l = 0;
#pragma unroll 1
    for (; l < k; ++l) {
        uint32_t(*x)[2][kWave] = L.x[l & 1];
        x[wave][0][lane] = c[0];
        x[wave][1][lane] = c[R - 1];
        const bool act = needed(k - 1 - l);
        __syncthreads();
        if (!act) break;
        // uniform; an even k's goes to the buffer that holds its ring, an odd one's (at
        // least 3) to one that does not
        if (KEEP && l + 1 == k && s.prev) store(s.prev, k & 1);
        uint32_t hp0, hp1, hc0, hc1, mc0, mc1, m0, m1;
        lt_sums(x[up][1][lane], hp0, hp1, m0, m1);
        lt_sums(c[0], hc0, hc1, mc0, mc1);
        const uint32_t below = x[dn][0][lane];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            uint32_t hn0, hn1, mn0, mn1;
            lt_sums(i + 1 < R ? c[i + 1 < R ? i + 1 : 0] : below, hn0, hn1, mn0, mn1);
            const uint32_t s0 = lt_xor3(hp0, hn0, mc0), c0 = lt_maj(hp0, hn0, mc0);
            const uint32_t t = lt_xor3(hp1, hn1, mc1), tc = lt_maj(hp1, hn1, mc1);
            // count = s0 + 2 (t + c0) + 4 tc: 2 or 3 where exactly one of t and c0 is set and tc is not
            c[i] = lt_and_or(lt_xor_andn(t, c0, tc), s0, c[i]);
            hp0 = hc0, hp1 = hc1;
            hc0 = hn0, hc1 = hn1, mc0 = mn0, mc1 = mn1;
        }
        if (edge) {  // level l + 1: the ring of the buffer it lives in
            const int odd = (l + 1) & 1;
#pragma unroll
            for (int i = 0; i < R; ++i) {
                if (has_top && i == itop) c[i] = L.ring[0][odd][lane];
                else if (has_bot && i == ibot) c[i] = L.ring[1][odd][lane];
                else if (edge_c) {
                    uint32_t v = 0;
                    if (cm) v = L.col[side][odd][wave * R + i];
                    c[i] = (c[i] & ~cm) | v;
                }
            }
        }
    }
    if (l < k) {  // a wave that is done keeps up with the barriers
#pragma unroll 1
        for (++l; l < k; ++l) __syncthreads();
        return;
    }

    store(s.dst, false);
}

template <int R, int NW, bool KEEP>
__global__ __launch_bounds__(NW * kWave, 8) void k_life_tiles(Sweep2D s, int ntx, int K)
{
    __shared__ LtLds<R, NW> L;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int t = (int)xcd_remap(blockIdx.x, gridDim.x);
    life_tile<R, NW, KEEP>(s, t % ntx, t / ntx, K, K, lane, wave, L);
}

}  // namespace
#endif  // PSKEL_LTILE_INSTANTIATE

}  // namespace pskel
