// Register-tiled 2D sweep bodies shared by the standalone tuned kernels and the
// batched persistent kernel.  A block of (64, NWY) threads computes one tile.
#pragma once

#include "k_common.hpp"

namespace pskel {

// ---------------------------------------------------------------------------
// point evaluation over a register window (radius 1 patterns)
// ---------------------------------------------------------------------------
// Window access: row i (0..2 = h-1..h+1), column j in -1..4 relative to the
// lane's float4 (-1: left halo, 4: right halo).
struct Win {
    const float4* v;  // 3 rows
    const float* lf;  // 3 left halos
    const float* rt;  // 3 right halos
    __device__ __forceinline__ float at(int i, int j) const
    {
        if (j < 0) return lf[i];
        if (j > 3) return rt[i];
        const float4 x = v[i];
        return j == 0 ? x.x : j == 1 ? x.y : j == 2 ? x.z : x.w;
    }
};

template <int PAT, class PT>
__device__ __forceinline__ float eval_pat(const Win& W, int j, const PT& p)
{
    if constexpr (PAT == PAT_J5) {
        float acc = W.at(0, j) + W.at(2, j);
        acc = acc + W.at(1, j - 1);
        acc = acc + W.at(1, j + 1);
        return p.coeff * acc;
    } else {  // PAT_BOX9, row-major weighted sum
        float acc = p.wt[0] * W.at(0, j - 1);
        acc = acc + p.wt[1] * W.at(0, j);
        acc = acc + p.wt[2] * W.at(0, j + 1);
        acc = acc + p.wt[3] * W.at(1, j - 1);
        acc = acc + p.wt[4] * W.at(1, j);
        acc = acc + p.wt[5] * W.at(1, j + 1);
        acc = acc + p.wt[6] * W.at(2, j - 1);
        acc = acc + p.wt[7] * W.at(2, j);
        acc = acc + p.wt[8] * W.at(2, j + 1);
        return acc;
    }
}

// ---------------------------------------------------------------------------
// tuned tile: 64 lanes x float4 = 256 columns per wave, RY rows per lane;
// block = (64, NWY), the NWY waves stack along h; tile (tx, ty) covers columns
// [256 tx, 256 tx + 256) and rows [NWY RY ty, NWY RY (ty + 1)).
// ---------------------------------------------------------------------------
template <int PAT, int RY, class PT>
__device__ __forceinline__ void tile_f32(const Sweep2D& s, const PT& p, int tx, int ty)
{
    const int lane = threadIdx.x;
    const int w0 = tx * 256;
    const int w = w0 + lane * 4;
    const int hb = (ty * (int)blockDim.y + (int)threadIdx.y) * RY;  // first output row
    const int H = s.H, Wd = s.W, r = s.radius;
    const float* __restrict__ src = (const float*)s.src;
    float* __restrict__ dst = (float*)s.dst;
    const size_t pitch = s.pitch;
    const bool col_live = w < Wd;

    float4 v[RY + 2];
    float lfl[RY + 2], rtl[RY + 2];
#pragma unroll
    for (int i = 0; i < RY + 2; ++i) {
        const int h = hb - 1 + i;
        v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        lfl[i] = 0.f;
        rtl[i] = 0.f;
        if (h >= 0 && h < H) {
            const float* row = src + (size_t)h * pitch;
            if (col_live) v[i] = *reinterpret_cast<const float4*>(row + w);
            if (lane == 0 && w0 > 0) lfl[i] = row[w0 - 1];
            if (lane == kWave - 1 && w0 + 256 < Wd) rtl[i] = row[w0 + 256];
        }
    }
    float lf[RY + 2], rt[RY + 2];
#pragma unroll
    for (int i = 0; i < RY + 2; ++i) {
        lf[i] = from_lower_lane(v[i].w, lfl[i]);  // lane 0: the cell loaded for it
        rt[i] = from_upper_lane(v[i].x, rtl[i]);  // lane 63: likewise
    }
    if (!col_live) return;
    const bool full = (w >= r) && (w + 3 < Wd - r);
#pragma unroll
    for (int i = 1; i <= RY; ++i) {
        const int h = hb - 1 + i;
        if (h < r || h >= H - r) continue;
        const Win win{&v[i - 1], &lf[i - 1], &rt[i - 1]};
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = eval_pat<PAT, PT>(win, j, p);
        float* row = dst + (size_t)h * pitch + w;
        if (full) {
            *reinterpret_cast<float4*>(row) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (w + j >= r && w + j < Wd - r) row[j] = o[j];
        }
    }
}

// ---------------------------------------------------------------------------
// SWAR helpers.  Byte k of a little-endian word is cell w0 + k.
// ---------------------------------------------------------------------------
constexpr uint64_t kOnes = 0x0101010101010101ull;
constexpr uint64_t kHigh = 0x8080808080808080ull;
constexpr uint64_t kLow7 = 0x7f7f7f7f7f7f7f7full;

// 0x01 in every byte equal to k (byte values <= 11, so no carry leaves a byte).
__device__ __forceinline__ uint64_t bytes_eq(uint64_t x, uint64_t k)
{
    const uint64_t y = x ^ (k * kOnes);
    const uint64_t nz = (y + kLow7) & kHigh;
    return ((~nz) & kHigh) >> 7;
}

__device__ __forceinline__ uint64_t life_rule(uint64_t cnt, uint64_t cur)
{
    return bytes_eq(cnt, 3) | (bytes_eq(cnt, 2) & cur);
}

// A 16-cell lane segment: lo = cells 0..7, hi = cells 8..15, plus the byte to
// the left (cell -1) and to the right (cell 16).
struct Seg {
    uint64_t lo, hi;
    uint32_t l, r;
};

// Horizontal sums for a row segment: with_c = left + centre + right,
// no_c = left + right (bytewise, <= 3).
__device__ __forceinline__ void hsum(const Seg& s, uint64_t& lo3, uint64_t& hi3, uint64_t& lo2,
                                     uint64_t& hi2)
{
    const uint64_t lo_l = (s.lo << 8) | (uint64_t)s.l;
    const uint64_t hi_l = (s.hi << 8) | (s.lo >> 56);
    const uint64_t lo_r = (s.lo >> 8) | (s.hi << 56);
    const uint64_t hi_r = (s.hi >> 8) | ((uint64_t)s.r << 56);
    lo2 = lo_l + lo_r;
    hi2 = hi_l + hi_r;
    lo3 = lo2 + s.lo;
    hi3 = hi2 + s.hi;
}

// ---------------------------------------------------------------------------
// SWAR kernel: wave = 64 lanes x 16 cells = 1024 columns; block = (64, NWY).
// ---------------------------------------------------------------------------
template <int RY>
__device__ __forceinline__ void tile_life(const Sweep2D& s, int tx, int ty)
{
    const int lane = threadIdx.x;
    const int w0 = tx * 1024;
    const int w = w0 + lane * 16;
    const int hb = (ty * (int)blockDim.y + (int)threadIdx.y) * RY;
    const int H = s.H, Wd = s.W, r = s.radius;
    const size_t pitch = s.pitch;
    const uint8_t* __restrict__ src = (const uint8_t*)s.src;
    uint8_t* __restrict__ dst = (uint8_t*)s.dst;
    const bool col_live = w < Wd;

    Seg g[RY + 2];
    uint32_t el[RY + 2], er[RY + 2];
#pragma unroll
    for (int i = 0; i < RY + 2; ++i) {
        const int h = hb - 1 + i;
        g[i].lo = 0;
        g[i].hi = 0;
        el[i] = 0;
        er[i] = 0;
        if (h >= 0 && h < H) {
            const uint8_t* row = src + (size_t)h * pitch;
            if (col_live) {
                const uint4 x = *reinterpret_cast<const uint4*>(row + w);
                g[i].lo = (uint64_t)x.x | ((uint64_t)x.y << 32);
                g[i].hi = (uint64_t)x.z | ((uint64_t)x.w << 32);
            }
            if (lane == 0 && w0 > 0) el[i] = row[w0 - 1];
            if (lane == kWave - 1 && w0 + 1024 < Wd) er[i] = row[w0 + 1024];
        }
    }
#pragma unroll
    for (int i = 0; i < RY + 2; ++i) {
        g[i].l = from_lower_lane((uint32_t)(g[i].hi >> 56), el[i]);
        g[i].r = from_upper_lane((uint32_t)(g[i].lo & 0xffu), er[i]);
    }
    if (!col_live) return;

    uint64_t s3lo[RY + 2], s3hi[RY + 2], s2lo[RY + 2], s2hi[RY + 2];
#pragma unroll
    for (int i = 0; i < RY + 2; ++i) hsum(g[i], s3lo[i], s3hi[i], s2lo[i], s2hi[i]);

    const bool full = (w >= r) && (w + 15 < Wd - r);
#pragma unroll
    for (int i = 1; i <= RY; ++i) {
        const int h = hb - 1 + i;
        if (h < r || h >= H - r) continue;
        const uint64_t clo = s3lo[i - 1] + s3lo[i + 1] + s2lo[i];
        const uint64_t chi = s3hi[i - 1] + s3hi[i + 1] + s2hi[i];
        const uint64_t nlo = life_rule(clo, g[i].lo);
        const uint64_t nhi = life_rule(chi, g[i].hi);
        uint8_t* row = dst + (size_t)h * pitch + w;
        if (full) {
            uint4 x;
            x.x = (uint32_t)nlo;
            x.y = (uint32_t)(nlo >> 32);
            x.z = (uint32_t)nhi;
            x.w = (uint32_t)(nhi >> 32);
            *reinterpret_cast<uint4*>(row) = x;
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                if (w + j >= r && w + j < Wd - r)
                    row[j] = (uint8_t)((j < 8 ? (nlo >> (8 * j)) : (nhi >> (8 * (j - 8)))) & 0xffu);
            }
        }
    }
}


// ---------------------------------------------------------------------------
// temporal tile: core CX x CY cells, loaded region (CX + 8) x (CY + 2K) with a
// 4-column aligned halo (K <= 4), kgen <= K sweeps in an LDS ping-pong (A, B:
// ttile_lds floats each); 256 threads, tid = 0..255, all of which must call it
// (it synchronises the block).  Tile (bx, by) has its core at columns
// [CX bx, CX bx + CX) and rows [CY by, CY by + CY).  Cells outside the
// interior are never computed: at level j an LDS buffer holds the ring of the
// global buffer that level j lives in (level parity alternates between src and
// ring_other), so halo reads near the grid edge see exactly what a single
// sweep would see.  Level j is exact on the core widened by K - j cells, so
// fewer levels than K still leave the core exact.
// ---------------------------------------------------------------------------
template <int K, int CX, int CY>
__host__ __device__ constexpr int ttile_lds()
{
    return (CY + 2 * K) * (CX + 8);
}

template <int PAT, int K, int CX, int CY, class PT>
__device__ __forceinline__ void ttile_body(const Sweep2D& s, const PT& p, int bx, int by, int kgen, int tid,
                                           float* __restrict__ A, float* __restrict__ B)
{
    constexpr int LX = CX + 8;
    constexpr int LY = CY + 2 * K;
    constexpr int NT = 256;
    const int w0 = bx * CX;                    // core origin
    const int h0 = by * CY;
    const int gx0 = w0 - 4, gy0 = h0 - K;      // loaded region origin
    const int H = s.H, Wd = s.W, r = s.radius;
    const size_t pitch = s.pitch;
    const float* __restrict__ src = (const float*)s.src;
    const float* __restrict__ oth = (const float*)s.ring_other;

    // load: float4 granules, LX/4 per row
    constexpr int G = LX / 4;
    for (int q = tid; q < G * LY; q += NT) {
        const int y = q / G, x4 = (q - y * G) * 4;
        const int gh = gy0 + y, gw = gx0 + x4;
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
        if (gh >= 0 && gh < H && gw >= 0 && gw < (int)pitch) {
            a = *reinterpret_cast<const float4*>(src + (size_t)gh * pitch + gw);
            const bool ring_row = gh < r || gh >= H - r;
            const bool ring_col = gw < r || gw + 3 >= Wd - r;
            if (ring_row || ring_col) b = *reinterpret_cast<const float4*>(oth + (size_t)gh * pitch + gw);
        }
        *reinterpret_cast<float4*>(&A[y * LX + x4]) = a;
        *reinterpret_cast<float4*>(&B[y * LX + x4]) = b;
    }
    __syncthreads();

    // Level j: each thread walks one column x of the level's region down one
    // of NS strips of rows, keeping the row above and its own row (x-1, x, x+1)
    // in registers, so a cell costs three LDS reads (the row below).  Sums keep
    // the mask order.
    constexpr int NS = NT / 128;  // strips per column
    static_assert(LX <= 128, "one thread per column of the loaded region");
    // a strip is two whole waves, so its row range is uniform across the wave
    const int col = tid % 128, strip = __builtin_amdgcn_readfirstlane(tid / 128);
#pragma unroll
    for (int j = 1; j <= K; ++j) {
        if (j > kgen) break;  // uniform
        const float* __restrict__ P = (j & 1) ? A : B;
        float* __restrict__ Q = (j & 1) ? B : A;
        const int xlo = 4 - (K - j), xhi = 4 + CX + (K - j);
        const int ylo = j, yhi = LY - j;
        const int nx = xhi - xlo, ny = yhi - ylo;
        const int rows = (ny + NS - 1) / NS;
        const int x = xlo + col;
        const int gw = gx0 + x;
        // only interior cells are written: a ring column's lane and the ring
        // rows of the strip compute nothing (their LDS cells keep the ring)
        if (col < nx && gw >= r && gw < Wd - r) {
            const int ys = ylo + strip * rows;
            const int ya = max(ys, r - gy0), yb = min(min(ys + rows, yhi), H - r - gy0);
            const float* c = P + (ya - 1) * LX + x;
            float um = c[-1], u0 = c[0], up = c[1];                 // row y - 1
            float cm = c[LX - 1], c0 = c[LX], cp = c[LX + 1];       // row y
#pragma unroll 3
            for (int y = ya; y < yb; ++y) {
                c += LX;
                const float dm = c[LX - 1], d0 = c[LX], dp = c[LX + 1];  // row y + 1
                float acc;
                if constexpr (PAT == PAT_J5) {
                    acc = u0 + d0;
                    acc = acc + cm;
                    acc = acc + cp;
                    acc = p.coeff * acc;
                } else {
                    acc = p.wt[0] * um;
                    acc = acc + p.wt[1] * u0;
                    acc = acc + p.wt[2] * up;
                    acc = acc + p.wt[3] * cm;
                    acc = acc + p.wt[4] * c0;
                    acc = acc + p.wt[5] * cp;
                    acc = acc + p.wt[6] * dm;
                    acc = acc + p.wt[7] * d0;
                    acc = acc + p.wt[8] * dp;
                }
                Q[y * LX + x] = acc;
                um = cm; u0 = c0; up = cp;
                cm = dm; c0 = d0; cp = dp;
            }
        }
        __syncthreads();
    }

    const float* __restrict__ R = (kgen & 1) ? B : A;
    float* __restrict__ dst = (float*)s.dst;
    for (int q = tid; q < CX * CY; q += NT) {
        const int y = q / CX, x = q % CX;
        const int gh = h0 + y, gw = w0 + x;
        if (gh < r || gh >= H - r || gw < r || gw >= Wd - r) continue;
        dst[(size_t)gh * pitch + gw] = R[(y + K) * LX + (x + 4)];
    }
    // the caller may reuse A and B for its next tile
    __syncthreads();
}

}  // namespace pskel
