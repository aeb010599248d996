// Game of Life (B3/S23) sweeps on u8 grids for gfx950, bit-exact integer work.
//
// Reference rule: the GOL_KERNEL formula (include/PSkelStencil.hpp:389-440),
// sum of the 8 Moore neighbours, alive if sum == 3 or (sum == 2 and alive).
// Interior-only like every 2D runner (include/PSkelStencil.hpp:576, 2235-2255).
//
//   k_life_plain  one lane per cell, the caller's block: the runCUDA shape.
//   k_life_swar   16 cells per lane packed in two u64 words; horizontal
//                 neighbours by byte shifts plus one cross-lane exchange per row,
//                 counts and rule evaluated bytewise (SWAR), RY rows per lane.
//   k_life_tiles  many generations per launch on cells packed one bit each, a
//                 tile in the registers of a block (k_ltile.hpp).
#include "k_tiles2d.hpp"
#define PSKEL_LTILE_INSTANTIATE
#include "k_ltile.hpp"

namespace pskel {

namespace {

// ---------------------------------------------------------------------------
// plain
// ---------------------------------------------------------------------------
template <int NP>
__global__ __launch_bounds__(1024) void k_life_plain(Sweep2D s, Points p)
{
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    const int h = blockIdx.y * blockDim.y + threadIdx.y;
    const int r = s.radius;
    if (w < r || w >= s.W - r || h < r || h >= s.H - r) return;
    const uint8_t* __restrict__ c = (const uint8_t*)s.src + (size_t)h * s.pitch + w;
    const ptrdiff_t pitch = (ptrdiff_t)s.pitch;
    int n = 0;
    const int np = NP > 0 ? NP : p.np;
#pragma unroll
    for (int i = 0; i < (NP > 0 ? NP : kMaxPoints); ++i) {
        if (NP == 0 && i >= np) break;
        n += c[p.dh[i] * pitch + p.dw[i]];
    }
    ((uint8_t*)s.dst)[(size_t)h * s.pitch + w] = (n == 3 || (n == 2 && c[0] == 1)) ? 1 : 0;
}

template <int RY>
__global__ __launch_bounds__(256) void k_life_swar(Sweep2D s)
{
    tile_life<RY>(s, blockIdx.x, blockIdx.y);
}

}  // namespace

bool life_tiles_ok(size_t pitch) { return lt_fits(pitch); }

static bool lt_depth_ok(int H, const RtPlan& q)
{
    return q.k >= 1 && q.k <= kLtMaxDepth && (H <= q.r * q.nw || 2 * q.k < q.r * q.nw);
}

// Tile shapes and the blocks of each that a CU holds.
struct LtShape {
    int r, nw, per_cu;
};
static constexpr LtShape kLtShapes[] = {{2, 8, 4}, {2, 16, 2}, {4, 16, 2}, {8, 8, 4}, {8, 16, 2}};

RtPlan life_tiles_plan(int W, int H, size_t rem, bool odd)
{
    return plan_fused(
        kLtShapes, rem, odd, kLtMaxDepth,
        [&](const LtShape& h, int k) {
            RtPlan q;
            q.r = h.r;
            q.nw = h.nw;
            q.k = k;
            return lt_depth_ok(H, q);
        },
        [&](const LtShape& h, int k) {
            const int rows = h.r * h.nw;
            const int64_t nb = (int64_t)lt_tiles(W, kLtCols, 32) * lt_tiles(H, rows, k);
            return lt_launch_time(rows, h.per_cu, nb, (double)W * H, k);
        });
}

hipError_t launch_life_tiles(const Sweep2D& s, const RtPlan& q, hipStream_t st)
{
    if (!lt_fits(s.pitch) || !lt_depth_ok(s.H, q)) return hipErrorInvalidValue;
    const int ntx = lt_tiles(s.W, kLtCols, 32);
    const dim3 grid((unsigned)(ntx * lt_tiles(s.H, q.r * q.nw, q.k))), block(q.nw * kWave);
#define PSKEL_LT(R, NW) \
    if (q.r == R && q.nw == NW && s.prev)                                                     \
        hipLaunchKernelGGL((k_life_tiles<R, NW, true>), grid, block, 0, st, s, ntx, q.k);     \
    else if (q.r == R && q.nw == NW)                                                          \
        hipLaunchKernelGGL((k_life_tiles<R, NW, false>), grid, block, 0, st, s, ntx, q.k)
    // the shapes of kLtShapes
    PSKEL_LT(2, 8);
    else PSKEL_LT(2, 16);
    else PSKEL_LT(4, 16);
    else PSKEL_LT(8, 8);
    else PSKEL_LT(8, 16);
    else return hipErrorInvalidValue;
#undef PSKEL_LT
    return hipGetLastError();
}

hipError_t launch_life_plain(const Sweep2D& s, const Points& p, int bx, int by, hipStream_t st)
{
    const dim3 block(bx, by);
    const dim3 grid((s.W + bx - 1) / bx, (s.H + by - 1) / by);
    if (p.np == 8) hipLaunchKernelGGL((k_life_plain<8>), grid, block, 0, st, s, p);
    else hipLaunchKernelGGL((k_life_plain<0>), grid, block, 0, st, s, p);
    return hipGetLastError();
}

hipError_t launch_life_tuned(const Sweep2D& s, const pskel_launch_cfg_t& cfg, hipStream_t st)
{
    const int ry = cfg.tile_y > 0 ? cfg.tile_y : 4;
    const int nwy = cfg.tile_z > 0 ? cfg.tile_z : 4;
    if (nwy < 1 || nwy > 4) return hipErrorInvalidValue;
    const dim3 block(kWave, nwy);
#define PSKEL_LIFE_CASE(RYV)                                                                     \
    case RYV: {                                                                                  \
        const dim3 grid((s.W + 1023) / 1024, (s.H + nwy * RYV - 1) / (nwy * RYV));               \
        hipLaunchKernelGGL((k_life_swar<RYV>), grid, block, 0, st, s);                           \
        break;                                                                                   \
    }
    switch (ry) {
        PSKEL_LIFE_CASE(1)
        PSKEL_LIFE_CASE(2)
        PSKEL_LIFE_CASE(4)
        PSKEL_LIFE_CASE(8)
        PSKEL_LIFE_CASE(16)
    default: return hipErrorInvalidValue;
    }
#undef PSKEL_LIFE_CASE
    return hipGetLastError();
}

}  // namespace pskel
