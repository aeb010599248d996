// Register tiles of the radius-1 2D stencils: launch plans and launches
// (the kernel is k_rtile2d.hpp).
#define PSKEL_RTILE_INSTANTIATE
#include "k_rtile2d.hpp"

namespace pskel {

bool rtile2d_ok(int pattern, int W, int H, size_t pitch)
{
    // the register march (k_march2d.hpp) holds the 9-point stencil's large
    // grids: both are at the VALU's rate there, and its waves overlap less
    // (4096^2: march 11.5 us a sweep, tiles 11.9; 8192^2 36-39 against 39-44;
    // 3000 x 3500 8.5 against 8.4; 2048^2 4.9 against 4.3)
    if (pattern == PAT_BOX9 && (double)W * H > 12e6) return false;
    return rt_fits(W, H, pitch);
}

// a tile outputs rows and columns after q.k sweeps
static bool rt_depth_ok(int W, int H, const RtPlan& q)
{
    return q.k >= 1 && (H <= q.r * q.nw || 2 * q.k < q.r * q.nw) && (W <= kRtCols || 2 * rt_halo_cols(q.k) < kRtCols);
}

namespace {

// Tile shapes and the blocks of each that a CU holds (registers, waves, LDS).
struct RtShape {
    int pattern, r, nw, per_cu;
};
constexpr RtShape kRtShapes[] = {
    {PAT_J5, 2, 16, 2},   {PAT_J5, 4, 8, 4},    {PAT_J5, 4, 16, 2},   {PAT_J5, 8, 8, 3},
    {PAT_BOX9, 2, 8, 4},  {PAT_BOX9, 2, 16, 2}, {PAT_BOX9, 4, 8, 4},  {PAT_BOX9, 4, 16, 2},
    {PAT_CLOUD, 2, 8, 4}, {PAT_CLOUD, 2, 16, 2}, {PAT_CLOUD, 4, 8, 3},
};

double rt_time(const RtShape& h, int W, int H, int k)
{
    const int rows = h.r * h.nw;
    const int64_t nb = (int64_t)rt_tiles(W, kRtCols, rt_halo_cols(k)) * rt_tiles(H, rows, k);
    return rt_launch_time(h.pattern, rows, h.per_cu, nb, (double)W * H, k);
}

}  // namespace

RtPlan rtile2d_plan(int pattern, int W, int H, size_t rem, bool odd)
{
    return plan_fused(
        kRtShapes, rem, odd, kRtMaxDepth,
        [&](const RtShape& h, int k) {
            RtPlan q;
            q.r = h.r;
            q.nw = h.nw;
            q.k = k;
            return h.pattern == pattern && rt_depth_ok(W, H, q);
        },
        [&](const RtShape& h, int k) { return rt_time(h, W, H, k); });
}

namespace {

template <int PAT, int R, int NW>
hipError_t rt_go(const Sweep2D& s, const RtParams& p, int k, double* partials, hipStream_t st)
{
    const int ntx = rt_tiles(s.W, kRtCols, rt_halo_cols(k)), nty = rt_tiles(s.H, R * NW, k);
    const dim3 grid((unsigned)(ntx * nty)), block(NW * kWave);
    if (partials) hipLaunchKernelGGL((k2d_rtile<PAT, R, NW, true, true>), grid, block, 0, st, s, p, ntx, k, partials);
    else if (s.prev) hipLaunchKernelGGL((k2d_rtile<PAT, R, NW, false, true>), grid, block, 0, st, s, p, ntx, k, partials);
    else hipLaunchKernelGGL((k2d_rtile<PAT, R, NW, false, false>), grid, block, 0, st, s, p, ntx, k, partials);
    return hipGetLastError();
}

template <int PAT>
hipError_t rt_shape(const Sweep2D& s, const RtParams& p, const RtPlan& q, double* partials, hipStream_t st)
{
#define PSKEL_RT(R, NW) \
    if (q.r == R && q.nw == NW) return rt_go<PAT, R, NW>(s, p, q.k, partials, st);
    // the shapes of kRtShapes
    PSKEL_RT(2, 16)
    PSKEL_RT(4, 8)
    if constexpr (PAT != PAT_J5) {
        PSKEL_RT(2, 8)
    }
    if constexpr (PAT != PAT_CLOUD) {
        PSKEL_RT(4, 16)
    }
    if constexpr (PAT == PAT_J5) {
        PSKEL_RT(8, 8)
    }
#undef PSKEL_RT
    return hipErrorInvalidValue;
}

}  // namespace

size_t rtile2d_blocks(int W, int H, const RtPlan& q)
{
    return (size_t)rt_tiles(W, kRtCols, rt_halo_cols(q.k)) * rt_tiles(H, q.r * q.nw, q.k);
}

hipError_t launch_2d_rtile(const Sweep2D& s, const Points& pts, const CloudArgs* cloud, int pattern, const RtPlan& q,
                           double* partials, hipStream_t st)
{
    if (!rt_fits(s.W, s.H, s.pitch) || !rt_depth_ok(s.W, s.H, q)) return hipErrorInvalidValue;
    RtParams p{};
    p.coeff = pts.coeff;
    for (int i = 0; i < 9; ++i) p.wt[i] = pts.wt[i];
    if (cloud) {
        p.coeff = cloud->dt;
        p.wx = cloud->wx;
        p.wy = cloud->wy;
        p.xpitch = (uint32_t)cloud->xpitch;
        p.ypitch = (uint32_t)cloud->ypitch;
    }
    if (pattern == PAT_J5) return rt_shape<PAT_J5>(s, p, q, partials, st);
    if (pattern == PAT_BOX9) return rt_shape<PAT_BOX9>(s, p, q, partials, st);
    if (pattern == PAT_CLOUD && cloud) return rt_shape<PAT_CLOUD>(s, p, q, partials, st);
    return hipErrorInvalidValue;
}

}  // namespace pskel
