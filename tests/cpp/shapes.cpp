// The 2D kernels of libpskel_amd.so by tile shape, for tests/test_gpu_tile_shapes.py
// and tests/test_tile_plans_cpu.py: a run's plan picks the shape by the grid's size,
// here the caller does.  Launches go to the null stream; a shape that is not built is
// an error (hipErrorInvalidValue), before any launch.
#include "../../pskel_amd/csrc/pskel_internal.hpp"

using namespace pskel;

namespace {

// one launch: src -> dst, ring_other holds the other parity's ring
struct Job {
    const void* src;
    void* dst;
    const void* ring;
    void* prev;        // the state before the last sweep (NULL: no)
    double* partials;  // residual partials (NULL: no)
    const float* wx;   // CLOUDSIM's fields
    const float* wy;
    uint64_t pitch, xpitch, ypitch;
    int32_t W, H, pattern, k;
    float coeff;
    float wt[9];
};

Sweep2D sweep(const Job& j)
{
    Sweep2D s;
    s.src = j.src;
    s.dst = j.dst;
    s.ring_other = j.ring;
    s.prev = j.prev;
    s.W = j.W;
    s.H = j.H;
    s.pitch = j.pitch;
    s.radius = 1;
    return s;
}

Points points(const Job& j)
{
    Points p{};
    p.coeff = j.coeff;
    p.radius = 1;
    for (int i = 0; i < 9; ++i) p.wt[i] = j.wt[i];
    return p;
}

RtPlan plan_of(int r, int nw, int k)
{
    RtPlan q;
    q.r = r;
    q.nw = nw;
    q.k = k;
    return q;
}

}  // namespace

extern "C" {

int shapes_job_size() { return (int)sizeof(Job); }

int shapes_rtile(const Job* j, int r, int nw)
{
    CloudArgs ca;
    ca.wx = j->wx;
    ca.wy = j->wy;
    ca.xpitch = j->xpitch;
    ca.ypitch = j->ypitch;
    ca.dt = j->coeff;
    return (int)launch_2d_rtile(sweep(*j), points(*j), j->pattern == PAT_CLOUD ? &ca : nullptr, j->pattern,
                                plan_of(r, nw, j->k), j->partials, nullptr);
}

uint64_t shapes_rtile_blocks(int W, int H, int r, int nw, int k) { return rtile2d_blocks(W, H, plan_of(r, nw, k)); }

int shapes_life(const Job* j, int r, int nw) { return (int)launch_life_tiles(sweep(*j), plan_of(r, nw, j->k), nullptr); }

int shapes_march(const Job* j, int seg)
{
    pskel_launch_cfg_t cfg{};
    cfg.tile_x = 4;
    cfg.tile_z = seg;
    return (int)launch_2d_march_f32(sweep(*j), points(*j), j->pattern, j->k, cfg, nullptr);
}

int shapes_ttile(const Job* j, int rows)
{
    pskel_launch_cfg_t cfg{};
    cfg.tile_y = rows;
    return (int)launch_2d_ttile_f32(sweep(*j), points(*j), j->pattern, j->k, cfg, nullptr);
}

// one sweep of an arbitrary mask through its LDS tile: (H, W, D) in 3D, D = 1 and
// pitched rows of W cells in 2D
int shapes_points(const pskel_stencil_desc_t* d, int ndim, const void* src, void* dst, double* partials, int W, int H,
                  int D, uint64_t pitch, int storage, float offset, int rounding, uint32_t seed, uint64_t sweep_no)
{
    Points p;
    fill_points(p, *d, ndim);
    if (ndim == 2) {
        Sweep2D s;
        s.src = src;
        s.dst = dst;
        s.ring_other = nullptr;
        s.W = W;
        s.H = H;
        s.pitch = pitch;
        s.radius = p.radius;
        return (int)launch_2d_points_f32(s, p, nullptr);
    }
    Sweep3D s{};
    s.src = src;
    s.dst = dst;
    s.W = W;
    s.H = H;
    s.D = D;
    s.pitch = pitch;
    s.radius = p.radius;
    s.store_offset = offset;
    s.partials = partials;
    s.rounding = rounding;
    s.seed = seed;
    s.sweep = sweep_no;
    s.c0 = storage == PSKEL_DTYPE_F32 ? 0.0f : scaled_sum_offset_term(p.coeff, p.np, offset);
    return (int)launch_3d_points(s, p, storage, nullptr);
}

// its blocks (0: the halo does not fit) and whether a run takes it over the plain
// kernel with blocks of bx by `by` lanes
uint64_t shapes_points_blocks(const pskel_stencil_desc_t* d, int W, int H, int D)
{
    Points p;
    fill_points(p, *d, 3);
    Sweep3D s{};
    s.W = W;
    s.H = H;
    s.D = D;
    return points3d_blocks(s, p);
}

int shapes_points_pay(const pskel_stencil_desc_t* d, int ndim, int W, int H, int D, int half, int bx, int by)
{
    Points p;
    fill_points(p, *d, ndim);
    return ndim == 2 ? points_pay(p, true, 1, H, W, half != 0, bx, by) : points_pay(p, false, H, W, D, half != 0, bx, by);
}

// the next launch of a run with `rem` sweeps to go: {r, nw, k}
void shapes_plan(int pattern, int W, int H, uint64_t rem, int odd, int32_t* out)
{
    const RtPlan q = pattern == PAT_LIFE8 ? life_tiles_plan(W, H, rem, odd != 0) : rtile2d_plan(pattern, W, H, rem, odd != 0);
    out[0] = q.r;
    out[1] = q.nw;
    out[2] = q.k;
}

}  // extern "C"
