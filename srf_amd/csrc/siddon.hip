// Siddon ray-driven projector for CDNA4 (gfx950): the untiled ops
// (siddon.cu.cc:424-675).  Ray setup, the walks and their precision are in
// siddon_core.h.
//
// Unlike the reference, a ray whose start voxel falls outside the grid is
// skipped (the reference indexes out of bounds there), and walks are bounded: the
// count by gx+gy+gz+3 steps, the others by the crossing that leaves the image, at
// most one slab for each plane of the dominant axis; both only affect degenerate
// rays.
#include "siddon_binned.h"

namespace srfx {
namespace {

// L lanes per ray (walk_ray).  The mode's reference semantics: projection,
// A^T(1 / v) over v > 0, the map likewise without TOF, plain adjoint, and the
// OSEM pass (both).
template <int MODE, int L, bool TOF>
__global__ __launch_bounds__(256) void siddon_kernel(SidParams p)
{
    constexpr int R = 256 / L; // rays of the workgroup (ray_sum)
    const int64_t e = (int64_t)blockIdx.x * R + (int)threadIdx.x % R;
    const int sub = (int)threadIdx.x / R;
    const bool valid = e < p.n;
    SidRay r;
    r.tend = -1.0;
    r.weight = 0.0f;
    r.t_tof = 0.0;
    if (valid) {
        Walk w;
        setup_walk<MODE>(p, e, w);
        if (w.ok)
            make_ray(w, r);
    }
    float scale = 0.0f;
    if (MODE == kProj || MODE == kOsem) {
        const float pv = ray_sum<L>(r.tend > 0.0 ? gather_ray<TOF, L>(p, r, sub) : 0.0f);
        if (MODE == kProj) {
            if (valid && sub == 0)
                p.out[e] = pv;
            return;
        }
        scale = pv > 0.0f ? 1.0f / pv : 0.0f;
    } else if (valid) {
        const float v = p.val[e];
        scale = MODE == kAdj ? v : (v > 0.0f ? 1.0f / v : 0.0f);
    }
    if (scale != 0.0f && r.tend > 0.0)
        scatter_ray<TOF, L>(p, r, sub, scale);
}

__global__ __launch_bounds__(256) void siddon_count(SidParams p)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int cnt = 0;
    if (e < p.n) {
        Walk w;
        setup_walk<kCount>(p, e, w);
        if (w.ok)
            cnt = p.use_tof ? count_segments<true>(p, w) : count_segments<false>(p, w);
        if (p.nnz)
            p.nnz[e] = cnt;
    }
    if (p.nnz_total) {
        unsigned long long c = (unsigned long long)cnt;
        for (int off = 32; off > 0; off >>= 1)
            c += __shfl_down(c, off, 64);
        if ((threadIdx.x & 63) == 0 && c)
            atomicAdd(p.nnz_total, c);
    }
}

template <int MODE, int L>
int launch_lanes(const SidParams &p, hipStream_t st)
{
    const dim3 grid(blocks_for(p.n * L, 256)), block(256);
    if constexpr (MODE != kMap) {
        if (p.use_tof) {
            hipLaunchKernelGGL((siddon_kernel<MODE, L, true>), grid, block, 0, st, p);
            return launch_status();
        }
    }
    hipLaunchKernelGGL((siddon_kernel<MODE, L, false>), grid, block, 0, st, p);
    return launch_status();
}

template <int MODE>
int launch(const SidParams &p, hipStream_t st)
{
    if (p.n == 0)
        return SRFX_OK;
    switch (lanes_per_ray(p.n)) {
    case 16:
        return launch_lanes<MODE, 16>(p, st);
    case 4:
        return launch_lanes<MODE, 4>(p, st);
    default:
        return launch_lanes<MODE, 1>(p, st);
    }
}

} // namespace

int siddon_setup(SidParams &p, const float *lors, int64_t n, int64_t ld, const srfx_grid &g,
                 float tof_bin, float tof_sigma2)
{
    if (n < 0 || (n > 0 && (!lors || ld < n)) || !grid_ok(g))
        return SRFX_EINVAL;
    p = SidParams{};
    p.lors = lors;
    p.n = n;
    p.ld = ld;
    for (int c = 0; c < 3; c++) {
        p.g[c] = g.shape[c];
        p.size[c] = g.size[c];
        p.center[c] = g.center[c];
    }
    Strides s = grid_strides(g);
    p.s[0] = p.o[0] = (int)s.x;
    p.s[1] = p.o[1] = (int)s.y;
    p.s[2] = p.o[2] = (int)s.z;
    p.tof_bin = tof_bin;
    p.tof_sigma2 = tof_sigma2;
    p.use_tof = tof_sigma2 < kTofThreshold ? 1 : 0;
    return SRFX_OK;
}

} // namespace srfx

using namespace srfx;

extern "C" int srfx_siddon_project(const float *lors, int64_t n, int64_t ld, const float *image,
                                   srfx_grid grid, float tof_bin, float tof_sigma2, float *proj,
                                   uint32_t flags, void *stream)
{
    (void)flags;
    SidParams p;
    int rc = siddon_setup(p, lors, n, ld, grid, tof_bin, tof_sigma2);
    if (rc)
        return rc;
    if (n > 0 && (!image || !proj))
        return SRFX_EINVAL;
    p.img = image;
    p.out = proj;
    return launch<kProj>(p, (hipStream_t)stream);
}

static int sid_scatter(int mode, const float *lors, int64_t n, int64_t ld, const float *vals,
                       srfx_grid grid, float tof_bin, float tof_sigma2, float *image,
                       uint32_t flags, void *stream)
{
    SidParams p;
    int rc = siddon_setup(p, lors, n, ld, grid, tof_bin, tof_sigma2);
    if (rc)
        return rc;
    if (!image || (n > 0 && !vals))
        return SRFX_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    rc = zero_grid(image, grid, flags, st);
    if (rc)
        return rc;
    p.val = vals;
    p.out = image;
    if (siddon_binned_ok(p, st)) {
        bool done = false;
        rc = siddon_binned_scatter(mode, p, st, &done);
        if (rc || done)
            return rc;
    }
    switch (mode) {
    case kBack:
        return launch<kBack>(p, st);
    case kAdj:
        return launch<kAdj>(p, st);
    default:
        return launch<kMap>(p, st);
    }
}

extern "C" int srfx_siddon_backproject(const float *lors, int64_t n, int64_t ld,
                                       const float *lors_value, srfx_grid grid, float tof_bin,
                                       float tof_sigma2, float *image, uint32_t flags,
                                       void *stream)
{
    return sid_scatter(kBack, lors, n, ld, lors_value, grid, tof_bin, tof_sigma2, image, flags,
                       stream);
}

extern "C" int srfx_siddon_backproject_adjoint(const float *lors, int64_t n, int64_t ld,
                                               const float *g, srfx_grid grid, float tof_bin,
                                               float tof_sigma2, float *image, uint32_t flags,
                                               void *stream)
{
    return sid_scatter(kAdj, lors, n, ld, g, grid, tof_bin, tof_sigma2, image, flags, stream);
}

extern "C" int srfx_siddon_maplors(const float *lors, int64_t n, int64_t ld,
                                   const float *lors_value, srfx_grid grid, float *image,
                                   uint32_t flags, void *stream)
{
    return sid_scatter(kMap, lors, n, ld, lors_value, grid, 0.0f, 1.0e6f, image, flags, stream);
}

extern "C" int srfx_siddon_osem_subset(const float *lors, int64_t n, int64_t ld,
                                       const float *image, srfx_grid grid, float tof_bin,
                                       float tof_sigma2, float *bp, uint32_t flags, void *stream)
{
    SidParams p;
    int rc = siddon_setup(p, lors, n, ld, grid, tof_bin, tof_sigma2);
    if (rc)
        return rc;
    if (!bp || (n > 0 && !image))
        return SRFX_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    rc = zero_grid(bp, grid, flags, st);
    if (rc)
        return rc;
    p.img = image;
    p.out = bp;
    if (siddon_binned_ok(p, st)) {
        bool done = false;
        rc = siddon_binned_scatter(kOsem, p, st, &done);
        if (rc || done)
            return rc;
    }
    return launch<kOsem>(p, st);
}

extern "C" int srfx_siddon_count_nnz(const float *lors, int64_t n, int64_t ld, srfx_grid grid,
                                     float tof_bin, float tof_sigma2, int32_t *nnz_per_event,
                                     uint64_t *nnz_total, void *stream)
{
    SidParams p;
    int rc = siddon_setup(p, lors, n, ld, grid, tof_bin, tof_sigma2);
    if (rc)
        return rc;
    p.nnz = nnz_per_event;
    p.nnz_total = (unsigned long long *)nnz_total;
    if (p.n == 0)
        return SRFX_OK;
    hipLaunchKernelGGL(siddon_count, dim3(blocks_for(p.n, 256)), dim3(256), 0,
                       (hipStream_t)stream, p);
    return launch_status();
}

extern "C" int srfx_siddon_scatter_rule(int64_t n, srfx_grid grid, float tof_bin,
                                        float tof_sigma2, int32_t *binned)
{
    SidParams p;
    if (n < 0 || !binned)
        return SRFX_EINVAL;
    const int rc = siddon_setup(p, nullptr, 0, 0, grid, tof_bin, tof_sigma2);
    if (rc)
        return rc;
    p.n = n;
    *binned = siddon_binned_rule(p) ? 1 : 0;
    return SRFX_OK;
}
