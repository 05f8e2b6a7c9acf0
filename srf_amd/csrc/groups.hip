// The OSEM step of one subset's plans, all axis groups in one launch per kernel
// (srfx_tor_plan_osem_groups): op-frame copies, projections into the walk
// records, tiled backprojection of 1/p.
#include <algorithm>

#include "frame_core.h"
#include "tile_core.h"

using namespace srfx;

namespace srfx {
namespace {

constexpr int kMaxGroups = 3;

// One group's plan: its parameters (img: the op frame, out: the
// backprojection), and where its workgroups start in the launches.
struct GroupJob {
    TorParams p;
    TileGeom g;
    const TileChunk *chunks;
    const int *list;
    float4 *rec;
    float *frame;
    const float *image;
    int64_t wx, wy, wz; // world strides of the op axes
    int tx, ty;         // frame tiles per slice
    int nchunks;
    unsigned frame0, proj0;
};

// The groups, most chunks first.
struct GroupSet {
    int n;
    GroupJob j[kMaxGroups];
};

__global__ __launch_bounds__(256) void group_frames(GroupSet s)
{
    __shared__ float tile[kFrameTile][kFrameTile + 1];
    int k = 0;
    while (k + 1 < s.n && blockIdx.x >= s.j[k + 1].frame0)
        k++;
    const GroupJob &j = s.j[k];
    const unsigned t = blockIdx.x - j.frame0, r = t / (unsigned)j.tx;
    frame_tile(j.image, j.p.gx, j.p.gy, j.wx, j.wy, j.wz, j.frame,
               (int)(t % (unsigned)j.tx) * kFrameTile, (int)(r % (unsigned)j.ty) * kFrameTile,
               r / (unsigned)j.ty, tile);
}

// record_proj_kernel over the events of every group.
template <int NB, int LPE>
__global__ __launch_bounds__(256, NB == 3 && LPE <= 4 ? 5 : 4) void group_project(GroupSet s)
{
    int k = 0;
    while (k + 1 < s.n && blockIdx.x >= s.j[k + 1].proj0)
        k++;
    const GroupJob &j = s.j[k];
    const int64_t gid = (int64_t)(blockIdx.x - j.proj0) * 256 + threadIdx.x;
    const int64_t e = gid / 64 * (64 / LPE) + (int)(gid % (64 / LPE));
    record_project<NB, LPE, true>(j.p, j.rec, e, (int)(gid % 64) / (64 / LPE), e < j.p.n);
}

// tile_scatter over the chunks of every group, the groups taking turns: a plan's
// chunks run longest first, so the last workgroups are the shortest of all.
template <int NB, bool ONE>
__global__ __launch_bounds__(256, NB == 4 ? (ONE ? 4 : 3) : (ONE ? 5 : 4)) void group_scatter(
    GroupSet s)
{
    extern __shared__ double ldsd[];
    const int n1 = s.n > 1 ? s.j[1].nchunks : 0, n2 = s.n > 2 ? s.j[2].nchunks : 0;
    const int c = (int)blockIdx.x, turns2 = c - 3 * n2;
    int k, i;
    if (turns2 < 0) {
        k = c % 3;
        i = c / 3;
    } else if (turns2 < 2 * (n1 - n2)) {
        k = turns2 % 2;
        i = n2 + turns2 / 2;
    } else {
        k = 0;
        i = c - n1 - n2;
    }
    const GroupJob &j = s.j[k];
    scatter_chunk<kBack, NB, true, ONE>(j.p, j.g, j.chunks[i], j.list, j.rec, ldsd);
}

template <int NB, bool ONE>
int launch_groups(const GroupSet &s, unsigned frames, unsigned waves, unsigned chunks, unsigned sh,
                  bool small, hipStream_t st)
{
    const dim3 block(256);
    hipLaunchKernelGGL(group_frames, dim3(frames), block, 0, st, s);
    if (small)
        hipLaunchKernelGGL((group_project<NB, 16>), dim3(waves), block, 0, st, s);
    else
        hipLaunchKernelGGL((group_project<NB, 4>), dim3(waves), block, 0, st, s);
    if (chunks)
        hipLaunchKernelGGL((group_scatter<NB, ONE>), dim3(chunks), block, sh, st, s);
    return launch_status();
}

} // namespace
} // namespace srfx

extern "C" int srfx_tor_plan_osem_groups(const srfx_tor_plan *plans, int32_t nplans,
                                         const float *image, float *frames, float *bp,
                                         uint32_t flags, void *stream)
{
    if (!plans || nplans < 1 || nplans > kMaxGroups || !image || !frames || !bp || image == bp ||
        (flags & ~SRFX_ACCUMULATE))
        return SRFX_EINVAL;
    const srfx_tor_plan_s *pl[kMaxGroups];
    int n = 0;
    for (int k = 0; k < nplans; k++) {
        if (!plans[k] || plans[k]->cols7)
            return SRFX_EINVAL;
        if (plans[k]->p.n > 0)
            pl[n++] = plans[k];
    }
    hipStream_t st = (hipStream_t)stream;
    if (n == 0)
        return zero_grid(bp, plans[0]->grid, flags, st);
    std::stable_sort(pl, pl + n, [](const srfx_tor_plan_s *a, const srfx_tor_plan_s *b) {
        return a->nchunks > b->nchunks;
    });
    GroupSet s{};
    s.n = n;
    unsigned sh = 0;
    int64_t most = 0;
    int one = 1;
    for (int k = 0; k < n; k++) {
        sh = std::max(sh, (unsigned)(sizeof(double) * pl[k]->g.S * pl[k]->g.Wx * pl[k]->g.Wy));
        most = std::max(most, pl[k]->p.n);
        one &= pl[k]->one;
    }
    const int box = pl[0]->p.box;
    one = (box == 3 && one && 5u * sh <= kCuLds) || (box == 4 && one && 4u * sh <= kCuLds);
    const bool small = lanes_per_event(most) == 16;
    const int lpe = small ? 16 : 4;
    int64_t fb = 0, pb = 0, cb = 0;
    float *frame = frames;
    for (int k = 0; k < n; k++) {
        GroupJob &j = s.j[k];
        j.p = pl[k]->p;
        if (j.p.box != box || j.p.full_patch || pl[k]->block != 256)
            return SRFX_EUNSUPPORTED;
        const int64_t nvox = (int64_t)j.p.gx * j.p.gy * j.p.gz;
        // the frame gathers' limits (32-bit offsets formed by 24-bit products)
        if (4 * nvox >= ((int64_t)1 << 31) || (int64_t)j.p.gx * j.p.gy >= ((int64_t)1 << 24))
            return SRFX_EUNSUPPORTED;
        const Strides w = grid_strides(pl[k]->grid);
        j.image = image;
        j.wx = w.x;
        j.wy = w.y;
        j.wz = w.z;
        j.frame = frame;
        frame += nvox;
        j.p.img = j.frame;
        j.p.img_bytes = (int)(4 * nvox);
        j.p.sx = 1;
        j.p.sy = j.p.gx;
        j.p.sz = j.p.gx * j.p.gy;
        j.p.out = bp;
        j.p.ox = (int)w.x;
        j.p.oy = (int)w.y;
        j.p.oz = (int)w.z;
        j.g = pl[k]->g;
        j.chunks = pl[k]->chunks;
        j.list = pl[k]->list;
        j.rec = pl[k]->rec;
        j.nchunks = pl[k]->nchunks;
        j.tx = (j.p.gx + kFrameTile - 1) / kFrameTile;
        j.ty = (j.p.gy + kFrameTile - 1) / kFrameTile;
        j.frame0 = (unsigned)fb;
        j.proj0 = (unsigned)pb;
        fb += (int64_t)j.tx * j.ty * j.p.gz;
        pb += blocks_for(j.p.n * lpe, 256);
        cb += j.nchunks;
    }
    if (fb > INT32_MAX || pb > INT32_MAX || cb > INT32_MAX)
        return SRFX_EUNSUPPORTED;
    const int rc = zero_grid(bp, pl[0]->grid, flags, st);
    if (rc)
        return rc;
    const auto f = (unsigned)fb, w = (unsigned)pb, c = (unsigned)cb;
    switch (box) {
    case 3:
        return one ? launch_groups<3, true>(s, f, w, c, sh, small, st)
                   : launch_groups<3, false>(s, f, w, c, sh, small, st);
    case 4:
        return one ? launch_groups<4, true>(s, f, w, c, sh, small, st)
                   : launch_groups<4, false>(s, f, w, c, sh, small, st);
    default:
        return launch_groups<0, false>(s, f, w, c, sh, small, st);
    }
}
