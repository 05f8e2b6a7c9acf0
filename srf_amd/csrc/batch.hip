// Batched TOF OSEM: many independent reconstructions (different image sizes
// and event counts) advance one subset together.
//
// At creation every (reconstruction, axis group, subset) gets a tile plan of
// its events (tile_core.h), its walk records in a locality order (locality.h)
// whatever order the events came in.  A subset step is five kernels or so on one
// stream:
//   batch_voxels   zero every reconstruction's backprojection buffer;
//   batch_frames   copy every reconstruction's image into the op frame of
//                  each of its axis groups (frame_core.h), which the
//                  projection reads (a box row of voxels shares a line);
//   batch_project  one wave per item of <= 256 events (of any reconstruction
//                  and group): walks them from their plan's walk records and
//                  writes their projections into the records' value slots;
//   batch_scatter  tiled backprojection of 1/p, one workgroup per tile chunk (of
//                  any plan): accumulates it in an FP64 LDS tile and flushes it
//                  into that reconstruction's backprojection buffer;
//   batch_voxels   x <- x * E * bp for every reconstruction.
// The projection and the scatter are one launch per box class present.  The step
// allocates nothing and issues no memset, so a caller can capture it in a HIP
// graph.
#include <algorithm>
#include <new>
#include <vector>

#include "frame_core.h"
#include "tile_core.h"

namespace srfx {

// One (reconstruction, axis group, subset): the subset's events and its plan.
struct BatchJob {
    TorParams p; // img: the reconstruction's image, out: its bp, val: proj
    TileGeom g;
    const int *list;
    const float4 *rec;
    float *proj;
};

struct EvChunk {
    int job, start, count, pad;
};

// Box classes of the batch's jobs: 0 = candidate box 3 with every event on
// the 3 x 2 box (the single-walk scatter), 1 = other box-3 jobs, 2 = box 4, 3 =
// wider tubes (the row walk).  Each class has its own work lists and kernels, so
// that a kernel holds only its class's walk (and its registers).
constexpr int kBoxClasses = 4;

inline int box_class(const TorParams &p, bool single_walk)
{
    if (p.box == 3)
        return single_walk ? 0 : 1;
    return p.box == 4 ? 2 : 3;
}

struct TileWork {
    int job, tile, start, count;
};

// One reconstruction's voxels: workgroups first, first + 1, ... of the
// elementwise kernels, kVoxBlock voxels each.
struct VoxRange {
    float *x;
    const float *e;
    float *bp;
    long long n;
    int first;
    int wide; // the three arrays are 16-byte aligned
};

namespace {

constexpr int kChunk = 256;

constexpr int kVoxBlock = 4096;

// The reconstruction of workgroup blockIdx.x.
__device__ __forceinline__ const VoxRange &find_range(const VoxRange *r, int nrec)
{
    int lo = 0, hi = nrec - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (r[mid].first <= (int)blockIdx.x)
            lo = mid;
        else
            hi = mid - 1;
    }
    return r[lo];
}

// The elementwise kernels: bound by memory, so one reconstruction per workgroup
// (the search once, in scalar registers) and 16-byte accesses, four in flight
// per thread and array.  UPDATE: x <- x * E * bp (model/recon_step.py:48-49),
// else bp <- 0.  8.9M voxels in 12 reconstructions: update 84 -> 24 us
// (143 MB), zero 31 -> 7.5, against a grid-stride loop that searched per
// voxel.
template <bool UPDATE>
__global__ __launch_bounds__(256) void batch_voxels(const VoxRange *__restrict__ r, int nrec)
{
    const VoxRange &v = find_range(r, nrec);
    const long long i0 = (long long)((int)blockIdx.x - v.first) * kVoxBlock;
    float *const x = v.x + i0, *const bp = v.bp + i0;
    const float *const e = v.e + i0;
    const int n = (int)min((long long)kVoxBlock, v.n - i0);
    if (v.wide && n == kVoxBlock) {
        constexpr int N = kVoxBlock / 1024;
        float4 fx[N], fe[N], fb[N];
        if (UPDATE) {
#pragma unroll
            for (int k = 0; k < N; k++) {
                fx[k] = reinterpret_cast<const float4 *>(x)[k * 256 + threadIdx.x];
                fe[k] = reinterpret_cast<const float4 *>(e)[k * 256 + threadIdx.x];
                fb[k] = reinterpret_cast<const float4 *>(bp)[k * 256 + threadIdx.x];
            }
        }
#pragma unroll
        for (int k = 0; k < N; k++) {
            if (UPDATE)
                reinterpret_cast<float4 *>(x)[k * 256 + threadIdx.x] =
                    make_float4((fx[k].x * fe[k].x) * fb[k].x, (fx[k].y * fe[k].y) * fb[k].y,
                                (fx[k].z * fe[k].z) * fb[k].z, (fx[k].w * fe[k].w) * fb[k].w);
            else
                reinterpret_cast<float4 *>(bp)[k * 256 + threadIdx.x] =
                    make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        return;
    }
    for (int i = threadIdx.x; i < n; i += 256) {
        if (UPDATE)
            x[i] = (x[i] * e[i]) * bp[i];
        else
            bp[i] = 0.0f;
    }
}

// Item of workgroup blockIdx.x (xcd_groups's grid): workgroup b runs on XCD
// b % 8, and each XCD takes runs of g neighbouring items, so that its L2 serves
// one part of one reconstruction's frame at a time while the XCDs stay level.
__device__ __forceinline__ int xcd_item(int g)
{
    const int x = blockIdx.x % 8, i = blockIdx.x / 8;
    return (i / g * 8 + x) * g + i % g;
}

// One wave per work item of T events (kChunk / T items per event chunk) of one
// box class (NB), walked in rounds of 64 / LPE events at LPE lanes per event.
// The hardware deals the waves out: pulling items from a counter in memory takes
// about 20 ns a pull whoever asks, 9300 items and 5120 waves that find it empty
// here.  594k events in 12 reconstructions (128 x 128 x 64), one lane per event:
// 340 us from a counter in the order the events came, 304 in locality order, 242
// dealt out by the hardware, 229 with the runs of xcd_item short enough that an
// XCD's waves share a frame's part (four lanes: 217).  The default schedule,
// LPE = 4 and T = 64 (quarter chunks), is the projection schedule of the plan
// OSEM step.  The gathers read the jobs' contiguous op frames
// (record_project<.., true>).  Five waves per SIMD for the 3 x 3 box at up to four
// lanes per event and items of up to 128 events (four lanes: 235 against 260 us at
// four waves); the other schedules measured slower at five and keep four.
template <int NB, int LPE, int T>
__global__ __launch_bounds__(64, NB == 3 && LPE <= 4 && T <= 128 ? 5 : 4) void batch_project(
    const BatchJob *__restrict__ jobs, const EvChunk *__restrict__ chunks, int nchunks, int group)
{
    constexpr int kParts = kChunk / T, kRound = 64 / LPE;
    static_assert(kChunk % T == 0 && T % kRound == 0, "items split chunks into whole rounds");
    const int q = xcd_item(group);
    if (q >= kParts * nchunks)
        return;
    const EvChunk ch = chunks[q / kParts];
    const BatchJob &job = jobs[__builtin_amdgcn_readfirstlane(ch.job)];
    float4 *rec = const_cast<float4 *>(job.rec);
    const int lane = (int)__lane_id(), sub = lane / kRound;
    for (int r = 0; r < T; r += kRound) {
        const int i = (q % kParts) * T + r + lane % kRound;
        const bool valid = i < ch.count;
        const int64_t e = (int64_t)ch.start + i;
        record_project<NB, LPE, true, false, true>(job.p, rec, e, sub, valid);
    }
}

// One workgroup per tile chunk of one box class (NB); four waves per SIMD where
// the walk fits, five for the single-walk class (ONE), as tile_scatter.
template <int NB, bool ONE = false>
__global__ __launch_bounds__(256, ONE ? 5 : (NB == 4 ? 3 : 4)) void batch_scatter(
    const BatchJob *__restrict__ jobs, const TileWork *__restrict__ work, int nwork, int group)
{
    extern __shared__ double ldsd[];
    const int c = xcd_item(group);
    if (c >= nwork)
        return;
    const TileWork w = work[c];
    const BatchJob &job = jobs[__builtin_amdgcn_readfirstlane(w.job)];
    const TileChunk ch{w.tile, w.start, w.count, 0};
    scatter_chunk<kBack, NB, true, ONE>(job.p, job.g, ch, job.list, job.rec, ldsd);
}

// One op-frame copy: the world image read with the group's op-frame strides
// into a contiguous [gz][gy][gx] buffer, tiles [first, first + tx * ty * gz)
// of the batch_frames grid.
struct FrameJob {
    const float *src;
    float *dst;
    int gx, gy, gz, tx, ty;
    int64_t sx, sy, sz;
    long long first;
};

__global__ __launch_bounds__(256) void batch_frames(const FrameJob *__restrict__ jobs, int njobs)
{
    __shared__ float tile[kFrameTile][kFrameTile + 1];
    const long long blk = blockIdx.x;
    int lo = 0, hi = njobs - 1;
    while (lo < hi) { // last job whose first tile is <= blk
        const int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].first <= blk)
            lo = mid;
        else
            hi = mid - 1;
    }
    const FrameJob &f = jobs[lo];
    const long long t = blk - f.first;
    const int bx = (int)(t % f.tx);
    const long long r = t / f.tx;
    const int by = (int)(r % f.ty);
    frame_tile(f.src, f.gx, f.gy, f.sx, f.sy, f.sz, f.dst, bx * kFrameTile, by * kFrameTile,
               r / f.ty, tile);
}

// Op frame of axis group a for a C-order (nx, ny, nz) world image, as
// physics/split_lors.py:54-85 derives it by transposing: op (x, y, z) =
// world (y, z, x) for the x group, (x, z, y) for y, (x, y, z) for z.
srfx_grid group_grid(const srfx_recon &r, int a)
{
    static const int perm[3][3] = {{1, 2, 0}, {0, 2, 1}, {0, 1, 2}};
    const int64_t st[3] = {(int64_t)r.shape[1] * r.shape[2], (int64_t)r.shape[2], 1};
    srfx_grid g;
    for (int k = 0; k < 3; k++) {
        int w = perm[a][k];
        g.shape[k] = r.shape[w];
        g.center[k] = r.center[w];
        g.size[k] = r.size[w];
        g.stride[k] = st[w];
    }
    return g;
}

// Tile of the batch's plans: 12 slices x 32 x 10 voxels, <= 2048 events per
// workgroup (the FP64 LDS tile is 30 KB: five workgroups per CU).
constexpr srfx_tile kBatchTile = {12, 32, 10, 2048, 256, 0};

} // namespace
} // namespace srfx

struct srfx_tor_batch {
    int nrec = 0, nsub = 0, njobs = 0;
    std::vector<srfx_tor_plan> plans;
    srfx::BatchJob *d_jobs = nullptr;
    // work lists per (subset, box class): index subset * kBoxClasses + class
    std::vector<srfx::EvChunk *> d_ev;
    std::vector<int> nev;
    std::vector<srfx::TileWork *> d_work;
    std::vector<int> nwork;
    srfx::VoxRange *d_vox = nullptr;
    unsigned vox_blocks = 0;
    // the block holding the op-frame copies, one per (reconstruction,
    // non-empty group)
    std::vector<float *> frames;
    srfx::FrameJob *d_frames = nullptr;
    int nframes = 0;
    long long frame_blocks = 0;
    unsigned scatter_lds = 0;
    int cus = 0;
    int proj_lanes = 4, proj_events = 64; // projection schedule (batch_project<LPE, T>)
};

using namespace srfx;

// Grid and run length of xcd_item for n items: runs of at most `room` (for the
// projection a fifth of the waves an XCD holds: 4 to 16 waves per CU measured
// 229 / 242 us, contiguous eighths 255; for the scatter one workgroup per CU, 155
// against 159 to 271).
static unsigned xcd_groups(int64_t n, int room, int &group)
{
    const int64_t k = std::max<int64_t>(1, (n + 8 * room - 1) / (8 * room));
    group = (int)std::max<int64_t>(1, (n + 8 * k - 1) / (8 * k));
    return (unsigned)(8 * k * group);
}

// Enqueue the projection of one box class with schedule (LPE, T) for a subset.
template <int NB, int LPE, int T>
static void project_class(const srfx_tor_batch *b, int c, int subset, hipStream_t st)
{
    const int w = subset * kBoxClasses + c;
    if (b->nev[w] == 0)
        return;
    int group;
    const unsigned grid = xcd_groups((int64_t)(kChunk / T) * b->nev[w], 4 * b->cus / 8, group);
    hipLaunchKernelGGL((batch_project<NB, LPE, T>), dim3(grid), dim3(64), 0, st, b->d_jobs,
                       b->d_ev[w], b->nev[w], group);
}

template <int LPE, int T>
static int project_launch(const srfx_tor_batch *b, int subset, hipStream_t st)
{
    if (subset < 0)
        return SRFX_OK;
    project_class<3, LPE, T>(b, 0, subset, st);
    project_class<3, LPE, T>(b, 1, subset, st);
    project_class<4, LPE, T>(b, 2, subset, st);
    project_class<0, LPE, T>(b, 3, subset, st);
    return SRFX_OK;
}

// Lanes per event {1, 4, 16} x events per work item {64, 128, 256}; subset < 0
// only checks the schedule.
static int project_schedule(const srfx_tor_batch *b, int lanes, int events, int subset,
                            hipStream_t st)
{
    if (lanes == 1 && events == 64)
        return project_launch<1, 64>(b, subset, st);
    if (lanes == 1 && events == 128)
        return project_launch<1, 128>(b, subset, st);
    if (lanes == 1 && events == 256)
        return project_launch<1, 256>(b, subset, st);
    if (lanes == 4 && events == 64)
        return project_launch<4, 64>(b, subset, st);
    if (lanes == 4 && events == 128)
        return project_launch<4, 128>(b, subset, st);
    if (lanes == 4 && events == 256)
        return project_launch<4, 256>(b, subset, st);
    if (lanes == 16 && events == 64)
        return project_launch<16, 64>(b, subset, st);
    if (lanes == 16 && events == 128)
        return project_launch<16, 128>(b, subset, st);
    if (lanes == 16 && events == 256)
        return project_launch<16, 256>(b, subset, st);
    return SRFX_EINVAL;
}

static void free_plan(srfx_tor_batch *b)
{
    if (!b)
        return;
    (void)hipDeviceSynchronize();
    for (srfx_tor_plan p : b->plans)
        (void)srfx_tor_plan_destroy(p);
    (void)hipFree(b->d_jobs);
    for (EvChunk *c : b->d_ev)
        (void)hipFree(c);
    for (TileWork *w : b->d_work)
        (void)hipFree(w);
    (void)hipFree(b->d_vox);
    for (float *f : b->frames)
        (void)hipFree(f);
    (void)hipFree(b->d_frames);
    delete b;
}

template <class T> static bool upload(T **dst, const std::vector<T> &v)
{
    *dst = nullptr;
    if (v.empty())
        return true;
    return hipMalloc((void **)dst, sizeof(T) * v.size()) == hipSuccess &&
           hipMemcpy(*dst, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice) == hipSuccess;
}

extern "C" int srfx_tor_batch_create(const srfx_recon *recons, int32_t nrecon,
                                     int32_t nb_subsets, srfx_tor_model m,
                                     srfx_tor_batch **out)
{
    if (!out || !recons || nrecon <= 0 || nb_subsets <= 0)
        return SRFX_EINVAL;
    *out = nullptr;
    for (int r = 0; r < nrecon; r++) {
        const srfx_recon &rc = recons[r];
        if (!rc.image || !rc.emap || !rc.bp)
            return SRFX_EINVAL;
        for (int a = 0; a < 3; a++) {
            TorParams p;
            int st = setup(p, rc.lors[a], rc.n[a], rc.ld[a], group_grid(rc, a), m.kernel_width,
                           m.geo_sigma2_flag, m.tof_bin, m.tof_sigma2);
            if (st)
                return st;
            // the frame gathers address an op frame with 32-bit byte offsets
            // and 24-bit slice products
            const srfx_grid gg = group_grid(rc, a);
            if (4 * (int64_t)rc.shape[0] * rc.shape[1] * rc.shape[2] >= ((int64_t)1 << 31) ||
                (int64_t)gg.shape[0] * gg.shape[1] >= ((int64_t)1 << 24))
                return SRFX_EUNSUPPORTED;
        }
    }
    srfx_tor_batch *b = new (std::nothrow) srfx_tor_batch;
    if (!b)
        return SRFX_ENOMEM;
    b->nrec = nrecon;
    b->nsub = nb_subsets;
    std::vector<BatchJob> jobs;
    std::vector<std::vector<EvChunk>> ev((size_t)nb_subsets * kBoxClasses);
    std::vector<std::vector<TileWork>> work((size_t)nb_subsets * kBoxClasses);
    std::vector<VoxRange> vox;
    std::vector<FrameJob> frames;
    long long vox_blocks = 0;
    int rc_status = SRFX_OK;
    // one block for the op-frame copies of every (reconstruction, non-empty
    // group), carved in the loop below
    size_t frame_floats = 0;
    for (int r = 0; r < nrecon; r++)
        for (int a = 0; a < 3; a++)
            if (recons[r].n[a] > 0)
                frame_floats += (size_t)recons[r].shape[0] * recons[r].shape[1] *
                                recons[r].shape[2];
    float *frame_next = nullptr;
    if (frame_floats > 0) {
        if (hipMalloc((void **)&frame_next, sizeof(float) * frame_floats) != hipSuccess) {
            delete b;
            return SRFX_ENOMEM;
        }
        b->frames.push_back(frame_next);
    }
    // Per subset: contiguous rows [k n / K, (k+1) n / K) of every group
    // (graph/reconstruction/worker.py:79-85), each with its own plan; the
    // plans of every (reconstruction, group) are built in one call.
    std::vector<std::vector<int64_t>> all_bounds((size_t)nrecon * 3,
                                                 std::vector<int64_t>(nb_subsets + 1));
    std::vector<SubsetRequest> requests;
    for (int r = 0; r < nrecon; r++)
        for (int a = 0; a < 3; a++) {
            const srfx_recon &rc = recons[r];
            std::vector<int64_t> &bd = all_bounds[(size_t)r * 3 + a];
            for (int k = 0; k <= nb_subsets; k++)
                bd[k] = k * rc.n[a] / nb_subsets;
            requests.push_back(SubsetRequest{rc.lors[a], rc.n[a], rc.ld[a], group_grid(rc, a),
                                             kBatchTile, nb_subsets, bd.data(), true});
        }
    std::vector<srfx_tor_plan> all_plans(requests.size() * nb_subsets, nullptr);
    rc_status = plan_create_subsets_many(requests.data(), (int)requests.size(), 10, m,
                                         all_plans.data(), nullptr);
    if (rc_status) {
        free_plan(b);
        return rc_status;
    }
    // the batch owns every plan from here (free_plan), the empty ones too:
    // they hold no device memory of their own, and destroying them here would
    // synchronise the device once each
    b->plans = all_plans;
    for (int r = 0; r < nrecon && !rc_status; r++) {
        const srfx_recon &rc = recons[r];
        for (int a = 0; a < 3 && !rc_status; a++) {
            const int64_t n = rc.n[a];
            // the group's op-frame copy of the image, read by its projections
            float *frame = nullptr;
            const srfx_grid gg = group_grid(rc, a);
            if (n > 0) {
                const size_t nv = (size_t)rc.shape[0] * rc.shape[1] * rc.shape[2];
                frame = frame_next;
                frame_next += nv;
                FrameJob f;
                f.src = rc.image;
                f.dst = frame;
                f.gx = gg.shape[0];
                f.gy = gg.shape[1];
                f.gz = gg.shape[2];
                f.tx = (f.gx + kFrameTile - 1) / kFrameTile;
                f.ty = (f.gy + kFrameTile - 1) / kFrameTile;
                f.sx = gg.stride[0];
                f.sy = gg.stride[1];
                f.sz = gg.stride[2];
                f.first = b->frame_blocks;
                b->frame_blocks += (long long)f.tx * f.ty * f.gz;
                frames.push_back(f);
            }
            // the group's subset plans
            const std::vector<int64_t> &bounds = all_bounds[(size_t)r * 3 + a];
            const srfx_tor_plan *sub = all_plans.data() + ((size_t)r * 3 + a) * nb_subsets;
            for (int k = 0; k < nb_subsets; k++) {
                const int64_t lo = bounds[k], hi = bounds[k + 1];
                srfx_tor_plan plan = sub[k];
                if (hi <= lo)
                    continue;
                BatchJob job;
                job.p = plan->p;
                job.p.img = frame; // contiguous op frame, read by the frame gathers
                job.p.sx = 1;
                job.p.sy = gg.shape[0];
                job.p.sz = gg.shape[0] * gg.shape[1];
                job.p.img_bytes = (int)(4 * (int64_t)job.p.sz * gg.shape[2]);
                const int bc = box_class(job.p, plan->one != 0);
                job.p.out = rc.bp;
                job.p.val = plan->proj;
                job.g = plan->g;
                job.list = plan->list;
                job.rec = plan->rec;
                job.proj = plan->proj;
                const int j = (int)jobs.size();
                jobs.push_back(job);
                for (int64_t s = 0; s < hi - lo; s += kChunk)
                    ev[(size_t)k * kBoxClasses + bc].push_back(
                        EvChunk{j, (int)s, (int)std::min<int64_t>(kChunk, hi - lo - s), 0});
                // the plan's chunk table, kept on the host by its build
                const std::vector<TileChunk> &ch = plan->hchunks;
                if ((int)ch.size() != plan->nchunks) {
                    rc_status = SRFX_ELAUNCH;
                    break;
                }
                for (const TileChunk &c : ch)
                    work[(size_t)k * kBoxClasses + bc].push_back(
                        TileWork{j, c.tile, c.start, c.count});
            }
        }
        long long nv = (long long)rc.shape[0] * rc.shape[1] * rc.shape[2];
        const uintptr_t at = (uintptr_t)rc.image | (uintptr_t)rc.emap | (uintptr_t)rc.bp;
        vox.push_back(VoxRange{rc.image, rc.emap, rc.bp, nv, (int)vox_blocks, at % 16 == 0});
        vox_blocks += (nv + kVoxBlock - 1) / kVoxBlock;
    }
    if (rc_status) {
        free_plan(b);
        return rc_status;
    }
    b->njobs = (int)jobs.size();
    b->vox_blocks = (unsigned)vox_blocks;
    b->nframes = (int)frames.size();
    bool ok = upload(&b->d_jobs, jobs) && upload(&b->d_vox, vox) && upload(&b->d_frames, frames);
    for (size_t w = 0; ok && w < ev.size(); w++) {
        EvChunk *e = nullptr;
        TileWork *t = nullptr;
        // The longest chunks first, so that the last workgroups to run are short
        // (5100 chunks on 1280 places: 180 us in plan order, 155 so); by 256 events,
        // to keep neighbours together.
        std::stable_sort(work[w].begin(), work[w].end(), [](const TileWork &a, const TileWork &b) {
            return a.count / 256 > b.count / 256;
        });
        ok = upload(&e, ev[w]) && upload(&t, work[w]);
        b->d_ev.push_back(e);
        b->nev.push_back((int)ev[w].size());
        b->d_work.push_back(t);
        b->nwork.push_back((int)work[w].size());
    }
    b->scatter_lds = (unsigned)(sizeof(double) * kBatchTile.slices * kBatchTile.wx * kBatchTile.wy);
    int dev = 0, cus = 0;
    ok = ok && hipGetDevice(&dev) == hipSuccess &&
         hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess;
    if (!ok) {
        free_plan(b);
        return SRFX_ELAUNCH;
    }
    b->cus = cus;
    *out = b;
    return SRFX_OK;
}

extern "C" int srfx_tor_batch_subset(srfx_tor_batch *b, int32_t subset, void *stream)
{
    if (!b || subset < 0 || subset >= b->nsub)
        return SRFX_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(batch_voxels<false>, dim3(b->vox_blocks), dim3(256), 0, st, b->d_vox,
                       b->nrec);
    if (b->nframes > 0)
        hipLaunchKernelGGL(batch_frames, dim3((unsigned)b->frame_blocks), dim3(256), 0, st,
                           b->d_frames, b->nframes);
    project_schedule(b, b->proj_lanes, b->proj_events, subset, st);
    for (int c = 0; c < kBoxClasses; c++) {
        const int w = subset * kBoxClasses + c;
        if (b->nwork[w] == 0)
            continue;
        int group;
        const dim3 grid(xcd_groups(b->nwork[w], b->cus / 8, group)), block(256);
        auto *kernel = c == 0   ? batch_scatter<3, true>
                       : c == 1 ? batch_scatter<3>
                       : c == 2 ? batch_scatter<4>
                                : batch_scatter<0>;
        hipLaunchKernelGGL(kernel, grid, block, b->scatter_lds, st, b->d_jobs, b->d_work[w],
                           b->nwork[w], group);
    }
    hipLaunchKernelGGL(batch_voxels<true>, dim3(b->vox_blocks), dim3(256), 0, st, b->d_vox,
                       b->nrec);
    return launch_status();
}

extern "C" int srfx_tor_batch_set_schedule(srfx_tor_batch *b, int32_t lanes_per_event,
                                           int32_t events_per_item)
{
    if (!b)
        return SRFX_EINVAL;
    // the grid changes only when the schedule exists and its occupancy query succeeds
    const int rc = project_schedule(b, lanes_per_event, events_per_item, -1, nullptr);
    if (rc == SRFX_OK) {
        b->proj_lanes = lanes_per_event;
        b->proj_events = events_per_item;
    }
    return rc;
}

extern "C" int srfx_tor_batch_destroy(srfx_tor_batch *b)
{
    free_plan(b);
    return SRFX_OK;
}
