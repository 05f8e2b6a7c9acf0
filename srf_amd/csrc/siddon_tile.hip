// Tiled Siddon backprojection: plans over a fixed LOR set (srfx_siddon_plan_*)
// and the binned form of the untiled scatters (siddon_binned.h).
//
// The untiled scatter (siddon.hip) adds every segment of every ray to the
// image with its own global FP32 atomic.  Those atomics land on scattered
// cache lines and bound the op: 100k LORs of 171 segments take 0.52 ms.  Here
// the rays are listed by the image tiles they cross; a workgroup takes up to
// `chunk` listings of one tile, accumulates them in an FP64 copy of the tile in
// LDS and flushes the tile once with coalesced atomics.
//
// A listing is the ray's index alone.  The ray's record holds its crossings
// (n + k t per axis, siddon_core.h), so the part of the ray inside a tile
// follows from the tile's faces: it enters at the last of the crossings into
// the tile and leaves at the first of those out of it.  Neighbouring tiles form
// a shared face's crossing with the same operation, so the parts join without
// gap or overlap, and the tiles of a ray are found by stepping from face to
// face (11 steps for 171 segments).
//
// A chunk's listings are ordered by the slabs they walk in the tile, longest
// first: a wave's 64 walks then end together, and the lanes hold rays from
// anywhere in the chunk, whose LDS atomics rarely meet on a voxel as those of
// neighbouring rays do.
//
// Layout.  List entry: ray index in bits 0..26, the slab count (up to 31) above
// (sets of 2^27 rays and more keep plain indices and the fill order).  Ray
// record (5 float4): [n0 n1] [n2 t0] [t1 t2] [tend t_tof] (FP64
// pairs) [weight, x | y << 16, z, steps].
#include <algorithm>
#include <atomic>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "chunk_sort.h"
#include "siddon_binned.h"

namespace srfx {
namespace {

constexpr int kRayF4 = 5;
// LDS tile: FP64, at most 64 KB.
constexpr int kMaxTileVox = 8192;

constexpr int kRayBits = 27;

// Listings per workgroup where the caller names no chunk: as few as let every
// workgroup of the scatter run at once (`slots`), so that a small set fills the
// chip, and no more than 2048, beyond which the flushes no longer count; no fewer
// than `least`.  A binned call's least is 256: projection and backprojection of 100k
// TOF LORs (128 x 128 x 64) take 204 us, 220 with 1024, and are 8.4e-8 from 64 bits
// (1.7e-7 with an atomic a segment).  A plan's least is 1024: every flush adds an FP32 rounding to
// the image, and an OSEM pass of 500k LORs (same image, four subsets) is
// 1.235e-7 from 64 bits with it, 1.313e-7 with 2048 alone and 1.338e-7 with 256;
// 519, 632 and 530 us.  A pass of 30k, 80k and 160k LORs takes 153, 213 and 324 us
// with 256 and 169, 225 and 285 with 1024.
constexpr int kChunkMin = 256, kPlanChunkMin = 1024, kChunkMax = 2048;

__host__ __device__ inline int auto_chunk(long long listings, int slots, int least)
{
    const long long c = (listings / slots + kChunkMin - 1) / kChunkMin * kChunkMin;
    return (int)(c < least ? least : (c > kChunkMax ? kChunkMax : c));
}

struct SidTileGeom {
    int t[3];   // tile extent per image axis (voxels)
    int nt[3];  // tiles per axis
    int ls[3];  // LDS stride of each axis inside a tile
    int ord[3]; // axes from the fastest LDS axis to the slowest
    int tvox;   // voxels per tile
    int keyed;  // list entries carry slab counts (kRayBits)
};

struct SidChunk {
    int64_t start;
    int tile, count;
};

__device__ __forceinline__ float4 pack_d2(double a, double b)
{
    return make_float4(__int_as_float(__double2loint(a)), __int_as_float(__double2hiint(a)),
                       __int_as_float(__double2loint(b)), __int_as_float(__double2hiint(b)));
}

__device__ __forceinline__ void unpack_d2(const float4 &f, double &a, double &b)
{
    a = __hiloint2double(__float_as_int(f.y), __float_as_int(f.x));
    b = __hiloint2double(__float_as_int(f.w), __float_as_int(f.z));
}

__device__ __forceinline__ void pack_ray(const SidRay &r, float4 *o)
{
    o[0] = pack_d2(r.n[0], r.n[1]);
    o[1] = pack_d2(r.n[2], r.t[0]);
    o[2] = pack_d2(r.t[1], r.t[2]);
    o[3] = pack_d2(r.tend, r.t_tof);
    o[4] = make_float4(r.weight, __int_as_float(r.pos[0] | (r.pos[1] << 16)),
                       __int_as_float(r.pos[2]),
                       __int_as_float((r.step[0] + 1) | ((r.step[1] + 1) << 2) |
                                      ((r.step[2] + 1) << 4)));
}

__device__ __forceinline__ void unpack_ray(const float4 *__restrict__ o, SidRay &r)
{
    const float4 a = o[0], b = o[1], c = o[2], d = o[3], e = o[4];
    unpack_d2(a, r.n[0], r.n[1]);
    unpack_d2(b, r.n[2], r.t[0]);
    unpack_d2(c, r.t[1], r.t[2]);
    unpack_d2(d, r.tend, r.t_tof);
    r.weight = e.x;
    const int pxy = __float_as_int(e.y), steps = __float_as_int(e.w);
    r.pos[0] = pxy & 0xffff;
    r.pos[1] = (int)((unsigned)pxy >> 16);
    r.pos[2] = __float_as_int(e.z);
    r.step[0] = (steps & 3) - 1;
    r.step[1] = ((steps >> 2) & 3) - 1;
    r.step[2] = ((steps >> 4) & 3) - 1;
}

// A ray that misses the image.
__device__ __forceinline__ void no_ray(SidRay &r)
{
#pragma unroll
    for (int c = 0; c < 3; c++) {
        r.n[c] = r.t[c] = 0.0;
        r.pos[c] = r.step[c] = 0;
    }
    r.tend = -1.0;
    r.t_tof = 0.0;
    r.weight = 0.0f;
}

// Crossing of axis c by which a ray leaves the tile that holds voxel `tile * t`
// .. `tile * t + t - 1` of the axis.
__device__ __forceinline__ int leave_crossing(int pos, int step, int tile, int t)
{
    return step > 0 ? tile * t + t - 1 - pos : (step < 0 ? pos - tile * t : 0);
}

// Calls f(tile, length along the ray inside it) for every image tile the ray
// crosses with a length (and, with TOF, inside its window), face by face.
template <bool TOF, typename F>
__device__ __forceinline__ void for_each_tile(const SidParams &p, const SidTileGeom &g,
                                              const SidRay &r, F &&f)
{
    if (!(r.tend > 0.0))
        return;
    int c0 = r.pos[0] / g.t[0], c1 = r.pos[1] / g.t[1], c2 = r.pos[2] / g.t[2];
    int k0 = leave_crossing(r.pos[0], r.step[0], c0, g.t[0]);
    int k1 = leave_crossing(r.pos[1], r.step[1], c1, g.t[1]);
    int k2 = leave_crossing(r.pos[2], r.step[2], c2, g.t[2]);
    double f0 = cross_time(r.n[0], r.t[0], (double)k0);
    double f1 = cross_time(r.n[1], r.t[1], (double)k1);
    double f2 = cross_time(r.n[2], r.t[2], (double)k2);
    double wa = 0.0, wb = 0.0;
    if (TOF)
        tof_window(p, r, fmin(r.t[0], fmin(r.t[1], r.t[2])), wa, wb);
    double T = 0.0;
    for (;;) {
        const int i = f0 <= f1 ? (f0 <= f2 ? 0 : 2) : (f1 <= f2 ? 1 : 2);
        const double Te = i == 0 ? f0 : (i == 1 ? f1 : f2);
        const double To = fmin(Te, r.tend);
        if (T < To && (!TOF || (T < wb && To > wa)))
            f((c0 * g.nt[1] + c1) * g.nt[2] + c2, To - T);
        if (!(Te < r.tend))
            return; // the ray leaves the image inside this tile
        T = Te;
        if (i == 0) {
            c0 += r.step[0];
            k0 += g.t[0];
            f0 = cross_time(r.n[0], r.t[0], (double)k0);
        } else if (i == 1) {
            c1 += r.step[1];
            k1 += g.t[1];
            f1 = cross_time(r.n[1], r.t[1], (double)k1);
        } else {
            c2 += r.step[2];
            k2 += g.t[2];
            f2 = cross_time(r.n[2], r.t[2], (double)k2);
        }
    }
}

// The plan set's two passes over the rays of all its plans (plan k holds
// rays bounds[k] .. bounds[k + 1] - 1), one lane per ray.  Count pass (FILL
// false): writes the ray records and counts the listings of each (plan, tile)
// counter.  Fill pass: writes each listing, the ray's index inside its plan, at
// its counter's cursor (which starts at the counter's offset).  LDS: the
// workgroup first counts its listings in LDS counters, so that the global
// counters take one atomic per (workgroup, counter) instead of one per listing;
// the fill pass then reserves one range per (workgroup, counter) and steps
// through its rays' tiles a second time to write into those ranges.  Needs 12
// bytes of LDS per counter.
template <int MODE, bool FILL, bool TOF, bool LDS>
__global__ __launch_bounds__(256) void sid_plan_pass(SidParams p, SidTileGeom g,
                                                     unsigned long long *tiles, float4 *rays,
                                                     int *list, unsigned long long nlist,
                                                     const int64_t *__restrict__ bounds,
                                                     int nplans, int ntiles)
{
    extern __shared__ unsigned lcnt[];
    const int ncnt = nplans * ntiles;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = e < p.n && e >= bounds[0] && e < bounds[nplans];
    // the plan of ray e: the last k with bounds[k] <= e
    int lo = 0;
    if (valid) {
        int hi = nplans - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (bounds[mid] <= e)
                lo = mid;
            else
                hi = mid - 1;
        }
    }
    const int c0 = lo * ntiles;
    const int el = valid ? (int)(e - bounds[lo]) : 0;
    SidRay r;
    r.tend = -1.0;
    if (valid) {
        if (FILL) {
            unpack_ray(rays + kRayF4 * e, r);
        } else {
            Walk w;
            setup_walk<MODE>(p, e, w);
            if (w.ok)
                make_ray(w, r);
            else
                no_ray(r);
            pack_ray(r, rays + kRayF4 * e);
        }
    }
    const float rtd = FILL && g.keyed && r.tend > 0.0
                          ? 1.0f / (float)fmin(r.t[0], fmin(r.t[1], r.t[2]))
                          : 0.0f;
    auto entry = [&](double len) {
        return g.keyed ? el | (int)((unsigned)min((int)((float)len * rtd) + 1, 31) << kRayBits)
                       : el;
    };
    if constexpr (!LDS) {
        for_each_tile<TOF>(p, g, r, [&](int tile, double len) {
            const unsigned long long slot = atomicAdd(tiles + c0 + tile, 1ull);
            if (FILL && slot < nlist) // (never past nlist: the passes find the same tiles)
                list[slot] = entry(len);
        });
    } else {
        for (int i = threadIdx.x; i < ncnt; i += blockDim.x)
            lcnt[i] = 0u;
        __syncthreads();
        for_each_tile<TOF>(p, g, r, [&](int tile, double) { atomicAdd(lcnt + c0 + tile, 1u); });
        __syncthreads();
        if (!FILL) {
            for (int i = threadIdx.x; i < ncnt; i += blockDim.x)
                if (lcnt[i])
                    atomicAdd(tiles + i, (unsigned long long)lcnt[i]);
            return;
        }
        auto *lbase = reinterpret_cast<unsigned long long *>(lcnt + ((ncnt + 1) & ~1));
        for (int i = threadIdx.x; i < ncnt; i += blockDim.x) {
            const unsigned c = lcnt[i];
            lbase[i] = c ? atomicAdd(tiles + i, (unsigned long long)c) : 0ull;
            lcnt[i] = 0u;
        }
        __syncthreads();
        for_each_tile<TOF>(p, g, r, [&](int tile, double len) {
            const unsigned long long slot = lbase[c0 + tile] + atomicAdd(lcnt + c0 + tile, 1u);
            if (slot < nlist)
                list[slot] = entry(len);
        });
    }
}

// Scatter of one chunk: zero the FP64 LDS tile, walk the part of every listed
// ray inside the tile into it (scale from vals: 1 / v for v > 0 as
// BackRayTracing's callers, siddon.cu.cc:363-371, or c / v with per-LOR counts
// c; ADJ: g itself, rays of g = 0 skipped), then add the tile's non-zero voxels
// to the image with one atomic each, consecutive lanes on consecutive voxels of
// the image's fastest axis.  vals (vperm) and counts (cperm) are read in the
// plan's LOR order or, through a permutation, in the caller's.
template <bool TOF, bool ADJ>
__device__ __forceinline__ void sid_scatter_chunk(const SidParams &p, const SidTileGeom &g,
                                                  int tile, const int *__restrict__ list,
                                                  int count, const float4 *__restrict__ rays,
                                                  const float *__restrict__ vals,
                                                  const int *__restrict__ vperm,
                                                  const float *__restrict__ counts,
                                                  const int *__restrict__ cperm, double *acc)
{
    for (int v = threadIdx.x; v < g.tvox; v += blockDim.x)
        acc[v] = 0.0;
    const int kz = tile % g.nt[2];
    const int ky = (tile / g.nt[2]) % g.nt[1];
    const int kx = tile / (g.nt[2] * g.nt[1]);
    const int org[3] = {kx * g.t[0], ky * g.t[1], kz * g.t[2]};
    __syncthreads();
    for (int j = threadIdx.x; j < count; j += blockDim.x) {
        const int e = g.keyed ? list[j] & ((1 << kRayBits) - 1) : list[j];
        const float v = vals[vperm ? vperm[e] : e];
        float scale;
        if (ADJ) {
            if (v == 0.0f)
                continue;
            scale = v;
        } else {
            if (!(v > 0.0f))
                continue;
            scale = counts ? counts[cperm ? cperm[e] : e] / v : 1.0f / v;
        }
        SidRay r;
        unpack_ray(rays + kRayF4 * (int64_t)e, r);
        // crossings before the tile (lo) and the one leaving it (hi), per axis
        int lo[3], hi[3];
        double ta = 0.0, tb = r.tend;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int x0 = org[c], x1 = org[c] + g.t[c] - 1;
            const int l = r.step[c] > 0 ? x0 - r.pos[c] : (r.step[c] < 0 ? r.pos[c] - x1 : 0);
            hi[c] = r.step[c] > 0 ? x1 - r.pos[c] : (r.step[c] < 0 ? r.pos[c] - x0 : 0);
            lo[c] = max(l, 0);
            if (l > 0)
                ta = fmax(ta, cross_time(r.n[c], r.t[c], (double)(l - 1)));
            tb = fmin(tb, cross_time(r.n[c], r.t[c], (double)hi[c]));
        }
        const SidAxes a = ray_axes(r);
        int ld, ly, lz, hd, hy, hz;
        by_axes(a, lo, ld, ly, lz);
        by_axes(a, hi, hd, hy, hz);
        const int kd = crossings(a.nd, a.td, ta, ld, hd);
        const int qy = crossings(a.ny, a.ty, ta, ly, hy);
        const int qz = crossings(a.nz, a.tz, ta, lz, hz);
        const int base = (r.pos[0] - org[0]) * g.ls[0] + (r.pos[1] - org[1]) * g.ls[1] +
                         (r.pos[2] - org[2]) * g.ls[2];
        const double w = (double)span_factor<TOF>(p, r) * (double)scale;
        walk_span<TOF>(p, r, a, SpanIndex(r, a, g.ls, base, kd, qy, qz), kd, qy, qz, ta, tb,
                       [&](int o0, float g0, int o1, float g1, int o2, float g2) {
                           if (g0 > 0.0f)
                               atomicAdd(acc + o0, (double)g0 * w);
                           if (g1 > 0.0f)
                               atomicAdd(acc + o1, (double)g1 * w);
                           if (g2 > 0.0f)
                               atomicAdd(acc + o2, (double)g2 * w);
                       });
    }
    __syncthreads();
    // voxel v of the tile = (f, m, s) along the axes from the fastest, each
    // with its first voxel, its voxel count inside the image and its stride
    auto axis = [&](int k, const int (&v)[3]) { return k == 0 ? v[0] : (k == 1 ? v[1] : v[2]); };
    const int in[3] = {p.g[0] - org[0], p.g[1] - org[1], p.g[2] - org[2]};
    const int tf = axis(g.ord[0], g.t), tm = axis(g.ord[1], g.t);
    const int nf = axis(g.ord[0], in), nm = axis(g.ord[1], in), ns = axis(g.ord[2], in);
    const int of = axis(g.ord[0], p.o), om = axis(g.ord[1], p.o), os = axis(g.ord[2], p.o);
    float *const base = p.out + (org[0] * p.o[0] + org[1] * p.o[1] + org[2] * p.o[2]);
    for (int v = threadIdx.x; v < g.tvox; v += blockDim.x) {
        const double sum = acc[v];
        if (sum == 0.0)
            continue;
        const int f = v % tf, r = v / tf, m = r % tm, s = r / tm;
        // a non-zero voxel lies inside the image (the rays stay inside it)
        if (f < nf && m < nm && s < ns)
            unsafeAtomicAdd(base + f * of + m * om + s * os, (float)sum);
    }
}

// One workgroup per chunk of a plan.
template <bool TOF, bool ADJ>
__global__ __launch_bounds__(256) void sid_tile_scatter(SidParams p, SidTileGeom g,
                                                        const SidChunk *__restrict__ chunks,
                                                        const int *__restrict__ list,
                                                        const float4 *__restrict__ rays,
                                                        const float *__restrict__ vals,
                                                        const int *__restrict__ vperm,
                                                        const float *__restrict__ counts,
                                                        const int *__restrict__ cperm)
{
    extern __shared__ double acc[];
    const SidChunk ch = chunks[blockIdx.x];
    sid_scatter_chunk<TOF, ADJ>(p, g, ch.tile, list + ch.start, ch.count, rays, vals, vperm,
                                counts, cperm, acc);
}

// The projection of the rays of a record array, L lanes per ray: the walk and
// the sums of siddon_kernel<kProj>, without its ray set-up.
template <bool TOF, int L>
__global__ __launch_bounds__(256) void sid_record_project(SidParams p,
                                                          const float4 *__restrict__ rays,
                                                          float *__restrict__ out)
{
    constexpr int R = 256 / L; // rays of the workgroup (ray_sum)
    const int64_t e = (int64_t)blockIdx.x * R + (int)threadIdx.x % R;
    const int sub = (int)threadIdx.x / R;
    float part = 0.0f;
    if (e < p.n) {
        SidRay r;
        unpack_ray(rays + kRayF4 * e, r);
        if (r.tend > 0.0)
            part = gather_ray<TOF, L>(p, r, sub);
    }
    const float pv = ray_sum<L>(part);
    if (e < p.n && sub == 0)
        out[e] = pv;
}

template <bool TOF>
int launch_record_project(const SidParams &p, const float4 *rays, float *out, hipStream_t st)
{
    const int L = lanes_per_ray(p.n);
    const dim3 grid(blocks_for(p.n * L, 256)), block(256);
    if (L == 16)
        hipLaunchKernelGGL((sid_record_project<TOF, 16>), grid, block, 0, st, p, rays, out);
    else if (L == 4)
        hipLaunchKernelGGL((sid_record_project<TOF, 4>), grid, block, 0, st, p, rays, out);
    else
        hipLaunchKernelGGL((sid_record_project<TOF, 1>), grid, block, 0, st, p, rays, out);
    return launch_status();
}

int record_project(const SidParams &p, const float4 *rays, float *out, hipStream_t st)
{
    return p.use_tof ? launch_record_project<true>(p, rays, out, st)
                     : launch_record_project<false>(p, rays, out, st);
}

// ------------------------------------------------------------------ binned ---

constexpr int64_t kBinPiece = 1 << 19;
constexpr int kScanThreads = 1024;

struct SidBinState {
    int nchunks;
    unsigned next;
};

struct SidBins {
    SidBinState *state;
    int64_t *bounds; // [2]
    unsigned long long *cnt; // listings per tile, then cursors
    TileSpan *chunks;
    int *list;
    float4 *rays;
    float *proj;
};

__global__ __launch_bounds__(256) void sid_bin_init(SidBins b, int nt, int64_t n)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    for (int k = i; k < nt; k += (int)(gridDim.x * blockDim.x))
        b.cnt[k] = 0ull;
    if (i == 0) {
        *b.state = SidBinState{};
        b.bounds[0] = 0;
        b.bounds[1] = n;
    }
}

// Cursors and chunks of every tile, one workgroup: a prefix sum of (listings,
// chunks) over 1024 tiles a round.
__global__ __launch_bounds__(kScanThreads) void sid_bin_scan(SidBins b, int nt, int slots)
{
    long long carry = 0, sum = 0; // listings | chunks << 40
    for (int q = threadIdx.x; q < nt; q += kScanThreads)
        sum += (long long)b.cnt[q];
    long long listings;
    (void)block_scan<kScanThreads>(sum, listings);
    const int chunk = auto_chunk(listings, slots, kChunkMin);
    for (int q0 = 0; q0 < nt; q0 += kScanThreads) {
        const int q = q0 + (int)threadIdx.x;
        const int c = q < nt ? (int)b.cnt[q] : 0;
        const int nch = (c + chunk - 1) / chunk;
        long long total;
        const long long ex =
            carry + block_scan<kScanThreads>((long long)c | ((long long)nch << 40), total);
        if (q < nt) {
            const int o = (int)(ex & ((1ll << 40) - 1)), ch = (int)(ex >> 40);
            b.cnt[q] = (unsigned long long)o;
            for (int k = 0; k < nch; k++)
                b.chunks[ch + k] = TileSpan{q, o + k * chunk, min(chunk, c - k * chunk)};
        }
        carry += total;
    }
    if (threadIdx.x == 0)
        b.state->nchunks = (int)(carry >> 40);
}

__device__ __forceinline__ void sort_listings(int *list, int count, int *sh)
{
    chunk_sort(list, count, sh, [](int ent) { return (int)((unsigned)ent >> kRayBits); });
}

__global__ __launch_bounds__(256) void sid_bin_sort(SidBins b)
{
    extern __shared__ int sh[];
    const int n = b.state->nchunks;
    for (int c = blockIdx.x; c < n; c += gridDim.x)
        sort_listings(b.list + b.chunks[c].start, b.chunks[c].count, sh);
}

// The chunks of a plan set: chunk c of the table belongs to the last plan k
// with chunk0[k] <= c, whose listings start at run0[k].
__global__ __launch_bounds__(256) void sid_sort_chunks(const SidChunk *__restrict__ chunks,
                                                       const int64_t *__restrict__ chunk0,
                                                       const int64_t *__restrict__ run0,
                                                       int nplans, int *list)
{
    extern __shared__ int sh[];
    int lo = 0, hi = nplans - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (chunk0[mid] <= (int64_t)blockIdx.x)
            lo = mid;
        else
            hi = mid - 1;
    }
    const SidChunk ch = chunks[blockIdx.x];
    sort_listings(list + run0[lo] + ch.start, ch.count, sh);
}

template <bool TOF, bool ADJ>
__global__ __launch_bounds__(256) void sid_bin_scatter(SidParams p, SidTileGeom g, SidBins b,
                                                       const float *__restrict__ vals)
{
    extern __shared__ double acc[];
    const int n = b.state->nchunks;
    for (;;) {
        const int c = next_item(&b.state->next);
        if (c >= n)
            break;
        const TileSpan ch = b.chunks[c];
        sid_scatter_chunk<TOF, ADJ>(p, g, ch.tile, b.list + ch.start, ch.count, b.rays, vals,
                                    nullptr, nullptr, nullptr, acc);
        __syncthreads(); // the flush reads the tile the next chunk clears
    }
}

// Sort key of a LOR for the sorted LOR stream: transaxial direction (8
// bits), tilt (6 bits), signed transaxial distance from the image axis (8
// bits), axial midpoint (10 bits), so that consecutive LORs run nearly
// parallel through neighbouring voxels.  The plan index rides above them, so
// each plan's LORs stay in its own range.  Any order gives the same results
// up to summation order; the key only buys locality.
__global__ __launch_bounds__(256) void sid_sort_key(SidParams p, const int64_t *__restrict__ bounds,
                                                    int nplans, unsigned long long *keys,
                                                    int *idx)
{
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t e = bounds[0] + j;
    if (e >= bounds[nplans])
        return;
    int lo = 0, hi = nplans - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (bounds[mid] <= e)
            lo = mid;
        else
            hi = mid - 1;
    }
    const float *L = p.lors;
    const int64_t ld = p.ld;
    const float x1 = L[e], y1 = L[ld + e], z1 = L[2 * ld + e];
    float dx = L[3 * ld + e] - x1, dy = L[4 * ld + e] - y1, dz = L[5 * ld + e] - z1;
    if (dx < 0.0f || (dx == 0.0f && dy < 0.0f)) {
        dx = -dx;
        dy = -dy;
        dz = -dz;
    }
    const float lxy = sqrtf(dx * dx + dy * dy);
    const float pi = 3.14159265f;
    const float fphi = lxy > 0.0f ? atan2f(dy, dx) / pi + 0.5f : 0.5f;
    const float fth = lxy > 0.0f ? atanf(dz / lxy) / pi + 0.5f : 1.0f;
    const float rad = 0.5f * sqrtf(p.size[0] * p.size[0] + p.size[1] * p.size[1]);
    const float s = lxy > 0.0f ? ((x1 - p.center[0]) * dy - (y1 - p.center[1]) * dx) / lxy : 0.0f;
    const float fs = s / (2.0f * rad) + 0.5f;
    const float fz = (0.5f * (z1 + L[5 * ld + e]) - p.center[2]) / p.size[2] + 0.5f;
    auto q = [](float f, int bits) {
        const float m = (float)(1 << bits);
        return (unsigned)fminf(fmaxf(f * m, 0.0f), m - 1.0f);
    };
    const unsigned key = (q(fphi, 8) << 24) | (q(fth, 6) << 18) | (q(fs, 8) << 10) | q(fz, 10);
    keys[j] = ((unsigned long long)lo << 32) | key;
    idx[j] = (int)j;
}

// The sorted LOR copy (7 columns, leading dimension n, LOR bounds[0] + j in
// sorted position j) and, for each sorted LOR, its index inside its plan in
// the caller's order.
__global__ __launch_bounds__(256) void sid_sort_gather(SidParams p, const int64_t *__restrict__ bounds,
                                                       int nplans,
                                                       const unsigned long long *__restrict__ keys,
                                                       const int *__restrict__ idx, float *slors,
                                                       int *perm)
{
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t e = bounds[0] + j;
    if (e >= bounds[nplans])
        return;
    const int64_t src = bounds[0] + idx[j];
    const int k = (int)(keys[j] >> 32);
#pragma unroll
    for (int c = 0; c < 7; c++)
        slors[c * p.n + e] = p.lors[c * p.ld + src];
    perm[e] = (int)(src - bounds[k]);
}

// out[perm[e]] = in[e]: a plan's buffer back in the caller's LOR order.
__global__ __launch_bounds__(256) void sid_unsort(const float *__restrict__ in,
                                                  const int *__restrict__ perm, int64_t n,
                                                  float *out)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n)
        out[perm[e]] = in[e];
}

} // namespace
} // namespace srfx

using namespace srfx;

struct srfx_siddon_plan_s {
    // device blocks shared by the plans of one set, freed with the last plan
    struct Arena {
        void *mem[3];
        std::atomic<int> refs;
    };
    SidParams p{};
    srfx_grid grid{};
    SidTileGeom g{};
    int nchunks = 0, block = 256;
    int64_t nruns = 0; // (LOR, tile) listings
    float4 *rays = nullptr;
    int *list = nullptr;
    SidChunk *chunks = nullptr;
    float *proj = nullptr;
    int *perm = nullptr; // sorted plans: plan order -> caller order
    Arena *arena = nullptr;
};

namespace {

void plan_release(srfx_siddon_plan_s *pl)
{
    if (pl->arena && pl->arena->refs.fetch_sub(1) == 1) {
        for (void *m : pl->arena->mem)
            (void)hipFree(m);
        delete pl->arena;
    }
    delete pl;
}

// LDS bytes per (plan, tile) counter of the LDS plan passes, and the most
// counters they take (64 KB of LDS).
constexpr int kLdsCounterBytes = 12;
constexpr int kMaxLdsCounters = 65536 / kLdsCounterBytes - 1;

template <int MODE, bool FILL>
void launch_pass(const SidParams &p, const SidTileGeom &g, unsigned long long *tiles,
                 float4 *rays, int *list, int64_t nlist, const int64_t *bounds, int nplans,
                 int ntiles, hipStream_t st)
{
    const dim3 grid(blocks_for(p.n, 256)), block(256);
    const int64_t ncnt = (int64_t)nplans * ntiles;
    const unsigned long long nr = (unsigned long long)nlist;
    if (ncnt <= kMaxLdsCounters) {
        const unsigned lds = (unsigned)(4 * ((ncnt + 1) & ~1) + 8 * ncnt);
        if (p.use_tof)
            hipLaunchKernelGGL((sid_plan_pass<MODE, FILL, true, true>), grid, block, lds, st, p,
                               g, tiles, rays, list, nr, bounds, nplans, ntiles);
        else
            hipLaunchKernelGGL((sid_plan_pass<MODE, FILL, false, true>), grid, block, lds, st, p,
                               g, tiles, rays, list, nr, bounds, nplans, ntiles);
    } else {
        if (p.use_tof)
            hipLaunchKernelGGL((sid_plan_pass<MODE, FILL, true, false>), grid, block, 0, st, p,
                               g, tiles, rays, list, nr, bounds, nplans, ntiles);
        else
            hipLaunchKernelGGL((sid_plan_pass<MODE, FILL, false, false>), grid, block, 0, st, p,
                               g, tiles, rays, list, nr, bounds, nplans, ntiles);
    }
}

// Scatter workgroups a CU runs at once, by its 160 KB of LDS and its waves.
int scatter_slots(unsigned lds)
{
    return std::max(1, std::min(8, (int)(160u * 1024u / std::max(lds, 1u))));
}

// Tiles of t voxels over the image of p, in LDS in the image's own axis order
// (fastest output stride first), so that a flush writes runs of consecutive
// voxels.
SidTileGeom tile_geom(const SidParams &p, const int (&t)[3])
{
    SidTileGeom g{};
    for (int c = 0; c < 3; c++) {
        g.t[c] = std::min(t[c], p.g[c]);
        g.nt[c] = (p.g[c] + g.t[c] - 1) / g.t[c];
    }
    int ord[3] = {0, 1, 2};
    std::stable_sort(ord, ord + 3, [&](int a, int b) { return p.o[a] < p.o[b]; });
    int ls = 1;
    for (int k = 0; k < 3; k++) {
        g.ord[k] = ord[k];
        g.ls[ord[k]] = ls;
        ls *= g.t[ord[k]];
    }
    g.tvox = ls;
    return g;
}

// vals in the caller's LOR order (vperm: the plan's sorted order to it) or,
// with vperm null, in the plan's order; counts (optional) likewise (cperm).
int plan_scatter(const srfx_siddon_plan_s *pl, bool adj, const float *vals, const int *vperm,
                 const float *counts, const int *cperm, float *image, uint32_t flags,
                 hipStream_t st)
{
    int rc = zero_grid(image, pl->grid, flags, st);
    if (rc || pl->nchunks == 0)
        return rc;
    SidParams p = pl->p;
    p.out = image;
    const dim3 grid(pl->nchunks), block(pl->block);
    const unsigned lds = (unsigned)(sizeof(double) * pl->g.tvox);
    if (p.use_tof) {
        if (adj)
            hipLaunchKernelGGL((sid_tile_scatter<true, true>), grid, block, lds, st, p, pl->g,
                               pl->chunks, pl->list, pl->rays, vals, vperm, counts, cperm);
        else
            hipLaunchKernelGGL((sid_tile_scatter<true, false>), grid, block, lds, st, p, pl->g,
                               pl->chunks, pl->list, pl->rays, vals, vperm, counts, cperm);
    } else {
        if (adj)
            hipLaunchKernelGGL((sid_tile_scatter<false, true>), grid, block, lds, st, p, pl->g,
                               pl->chunks, pl->list, pl->rays, vals, vperm, counts, cperm);
        else
            hipLaunchKernelGGL((sid_tile_scatter<false, false>), grid, block, lds, st, p, pl->g,
                               pl->chunks, pl->list, pl->rays, vals, vperm, counts, cperm);
    }
    return launch_status();
}

// The plans of rays bounds[k] .. bounds[k + 1] - 1 of one LOR array, built
// together: one count pass and one fill pass over all the rays, two host
// synchronisations and two device blocks for the whole set.
int build_set(const float *lors, int64_t n, int64_t ld, const srfx_grid &grid, float tof_bin,
              float tof_sigma2, const srfx_siddon_tile &tile, int K, const int64_t *bounds,
              srfx_siddon_plan *plans, hipStream_t st)
{
    if (K < 1 || !plans || !bounds)
        return SRFX_EINVAL;
    for (int k = 0; k < K; k++)
        plans[k] = nullptr;
    if (bounds[0] < 0 || bounds[K] > n)
        return SRFX_EINVAL;
    for (int k = 0; k < K; k++)
        if (bounds[k + 1] < bounds[k] || bounds[k + 1] - bounds[k] > (int64_t)INT32_MAX)
            return SRFX_EINVAL;
    const int t[3] = {tile.tx, tile.ty, tile.tz};
    for (int c = 0; c < 3; c++)
        if (t[c] <= 0 || grid.shape[c] >= 65536)
            return SRFX_EINVAL;
    if ((int64_t)t[0] * t[1] * t[2] > kMaxTileVox || tile.chunk < 0 ||
        !(tile.block == 0 || tile.block == 64 || tile.block == 128 || tile.block == 256))
        return SRFX_EINVAL;
    SidParams p;
    int rc = siddon_setup(p, lors, n, ld, grid, tof_bin, tof_sigma2);
    if (rc)
        return rc;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return SRFX_ELAUNCH;
    SidTileGeom g = tile_geom(p, t);
    g.keyed = n < ((int64_t)1 << kRayBits) && tile.chunk <= 16 * 256;
    const int slots = cus * scatter_slots((unsigned)(sizeof(double) * g.tvox));
    const int ntiles = g.nt[0] * g.nt[1] * g.nt[2];
    const int64_t ncnt = (int64_t)K * ntiles;
    // block 0: ray records, projection buffer, (plan, tile) counters, bounds
    const size_t nr = (size_t)std::max<int64_t>(n, 1);
    const size_t o_proj = align256(sizeof(float4) * kRayF4 * nr);
    const size_t o_cnt = o_proj + align256(sizeof(float) * nr);
    const size_t o_bnd = o_cnt + align256(sizeof(unsigned long long) * std::max<int64_t>(ncnt, 2 * K));
    const size_t b0 = o_bnd + align256(sizeof(int64_t) * (K + 1));
    char *blk0 = nullptr, *blk1 = nullptr, *blk2 = nullptr;
    if (hipMalloc(&blk0, b0) != hipSuccess)
        return SRFX_ENOMEM;
    auto fail = [&](int code) {
        (void)hipStreamSynchronize(st);
        (void)hipFree(blk0);
        (void)hipFree(blk1);
        (void)hipFree(blk2);
        return code;
    };
    float4 *rays = (float4 *)blk0;
    float *proj = (float *)(blk0 + o_proj);
    auto *cnt = (unsigned long long *)(blk0 + o_cnt);
    auto *dbounds = (int64_t *)(blk0 + o_bnd);
    std::vector<unsigned long long> hc(ncnt, 0ull);
    const bool any = bounds[K] > bounds[0];
    const int64_t m = bounds[K] - bounds[0];
    int *perm = nullptr;
    if (any && (hipMemsetAsync(cnt, 0, sizeof(unsigned long long) * ncnt, st) != hipSuccess ||
                hipMemcpyAsync(dbounds, bounds, sizeof(int64_t) * (K + 1),
                               hipMemcpyHostToDevice, st) != hipSuccess))
        return fail(SRFX_ELAUNCH);
    if (any && tile.sort) {
        // the sorted LOR stream: keys, a radix sort of (key, index), then the
        // sorted copy of the LORs that every pass and projection reads
        if (m > (int64_t)INT32_MAX - 1)
            return fail(SRFX_EINVAL);
        size_t tmp_bytes = 0;
        const int key_bits = 32 + std::max(1, 32 - __builtin_clz((unsigned)K));
        if (hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, (unsigned long long *)nullptr,
                                               (unsigned long long *)nullptr, (int *)nullptr,
                                               (int *)nullptr, (int)m, 0, key_bits, st) !=
            hipSuccess)
            return fail(SRFX_ELAUNCH);
        const size_t o_perm = align256(sizeof(float) * 7 * nr);
        const size_t o_k0 = o_perm + align256(sizeof(int) * nr);
        const size_t o_k1 = o_k0 + align256(sizeof(unsigned long long) * m);
        const size_t o_i0 = o_k1 + align256(sizeof(unsigned long long) * m);
        const size_t o_i1 = o_i0 + align256(sizeof(int) * m);
        const size_t o_tmp = o_i1 + align256(sizeof(int) * m);
        if (hipMalloc(&blk2, o_tmp + tmp_bytes) != hipSuccess)
            return fail(SRFX_ENOMEM);
        auto *slors = (float *)blk2;
        perm = (int *)(blk2 + o_perm);
        auto *k0 = (unsigned long long *)(blk2 + o_k0), *k1 = (unsigned long long *)(blk2 + o_k1);
        auto *i0 = (int *)(blk2 + o_i0), *i1 = (int *)(blk2 + o_i1);
        const dim3 sg(blocks_for(m, 256)), sb(256);
        hipLaunchKernelGGL(sid_sort_key, sg, sb, 0, st, p, dbounds, K, k0, i0);
        if (launch_status() ||
            hipcub::DeviceRadixSort::SortPairs(blk2 + o_tmp, tmp_bytes, k0, k1, i0, i1, (int)m, 0,
                                               key_bits, st) != hipSuccess)
            return fail(SRFX_ELAUNCH);
        hipLaunchKernelGGL(sid_sort_gather, sg, sb, 0, st, p, dbounds, K, k1, i1, slors, perm);
        if (launch_status())
            return fail(SRFX_ELAUNCH);
        p.lors = slors;
        p.ld = n;
    }
    if (any) {
        launch_pass<kBack, false>(p, g, cnt, rays, nullptr, 0, dbounds, K, ntiles, st);
        if (launch_status() ||
            hipMemcpyAsync(hc.data(), cnt, sizeof(unsigned long long) * ncnt,
                           hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            return fail(SRFX_ELAUNCH);
    }
    // (plan, tile) offsets into one run array, then each plan's chunks of at
    // most `chunk` runs of one tile (starts relative to the plan's runs)
    std::vector<unsigned long long> off(ncnt);
    std::vector<SidChunk> chunks;
    std::vector<int64_t> run0(K + 1), chunk0(K + 1);
    unsigned long long total = 0;
    int max_chunk = 0;
    for (int k = 0; k < K; k++) {
        run0[k] = (int64_t)total;
        chunk0[k] = (int64_t)chunks.size();
        unsigned long long listings = 0;
        for (int tt = 0; tt < ntiles; tt++)
            listings += hc[(size_t)k * ntiles + tt];
        const int chunk =
            tile.chunk ? tile.chunk : auto_chunk((long long)listings, slots, kPlanChunkMin);
        max_chunk = std::max(max_chunk, chunk);
        for (int tt = 0; tt < ntiles; tt++) {
            const unsigned long long c = hc[(size_t)k * ntiles + tt];
            off[(size_t)k * ntiles + tt] = total;
            for (unsigned long long s0 = 0; s0 < c; s0 += (unsigned long long)chunk)
                chunks.push_back({(int64_t)(total + s0) - run0[k], tt,
                                  (int)std::min<unsigned long long>(chunk, c - s0)});
            total += c;
        }
    }
    run0[K] = (int64_t)total;
    chunk0[K] = (int64_t)chunks.size();
    int *list = nullptr;
    SidChunk *dchunks = nullptr;
    if (total > 0) {
        const size_t o_ch = align256(sizeof(int) * total);
        if (hipMalloc(&blk1, o_ch + sizeof(SidChunk) * chunks.size()) != hipSuccess)
            return fail(SRFX_ENOMEM);
        list = (int *)blk1;
        dchunks = (SidChunk *)(blk1 + o_ch);
        if (hipMemcpyAsync(cnt, off.data(), sizeof(unsigned long long) * ncnt,
                           hipMemcpyHostToDevice, st) != hipSuccess ||
            hipMemcpyAsync(dchunks, chunks.data(), sizeof(SidChunk) * chunks.size(),
                           hipMemcpyHostToDevice, st) != hipSuccess)
            return fail(SRFX_ELAUNCH);
        launch_pass<kBack, true>(p, g, cnt, rays, list, (int64_t)total, dbounds, K, ntiles, st);
        if (g.keyed) {
            // the sort's plan tables go where the counters were
            auto *tab = (int64_t *)cnt;
            if (hipMemcpyAsync(tab, chunk0.data(), sizeof(int64_t) * K, hipMemcpyHostToDevice,
                               st) != hipSuccess ||
                hipMemcpyAsync(tab + K, run0.data(), sizeof(int64_t) * K, hipMemcpyHostToDevice,
                               st) != hipSuccess)
                return fail(SRFX_ELAUNCH);
            hipLaunchKernelGGL(sid_sort_chunks, dim3((unsigned)chunks.size()), dim3(256),
                               sizeof(int) * (kSortBuckets + 1 + max_chunk), st, dchunks, tab, tab + K,
                               K, list);
        }
        if (launch_status())
            return fail(SRFX_ELAUNCH);
    }
    if (hipStreamSynchronize(st) != hipSuccess)
        return fail(SRFX_ELAUNCH);
    auto *arena = new srfx_siddon_plan_s::Arena;
    arena->mem[0] = blk0;
    arena->mem[1] = blk1;
    arena->mem[2] = blk2;
    arena->refs.store(K);
    for (int k = 0; k < K; k++) {
        auto *pl = new srfx_siddon_plan_s;
        pl->p = p;
        pl->p.lors = n > 0 ? p.lors + bounds[k] : p.lors;
        pl->perm = perm ? perm + bounds[k] : nullptr;
        pl->p.n = bounds[k + 1] - bounds[k];
        pl->grid = grid;
        pl->g = g;
        pl->block = tile.block ? tile.block : 256;
        pl->rays = rays + kRayF4 * bounds[k];
        pl->proj = proj + bounds[k];
        pl->list = list ? list + run0[k] : nullptr;
        pl->nruns = run0[k + 1] - run0[k];
        pl->chunks = dchunks ? dchunks + chunk0[k] : nullptr;
        pl->nchunks = (int)(chunk0[k + 1] - chunk0[k]);
        pl->arena = arena;
        plans[k] = pl;
    }
    return SRFX_OK;
}

// Weights (ray, voxel) from which an untiled scatter runs binned, by the
// estimate below.
constexpr double kBinnedWeights = 2.0e6;

} // namespace

namespace srfx {

bool siddon_binned_rule(const SidParams &p)
{
    for (int c = 0; c < 3; c++)
        if (p.g[c] >= 65536)
            return false;
    // a ray through the middle crosses about half the planes of all axes, or
    // those of the +-3 sigma its TOF test leaves
    double planes = 0.0, per_mm = 0.0;
    for (int c = 0; c < 3; c++) {
        planes += 0.5 * p.g[c];
        per_mm += 0.45 * p.g[c] / p.size[c];
    }
    if (p.use_tof && p.tof_sigma2 > 0.0f)
        planes = std::min(planes, 6.0 * std::sqrt((double)p.tof_sigma2) * per_mm);
    if (planes * (double)p.n < kBinnedWeights)
        return false;
    const SidTileGeom g = tile_geom(p, {16, 16, 8});
    return (int64_t)g.nt[0] * g.nt[1] * g.nt[2] < (1 << 20);
}

bool siddon_binned_ok(const SidParams &p, hipStream_t st)
{
    return siddon_binned_rule(p) && workspace_ok(st);
}

int siddon_binned_scatter(int mode, const SidParams &p, hipStream_t st, bool *done)
{
    *done = false;
    SidTileGeom g = tile_geom(p, {16, 16, 8});
    g.keyed = 1;
    const int nt = g.nt[0] * g.nt[1] * g.nt[2];
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return SRFX_ELAUNCH;
    // a ray steps through at most this many tiles
    const int64_t per = (int64_t)g.nt[0] + g.nt[1] + g.nt[2] - 2;
    const int64_t most = std::min<int64_t>(kBinPiece, std::max<int64_t>(4096, (1 << 28) / (4 * per)));
    const int64_t pieces = (p.n + most - 1) / most, piece = (p.n + pieces - 1) / pieces;
    const int64_t cap = piece * per, nch = nt + cap / kChunkMin + 1;
    const size_t o_bnd = align256(sizeof(SidBinState));
    const size_t o_cnt = o_bnd + 256;
    const size_t o_ch = o_cnt + align256(sizeof(unsigned long long) * (size_t)nt);
    const size_t o_ray = o_ch + align256(sizeof(TileSpan) * (size_t)nch);
    const size_t o_proj = o_ray + align256(sizeof(float4) * kRayF4 * (size_t)piece);
    const size_t o_list = o_proj + align256(mode == kOsem ? sizeof(float) * (size_t)piece : 0);
    char *ws = nullptr;
    if (ws_alloc((void **)&ws, o_list + sizeof(int) * (size_t)cap, st))
        return SRFX_OK; // no workspace: the direct kernels
    SidBins b{};
    b.state = (SidBinState *)ws;
    b.bounds = (int64_t *)(ws + o_bnd);
    b.cnt = (unsigned long long *)(ws + o_cnt);
    b.chunks = (TileSpan *)(ws + o_ch);
    b.rays = (float4 *)(ws + o_ray);
    b.proj = (float *)(ws + o_proj);
    b.list = (int *)(ws + o_list);
    const unsigned lds = (unsigned)(sizeof(double) * g.tvox);
    const dim3 sb((unsigned)(cus * scatter_slots(lds))), block(256);
    int rc = SRFX_OK;
    for (int64_t e0 = 0; e0 < p.n && !rc; e0 += piece) {
        SidParams q = p;
        q.n = std::min(piece, p.n - e0);
        q.lors = p.lors + e0;
        q.val = p.val ? p.val + e0 : nullptr;
        hipLaunchKernelGGL(sid_bin_init, dim3((unsigned)std::min(64, (nt + 255) / 256)), block, 0,
                           st, b, nt, q.n);
        if (mode == kMap)
            launch_pass<kMap, false>(q, g, b.cnt, b.rays, nullptr, 0, b.bounds, 1, nt, st);
        else
            launch_pass<kBack, false>(q, g, b.cnt, b.rays, nullptr, 0, b.bounds, 1, nt, st);
        hipLaunchKernelGGL(sid_bin_scan, dim3(1), dim3(kScanThreads), 0, st, b, nt, (int)sb.x);
        launch_pass<kBack, true>(q, g, b.cnt, b.rays, b.list, cap, b.bounds, 1, nt, st);
        hipLaunchKernelGGL(sid_bin_sort, dim3((unsigned)std::min<int64_t>(nch, 8 * cus)), block,
                           sizeof(int) * (kSortBuckets + 1 + kChunkMax), st, b);
        const float *vals = q.val;
        if (mode == kOsem) {
            rc = record_project(q, b.rays, b.proj, st);
            vals = b.proj;
        }
        const bool adj = mode == kAdj;
        if (q.use_tof && adj)
            hipLaunchKernelGGL((sid_bin_scatter<true, true>), sb, block, lds, st, q, g, b, vals);
        else if (q.use_tof)
            hipLaunchKernelGGL((sid_bin_scatter<true, false>), sb, block, lds, st, q, g, b, vals);
        else if (adj)
            hipLaunchKernelGGL((sid_bin_scatter<false, true>), sb, block, lds, st, q, g, b, vals);
        else
            hipLaunchKernelGGL((sid_bin_scatter<false, false>), sb, block, lds, st, q, g, b, vals);
        rc = rc ? rc : launch_status();
    }
    *done = true;
    const int rf = ws_free(ws, st);
    return rc ? rc : rf;
}

} // namespace srfx

extern "C" int srfx_siddon_plan_create(const float *lors, int64_t n, int64_t ld, srfx_grid grid,
                                       float tof_bin, float tof_sigma2, srfx_siddon_tile tile,
                                       srfx_siddon_plan *plan, void *stream)
{
    if (!plan)
        return SRFX_EINVAL;
    const int64_t bounds[2] = {0, n < 0 ? 0 : n};
    if (n < 0)
        return SRFX_EINVAL;
    return build_set(lors, n, ld, grid, tof_bin, tof_sigma2, tile, 1, bounds, plan,
                     (hipStream_t)stream);
}

extern "C" int srfx_siddon_plan_create_subsets(const float *lors, int64_t n, int64_t ld,
                                               srfx_grid grid, float tof_bin, float tof_sigma2,
                                               srfx_siddon_tile tile, int32_t nplans,
                                               const int64_t *bounds, srfx_siddon_plan *plans,
                                               void *stream)
{
    return build_set(lors, n, ld, grid, tof_bin, tof_sigma2, tile, nplans, bounds, plans,
                     (hipStream_t)stream);
}

extern "C" int srfx_siddon_plan_info(srfx_siddon_plan plan, int64_t *nruns, int32_t *nchunks)
{
    if (!plan)
        return SRFX_EINVAL;
    if (nruns)
        *nruns = plan->nruns;
    if (nchunks)
        *nchunks = plan->nchunks;
    return SRFX_OK;
}

extern "C" int srfx_siddon_plan_destroy(srfx_siddon_plan plan)
{
    if (!plan)
        return SRFX_OK;
    (void)hipDeviceSynchronize();
    plan_release(plan);
    return SRFX_OK;
}

extern "C" int srfx_siddon_plan_backproject(srfx_siddon_plan plan, const float *lors_value,
                                            float *image, uint32_t flags, void *stream)
{
    if (!plan || !image || (plan->p.n > 0 && !lors_value))
        return SRFX_EINVAL;
    return plan_scatter(plan, false, lors_value, plan->perm, nullptr, nullptr, image, flags,
                        (hipStream_t)stream);
}

extern "C" int srfx_siddon_plan_backproject_adjoint(srfx_siddon_plan plan, const float *g,
                                                    float *image, uint32_t flags, void *stream)
{
    if (!plan || !image || (plan->p.n > 0 && !g))
        return SRFX_EINVAL;
    return plan_scatter(plan, true, g, plan->perm, nullptr, nullptr, image, flags,
                        (hipStream_t)stream);
}

extern "C" int srfx_siddon_plan_osem_subset(srfx_siddon_plan plan, const float *image,
                                            const float *counts, float *bp, uint32_t flags,
                                            void *stream)
{
    const bool project = !(flags & SRFX_OSEM_SCATTER_ONLY);
    const bool scatter = !(flags & SRFX_OSEM_PROJECT_ONLY);
    if (!plan || (scatter && !bp) || (project && plan->p.n > 0 && !image) ||
        (!project && !scatter))
        return SRFX_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    const SidParams &p = plan->p;
    if (project && p.n > 0) {
        SidParams q = p;
        q.img = image;
        const int rc = record_project(q, plan->rays, plan->proj, st);
        if (rc)
            return rc;
    }
    if (!scatter)
        return SRFX_OK;
    return plan_scatter(plan, false, plan->proj, nullptr, counts, plan->perm, bp,
                        flags & SRFX_ACCUMULATE, st);
}

extern "C" int srfx_siddon_plan_projection(srfx_siddon_plan plan, float *out, void *stream)
{
    if (!plan || (plan->p.n > 0 && !out))
        return SRFX_EINVAL;
    if (plan->p.n == 0)
        return SRFX_OK;
    hipStream_t st = (hipStream_t)stream;
    if (plan->perm) {
        hipLaunchKernelGGL(sid_unsort, dim3(blocks_for(plan->p.n, 256)), dim3(256), 0, st,
                           (const float *)plan->proj, (const int *)plan->perm, plan->p.n, out);
        return launch_status();
    }
    if (hipMemcpyAsync(out, plan->proj, sizeof(float) * plan->p.n, hipMemcpyDeviceToDevice,
                       st) != hipSuccess)
        return SRFX_ELAUNCH;
    return SRFX_OK;
}
