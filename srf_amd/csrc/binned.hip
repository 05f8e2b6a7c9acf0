// Binned scatter: the untiled TOR scatters (backprojection, adjoint, Maplors,
// OSEM pass) over a large event set, through image tiles like a plan
// (tile_core.h) that is built, used once and dropped inside the call.
//
// The direct scatter (tor_kernel) adds every weight to the image with an FP32
// global atomic of its own and runs at the L2's rate for scattered atomics,
// 2e10 a second: 14.3 ms per 1M events at 200 x 200 x 100, whatever the
// event order.  Here the events of the call are listed by image tile and each
// tile is accumulated in LDS and flushed with coalesced atomics.  Everything
// stays on the device: no count is read back, so the call does not
// synchronise.  Per piece of at most kPieceEvents events:
//   bin_init            tables and counters;
//   plan_set_pass<0>    walk records, listings per tile;
//   bin_scan            slots and chunks of the tiles (one workgroup);
//   plan_set_pass<1>    the listings with their slices;
//   bin_sort            listings of a chunk ordered by length;
//   bin_project         (OSEM pass) projections into the records;
//   bin_scatter         workgroups pull chunks: LDS tile, flush.
// The listing array is sized for the longest average an event set of one axis
// group can have (every event across the whole frame at 45 degrees along both
// in-slice axes).  An event set beyond that (events far from the slice axis)
// leaves the chunk table empty and sets a flag on which the passes after the scan
// return at once and bin_direct, the direct scatter, runs.
#include <algorithm>

#include "binned.h"
#include "locality.h"
#include "tile_core.h"

namespace srfx {

namespace {

constexpr int64_t kPieceEvents = 1 << 19;
constexpr int64_t kWorkspace = (int64_t)256 << 20; // bytes of one piece
constexpr int kBinChunk = 2048;                    // listings per workgroup
constexpr int kScanThreads = 1024;

// Words the scan and the kernels behind it share.
struct BinState {
    int over;    // the listings do not fit: run the direct scatter
    int other;   // an event needs another walk than the NB x (NB - 1) box
    int err;     // fill pass (always 0: the passes enumerate alike)
    int nchunks; // chunks in the table
    unsigned next[2]; // work counters of bin_scatter (single walk, general)
};

struct BinTables {
    BinState *state;
    int64_t *first; // [2]
    float4 **rec;   // [1]
    int **list;     // [1]
    int *cnt, *fill, *off; // [nt] each
    TileChunk *chunks;
    float4 *rec0;
    int *list0;
    int cap, max_chunks; // slots of list0, entries of chunks
};

__global__ __launch_bounds__(256) void bin_init(BinTables b, int nt, int64_t n)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    for (int k = i; k < 2 * nt; k += (int)(gridDim.x * blockDim.x))
        b.cnt[k] = 0; // cnt and fill are adjacent
    if (i == 0) {
        *b.state = BinState{};
        b.first[0] = 0;
        b.first[1] = n;
        b.rec[0] = b.rec0;
        b.list[0] = b.list0;
    }
}

// Slot and chunk offsets of every tile: one pass over the tiles window by
// window, each window's slabs in order (an event's listings in consecutive
// slabs mostly share a window, so its record is read again while the L2 holds
// it), 1024 tiles a round with a prefix sum of (listings, chunks).
__global__ __launch_bounds__(kScanThreads) void bin_scan(BinTables b, TileGeom g, int nt)
{
    const int nw = g.nwx * g.nwy;
    long long carry = 0; // listings | chunks << 40
    for (int q0 = 0; q0 < nt; q0 += kScanThreads) {
        const int q = q0 + (int)threadIdx.x;
        const int t = q < nt ? (q % g.nslab) * nw + q / g.nslab : 0;
        const int c = q < nt ? b.cnt[t] : 0;
        const int nch = (c + kBinChunk - 1) / kBinChunk;
        long long total;
        const long long ex =
            carry + block_scan<kScanThreads>((long long)c | ((long long)nch << 40), total);
        const long long o = ex & ((1ll << 40) - 1);
        const int ch = (int)(ex >> 40);
        if (q < nt) {
            b.off[t] = (int)o;
            for (int k = 0; k < nch; k++)
                if (ch + k < b.max_chunks)
                    b.chunks[ch + k] = TileChunk{t, (int)o + k * kBinChunk,
                                                 min(kBinChunk, c - k * kBinChunk), 0};
        }
        carry += total;
    }
    const long long listings = carry & ((1ll << 40) - 1);
    const int nch = (int)(carry >> 40);
    const bool over = listings > b.cap || nch > b.max_chunks;
    if (threadIdx.x == 0) {
        b.state->over = over;
        b.state->nchunks = over ? 0 : nch;
    }
}

__global__ __launch_bounds__(256) void bin_sort(BinTables b)
{
    extern __shared__ int sh[];
    const int n = b.state->nchunks;
    for (int c = blockIdx.x; c < n; c += gridDim.x)
        sort_chunk<true>(TorParams{}, TileGeom{}, b.chunks[c], b.list0, nullptr, sh);
}

// tile_scatter over the device's chunk table: workgroups pull chunks.  Both
// forms are launched; the one whose walk does not fit the events returns.  The
// scale stays out of the weights' exponent, as in the direct scatter.
template <int MODE, int NB, bool VREC, bool ONE>
__global__ __launch_bounds__(256, NB == 4 ? (ONE ? 4 : 3) : (ONE ? 5 : 4)) void bin_scatter(
    TorParams p, TileGeom g, BinTables b)
{
    extern __shared__ double ldsd[];
    if (NB > 0 && (b.state->other == 0) != ONE)
        return;
    const int n = b.state->nchunks;
    for (;;) {
        const int c = next_item(&b.state->next[ONE ? 0 : 1]);
        if (c >= n)
            break;
        scatter_chunk<MODE, NB, VREC, ONE, false>(p, g, b.chunks[c], b.list0, b.rec0, ldsd);
    }
}

// record_proj_kernel<NB, 4, FRAME> of a set that fits.
template <int NB, bool FRAME>
__global__ __launch_bounds__(256, NB == 3 && FRAME ? 5 : 4) void bin_project(
    TorParams p, float4 *rec, const BinState *state)
{
    if (state->over)
        return;
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t e = gid / 64 * 16 + (int)(gid % 16);
    record_project<NB, 4, FRAME>(p, rec, e, (int)(gid % 64) / 16, e < p.n);
}

// The direct scatter, for an event set that did not fit.
template <int MODE, int NB>
__global__ __launch_bounds__(256) void bin_direct(TorParams p, const BinState *state)
{
    if (state->over == 0)
        return;
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < p.n; e += step)
        run_event<MODE, NB, 1>(p, e, 0, true);
}

// The tile of a binned pass: that of the plans (30 KB of FP64 LDS, five
// workgroups per CU; row walks list fewer pairs in a wider window).
TileGeom bin_geom(const TorParams &p)
{
    TileGeom g{};
    g.S = 12;
    g.Wx = 32;
    g.Wy = p.box ? 10 : 12;
    g.nwx = (p.gx + g.Wx - 1) / g.Wx;
    g.nwy = (p.gy + g.Wy - 1) / g.Wy;
    g.nslab = (p.gz + g.S - 1) / g.S;
    g.sorted = g.spans = 1;
    return g;
}

// Listings per event of a set whose events all cross the whole frame at 45
// degrees along both in-slice axes (an axis group's largest slopes), plus one
// slab's.
int bin_listings(const TorParams &p, const TileGeom &g)
{
    const double h = std::sqrt(2.0 * 9.0 * p.tor_sigma2);
    const double wx = 1.0 + (g.S * p.inter_z + 2.0 * h) * p.rinter_x / g.Wx;
    const double wy = 1.0 + (g.S * p.inter_z + 2.0 * h) * p.rinter_y / g.Wy;
    return (int)std::min(4096.0, std::ceil((g.nslab + 1) * std::min(wx, (double)g.nwx + 1.0) *
                                           std::min(wy, (double)g.nwy + 1.0)));
}

template <int MODE, int NB, bool VREC>
int launch_bin_scatter(const TorParams &p, const TileGeom &g, const BinTables &b, int cus,
                       hipStream_t st)
{
    const unsigned sh = (unsigned)(sizeof(double) * g.S * g.Wx * g.Wy);
    auto blocks = [&](unsigned per_cu) {
        return dim3((unsigned)std::min<int64_t>(b.max_chunks, (int64_t)cus * per_cu));
    };
    if constexpr (NB > 0)
        hipLaunchKernelGGL((bin_scatter<MODE, NB, VREC, true>), blocks(NB == 4 ? 4 : 5), dim3(256),
                           sh, st, p, g, b);
    hipLaunchKernelGGL((bin_scatter<MODE, NB, VREC, false>), blocks(NB == 4 ? 3 : 4), dim3(256),
                       sh, st, p, g, b);
    return launch_status();
}

// The direct fallback runs the OSEM pass as such (it projects again).
template <int MODE, int NB>
int launch_bin(const TorParams &p, const TileGeom &g, const BinTables &b, int cus, hipStream_t st)
{
    constexpr bool osem = MODE == kOsem;
    if (osem) {
        TorParams q = p;
        const int64_t bytes = (int64_t)4 * p.gx * p.gy * p.gz;
        q.img_bytes = (int)bytes;
        if (p.sx == 1 && p.sy == p.gx && p.sz == p.gx * p.gy && bytes < ((int64_t)1 << 31) &&
            (int64_t)p.gx * p.gy < ((int64_t)1 << 24))
            hipLaunchKernelGGL((bin_project<NB, true>), dim3(blocks_for(4 * p.n, 256)), dim3(256),
                               0, st, q, b.rec0, b.state);
        else
            hipLaunchKernelGGL((bin_project<NB, false>), dim3(blocks_for(4 * p.n, 256)),
                               dim3(256), 0, st, q, b.rec0, b.state);
    }
    int rc = launch_bin_scatter<osem ? kBack : MODE, NB, osem>(p, g, b, cus, st);
    if (rc)
        return rc;
    hipLaunchKernelGGL((bin_direct<MODE, NB>),
                       dim3((unsigned)std::min<int64_t>(blocks_for(p.n, 256), 8 * cus)), dim3(256),
                       0, st, p, b.state);
    return launch_status();
}

template <int MODE>
int launch_bin_box(const TorParams &p, const TileGeom &g, const BinTables &b, int cus,
                   hipStream_t st)
{
    switch (p.box) {
    case 3:
        return launch_bin<MODE, 3>(p, g, b, cus, st);
    case 4:
        return launch_bin<MODE, 4>(p, g, b, cus, st);
    default:
        return launch_bin<MODE, 0>(p, g, b, cus, st);
    }
}

} // namespace

// Weights (event, voxel) from which an untiled scatter runs binned.  The direct
// scatter takes 1 s per 2e10 weights, the binned one 0.09 ms and up for its
// passes; they meet at (events, direct and binned ms) 8000, 0.117 and 0.105 at
// 200 x 200 x 100 (2 mm, 4 mm tube, 530 ps), 64000, 0.133 and 0.124 at
// 96 x 96 x 48 (4 mm), 2000, 0.120 and 0.119 with an 8 mm tube, 4000, 0.124
// and 0.137 without TOF: 2.1e6 to 2.4e6 weights by the estimate below.  Beyond,
// 1M events take 14.0 against 0.98 ms, 1.95 against 0.56, and 55 against 2.4.
constexpr double kBinnedWeights = 2.4e6;
// And weights per event: the passes take 0.3 ns and more an event, the time of six
// direct weights.  Tubes thinner than the voxels have few: 800k events a group,
// direct and binned us of two groups, 64 x 64 x 32 (6.3 mm, 3 mm tube, 530 ps; 5.7 an
// event) 541 and 840, 40 x 40 x 20 (10 mm, 4 mm tube; 5.0) 582 and 829, (3 mm, 530 ps;
// 1.4) 234 and 712; 64 x 64 x 32 (4 mm, 530 ps; 10.2) 900 and 887, 80 x 80 x 40 (5 mm,
// 3 mm, 530 ps; 11.5) 944 and 935, 40 x 40 x 20 (6 mm; 11.4) 1043 and 874.
constexpr double kBinnedPerEvent = 10.0;

// Weights of an event: the tube's cross-section in voxels times its slices, those
// of the frame or, with TOF, of the +-3 sigma its end points are cut to.
static double event_weights(const TorParams &p)
{
    const double area = 9.0 * M_PI * p.tor_sigma2 * p.rinter_x * p.rinter_y;
    const double cut =
        p.use_tof ? 6.0 / std::sqrt((double)p.tse_inv) * p.rinter_z : (double)p.gz;
    return area * std::min(cut, (double)p.gz);
}

bool binned_rule(const TorParams &p, uint32_t flags)
{
    // a schedule in the flags asks for the direct kernels
    constexpr uint32_t sched = (3u << SRFX_LPE_SHIFT) | (3u << SRFX_BLOCK_SHIFT) |
                               (3u << SRFX_SLAB_SHIFT) | SRFX_FULL_PATCH;
    const double w = event_weights(p);
    if ((flags & sched) || w < kBinnedPerEvent || w * (double)p.n < kBinnedWeights)
        return false;
    // the tables of the plan passes index tiles with 24 bits
    const TileGeom g = bin_geom(p);
    return (int64_t)g.nwx * g.nwy * g.nslab < (1 << 20);
}

bool binned_ok(const TorParams &p, uint32_t flags, hipStream_t st)
{
    return binned_rule(p, flags) && workspace_ok(st);
}

int binned_scatter(int mode, const TorParams &p, hipStream_t st, bool *done)
{
    *done = false;
    const TileGeom g = bin_geom(p);
    const int nt = g.nwx * g.nwy * g.nslab;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return SRFX_ELAUNCH;
    const int64_t per = bin_listings(p, g);
    const int64_t most = std::min<int64_t>(
        kPieceEvents, std::max<int64_t>(4096, kWorkspace / (16 * kWalkF4 + 4 * per)));
    const int64_t pieces = (p.n + most - 1) / most, piece = (p.n + pieces - 1) / pieces;
    const int64_t cap = std::min<int64_t>(piece * per, INT32_MAX / 2);
    const int64_t nch = nt + cap / kBinChunk + 1;
    const size_t o_state = 0, o_head = align256(sizeof(BinState));
    const size_t o_ctr = o_head + 256;
    const size_t o_ch = o_ctr + align256(sizeof(int) * 3 * (size_t)nt);
    const size_t o_rec = o_ch + align256(sizeof(TileChunk) * (size_t)nch);
    const size_t o_list = o_rec + align256(sizeof(float4) * kWalkF4 * (size_t)piece);
    const size_t bytes = o_list + sizeof(int) * (size_t)cap;
    char *ws = nullptr;
    if (ws_alloc((void **)&ws, bytes, st))
        return SRFX_OK; // no workspace: the direct kernels
    BinTables b{};
    b.state = (BinState *)(ws + o_state);
    b.first = (int64_t *)(ws + o_head);
    b.rec = (float4 **)(ws + o_head + 16);
    b.list = (int **)(ws + o_head + 32);
    b.cnt = (int *)(ws + o_ctr);
    b.fill = b.cnt + nt;
    b.off = b.fill + nt;
    b.chunks = (TileChunk *)(ws + o_ch);
    b.rec0 = (float4 *)(ws + o_rec);
    b.list0 = (int *)(ws + o_list);
    b.cap = (int)cap;
    b.max_chunks = (int)nch;
    PlanSetArgs a{};
    a.cols7 = mode == kMap;
    a.ntiles = nt;
    a.nplans = 1;
    a.lds = 3u * sizeof(int) * nt <= 65536u;
    a.queue = fill_queue_entries(nt);
    a.first = b.first;
    a.rec = b.rec;
    a.list = b.list;
    a.cnt = b.cnt;
    a.fill = b.fill;
    a.off = b.off;
    a.err = &b.state->err;
    a.skip = &b.state->over;
    a.other = &b.state->other;
    int rc = SRFX_OK;
    for (int64_t e0 = 0; e0 < p.n && !rc; e0 += piece) {
        TorParams q = p;
        q.n = std::min(piece, p.n - e0);
        q.lors = p.lors + e0;
        q.val = p.val ? p.val + e0 : nullptr;
        const dim3 eb(blocks_for(q.n, 256));
        hipLaunchKernelGGL(bin_init, dim3((unsigned)std::min(64, (2 * nt + 255) / 256)),
                           dim3(256), 0, st, b, nt, q.n);
        hipLaunchKernelGGL(plan_set_pass<false>, eb, dim3(256),
                           a.lds ? sizeof(int) * (unsigned)nt : 0u, st, q, g, a);
        hipLaunchKernelGGL(bin_scan, dim3(1), dim3(kScanThreads), 0, st, b, g, nt);
        hipLaunchKernelGGL(plan_set_pass<true>, eb, dim3(256),
                           (a.lds ? 3u * sizeof(int) * (unsigned)nt : 0u) +
                               (a.queue ? fill_queue_lds(a.queue) : 0u),
                           st, q, g, a);
        hipLaunchKernelGGL(bin_sort, dim3((unsigned)std::min<int64_t>(nch, 8 * cus)), dim3(256),
                           sizeof(int) * (33 + kBinChunk), st, b);
        switch (mode) {
        case kBack:
            rc = launch_bin_box<kBack>(q, g, b, cus, st);
            break;
        case kAdj:
            rc = launch_bin_box<kAdj>(q, g, b, cus, st);
            break;
        case kMap:
            rc = launch_bin_box<kMap>(q, g, b, cus, st);
            break;
        default:
            rc = launch_bin_box<kOsem>(q, g, b, cus, st);
            break;
        }
    }
    *done = true;
    const int rf = ws_free(ws, st);
    return rc ? rc : rf;
}

namespace {

// Walk records of a set's events at their places in its locality order, the
// event's number in the record's value slot.  FP64 event set-up once per event.
__global__ __launch_bounds__(256) void sorted_place_kernel(TorParams p, LocalityOrder o,
                                                           float4 *rec)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= p.n)
        return;
    RawEvent r;
    fetch_event<kProj>(p, e, r);
    const ExactGeom eg = exact_geom(p, r);
    Event ev;
    Track t;
    const bool valid = init_event<kProj>(p, r, eg, ev);
    if (valid)
        make_track(p, ev, eg, r, t);
    const int64_t j = (int64_t)atomicAdd(&o.cursor[o.key[e]], 1u);
    pack_walk(p, r, ev, t, valid, rec, j);
    reinterpret_cast<int *>(rec)[4 * kWalkHead * j + kWalkValue] = (int)e;
}

// The projection of events in locality order from their records, as
// record_proj_kernel's (four lanes per event, the 16 events of a wave on the
// same slices at the same time, so that their gathers share cache lines), to the
// events' own numbers.  FRAME: p.img is a contiguous op frame of p.img_bytes.
template <int NB, bool FRAME>
__global__ __launch_bounds__(256, NB == 3 && FRAME ? 5 : 4) void sorted_proj_kernel(
    TorParams p, float4 *rec)
{
    const int64_t gid = (int64_t)xcd_block() * blockDim.x + threadIdx.x;
    const int64_t e = gid / 64 * 16 + (int)(gid % 16);
    record_project<NB, 4, FRAME, true>(p, rec, e, (int)(gid % 64) / 16, e < p.n, p.out);
}

template <bool FRAME>
int launch_sorted(const TorParams &p, float4 *rec, hipStream_t st)
{
    const dim3 grid(blocks_for(4 * p.n, 256)), block(256);
    switch (p.box) {
    case 3:
        hipLaunchKernelGGL((sorted_proj_kernel<3, FRAME>), grid, block, 0, st, p, rec);
        break;
    case 4:
        hipLaunchKernelGGL((sorted_proj_kernel<4, FRAME>), grid, block, 0, st, p, rec);
        break;
    default:
        hipLaunchKernelGGL((sorted_proj_kernel<0, FRAME>), grid, block, 0, st, p, rec);
        break;
    }
    return launch_status();
}

// Where ordering the events first pays: from 131073 events on (below, lanes
// that share an event hide the gathers' latency and the four ordering kernels
// are launch-bound) over images whose gathers miss L2.  Events in time order, one
// lane per event against this path, us: 200 x 200 x 100 x 200k events 298 / 190,
// x 1M 1165 / 607; 256 x 256 x 160 x 1M 1989 / 798; 181 x 175 x 83 x 400k 380 / 271;
// 160 x 160 x 80 (8.2 MB) x 400k 213 / 250.  Events that come in locality order
// already, same columns: 197 / 187, 565 / 642, 1112 / 838, 241 / 290, 180 / 258.
// Tubes wider than four voxels, four lanes per event against this path: 181 x 175
// x 83 x 280k 672 / 511, x 600k 1301 / 847; 150 x 150 x 64 (5.8 MB) x 280k 326 /
// 379, x 600k 607 / 619; 128 x 128 x 64 x 600k 523 / 568.
constexpr int64_t kSortedEvents = 131073;
constexpr int64_t kSortedBytes = 10000000; // of the image
constexpr int64_t kSortedPiece = (int64_t)1 << 20; // 151 MB of records

} // namespace

int sorted_project(const TorParams &p, uint32_t flags, hipStream_t st, bool *done)
{
    *done = false;
    constexpr uint32_t sched = (3u << SRFX_LPE_SHIFT) | (3u << SRFX_BLOCK_SHIFT) |
                               (3u << SRFX_SLAB_SHIFT) | SRFX_FULL_PATCH;
    const int64_t bytes = (int64_t)4 * p.gx * p.gy * p.gz;
    if ((flags & sched) || p.n < kSortedEvents ||
        bytes < kSortedBytes || !workspace_ok(st))
        return SRFX_OK;
    const int64_t piece = std::min<int64_t>(p.n, kSortedPiece);
    const size_t rb = align256(sizeof(float4) * kWalkF4 * (size_t)piece);
    char *ws = nullptr;
    if (ws_alloc((void **)&ws, rb + locality_bytes(piece, 1), st))
        return SRFX_OK;
    const bool frame = p.sx == 1 && p.sy == p.gx && p.sz == p.gx * p.gy &&
                       bytes < ((int64_t)1 << 31) && (int64_t)p.gx * p.gy < ((int64_t)1 << 24);
    int rc = SRFX_OK;
    for (int64_t e0 = 0; e0 < p.n && !rc; e0 += piece) {
        TorParams q = p;
        q.n = std::min(piece, p.n - e0);
        q.lors = p.lors + e0;
        q.out = p.out + e0;
        q.img_bytes = (int)bytes;
        LocalityOrder order;
        rc = locality_order(q, 1, order, ws + rb, st);
        if (rc)
            break;
        hipLaunchKernelGGL(sorted_place_kernel, dim3(blocks_for(q.n, 256)), dim3(256), 0, st, q,
                           order, (float4 *)ws);
        rc = frame ? launch_sorted<true>(q, (float4 *)ws, st)
                   : launch_sorted<false>(q, (float4 *)ws, st);
    }
    *done = true;
    const int rf = ws_free(ws, st);
    return rc ? rc : rf;
}

} // namespace srfx
