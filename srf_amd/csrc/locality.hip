// Locality order of TOR events, for kernels whose lanes should walk neighbouring
// tubes: buckets by where an event is (position of its tube at the TOF centre's
// slice, slopes, slice), with bins taken from the events themselves.
//
// Five quantities per event, in voxels: the tube's column and row at the slice of
// the TOF centre (without TOF the middle of the event), the slopes times the
// slices a walk extends to either side, and that slice, which matters less.
// Their ranges over the set decide how many of the key's bits each gets, a bit
// at a time to the one with the widest bins, most significant first, so that
// neighbouring buckets are neighbours too.  200k events: 45 us for the four
// kernels, launch-bound (range 10, bits 10, count 16, scan 8), where a radix
// sort of keys takes 130.
#include <algorithm>

#include "locality.h"

namespace srfx {
namespace {

constexpr int kDims = 5;
constexpr int kMaxBits = 16; // of a subset's key
constexpr int kScan = 1024;

struct LocalityState {
    float base[kDims], scale[kDims];
    int seq[kMaxBits]; // dimension | bit << 8 of each key bit, top first
};

constexpr int kRangeBlocks = 256;

// The five quantities of event e, clamped to the frame (NaN: the lower end).
__device__ __forceinline__ void locality_coords(const TorParams &p, int64_t e,
                                                float (&q)[kDims])
{
    const float *L = p.lors + e;
    const int64_t ld = p.ld;
    const float x1 = L[0], y1 = L[ld], z1 = L[2 * ld];
    const float dx = L[3 * ld] - x1, dy = L[4 * ld] - y1, dz = L[5 * ld] - z1;
    const bool tof = p.use_tof;
    float zc = tof ? L[8 * ld] : z1 + 0.5f * dz;
    const float rz = (float)p.rinter_z, zb = (float)p.zbase;
    zc = fminf(fmaxf(zc, zb), zb + (float)(p.gz - 1) / rz);
    const float r = dz != 0.0f ? 1.0f / dz : 0.0f;
    const float t = (zc - z1) * r;
    // slices a walk extends to either side of zc: TOF cuts at three sigma
    const float reach = tof && p.tse_inv > 0.0f ? fminf(3.0f * rsqrtf(p.tse_inv) * rz, 0.5f * p.gz)
                                                : 0.5f * p.gz;
    const float v[kDims] = {(fmaf(dx, t, x1) - (float)p.l_bound) * p.rfinter_x,
                            (fmaf(dy, t, y1) - (float)p.b_bound) * p.rfinter_y,
                            dx * r * p.rfinter_x * reach / rz, dy * r * p.rfinter_y * reach / rz,
                            (zc - zb) * rz};
    const float top[kDims] = {(float)p.gx, (float)p.gy, 2.0f * p.gx, 2.0f * p.gy, (float)p.gz};
#pragma unroll
    for (int d = 0; d < kDims; d++)
        q[d] = fminf(fmaxf(v[d], d == 2 || d == 3 ? -top[d] : 0.0f), top[d]);
}

// Ranges of the five quantities, one partial per workgroup (min, max each), and
// the counts zeroed.
__global__ __launch_bounds__(256) void locality_range(TorParams p, float *part,
                                                      unsigned *hist, int64_t nh)
{
    __shared__ float red[4][2 * kDims];
    const int64_t first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t k = first; k < nh; k += step)
        hist[k] = 0u;
    float lo[kDims], hi[kDims];
#pragma unroll
    for (int d = 0; d < kDims; d++) {
        lo[d] = INFINITY;
        hi[d] = -INFINITY;
    }
    for (int64_t e = first; e < p.n; e += step) {
        float q[kDims];
        locality_coords(p, e, q);
#pragma unroll
        for (int d = 0; d < kDims; d++) {
            lo[d] = fminf(lo[d], q[d]);
            hi[d] = fmaxf(hi[d], q[d]);
        }
    }
#pragma unroll
    for (int d = 0; d < kDims; d++) {
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            lo[d] = fminf(lo[d], __shfl_xor(lo[d], m, 64));
            hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], m, 64));
        }
        if ((threadIdx.x & 63) == 0) {
            red[threadIdx.x / 64][d] = lo[d];
            red[threadIdx.x / 64][kDims + d] = hi[d];
        }
    }
    __syncthreads();
    if (threadIdx.x < 2 * kDims) {
        const int d = threadIdx.x;
        float v = red[0][d];
        for (int w = 1; w < 4; w++)
            v = d < kDims ? fminf(v, red[w][d]) : fmaxf(v, red[w][d]);
        part[d * kRangeBlocks + blockIdx.x] = v;
    }
}

// Ranges of the whole set, then the key's bits shared out by thread 0: one
// workgroup of kRangeBlocks threads.
__global__ __launch_bounds__(kRangeBlocks) void locality_bits(const float *__restrict__ part,
                                                              int nparts, LocalityState *s,
                                                              int bits)
{
    __shared__ float red[2 * kDims][kRangeBlocks / 64];
    __shared__ float range[2 * kDims];
#pragma unroll
    for (int d = 0; d < 2 * kDims; d++) {
        float v = d < kDims ? INFINITY : -INFINITY;
        if ((int)threadIdx.x < nparts)
            v = part[d * kRangeBlocks + threadIdx.x];
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const float o = __shfl_xor(v, m, 64);
            v = d < kDims ? fminf(v, o) : fmaxf(v, o);
        }
        if ((threadIdx.x & 63) == 0)
            red[d][threadIdx.x / 64] = v;
    }
    __syncthreads();
    if (threadIdx.x < 2 * kDims) {
        const int d = threadIdx.x;
        float v = red[d][0];
        for (int w = 1; w < kRangeBlocks / 64; w++)
            v = d < kDims ? fminf(v, red[d][w]) : fmaxf(v, red[d][w]);
        range[d] = v;
    }
    __syncthreads();
    if (threadIdx.x)
        return;
    float width[kDims];
    int have[kDims], dim[kMaxBits];
#pragma unroll
    for (int d = 0; d < kDims; d++) {
        width[d] = (range[kDims + d] - range[d]) * (d == 4 ? 0.25f : 1.0f);
        have[d] = 0;
    }
#pragma unroll
    for (int b = 0; b < kMaxBits; b++) {
        if (b >= bits)
            break;
        int w = 0;
        float best = width[0];
#pragma unroll
        for (int d = 1; d < kDims; d++)
            if (width[d] > best) {
                best = width[d];
                w = d;
            }
#pragma unroll
        for (int d = 0; d < kDims; d++)
            if (d == w) {
                width[d] *= 0.5f;
                dim[b] = d | (have[d] << 8); // the have-th bit of d from its top
                have[d]++;
            }
    }
#pragma unroll
    for (int d = 0; d < kDims; d++) {
        s->base[d] = range[d];
        s->scale[d] = (float)(1 << have[d]) * 0.99999f / fmaxf(range[kDims + d] - range[d], 1.0e-6f);
    }
#pragma unroll
    for (int b = 0; b < kMaxBits; b++) {
        if (b >= bits)
            break;
#pragma unroll
        for (int d = 0; d < kDims; d++)
            if ((dim[b] & 255) == d)
                s->seq[b] = d | ((have[d] - 1 - (dim[b] >> 8)) << 8);
    }
}

// Bucket of every event and the buckets' counts.
__global__ __launch_bounds__(256) void locality_count(TorParams p, int64_t K, int bits,
                                                      const LocalityState *s, int *key,
                                                      unsigned *hist)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= p.n)
        return;
    float q[kDims];
    locality_coords(p, e, q);
    int v[kDims];
#pragma unroll
    for (int d = 0; d < kDims; d++)
        v[d] = (int)((q[d] - s->base[d]) * s->scale[d]);
    int k = 0;
    for (int b = 0; b < bits; b++) {
        const int sq = s->seq[b], d = sq & 255;
        const int x = d == 0 ? v[0] : (d == 1 ? v[1] : (d == 2 ? v[2] : (d == 3 ? v[3] : v[4])));
        k = 2 * k + ((x >> (sq >> 8)) & 1);
    }
    int64_t sub = 0;
    if (K > 1) { // the subset with sub n / K <= e < (sub + 1) n / K
        sub = e * K / p.n;
        while (sub + 1 < K && (sub + 1) * p.n / K <= e)
            sub++;
        while (sub > 0 && sub * p.n / K > e)
            sub--;
    }
    k |= (int)(sub << bits);
    key[e] = k;
    atomicAdd(&hist[k], 1u);
}

// Exclusive prefix sums of the counts: workgroup b scans kScan counts and adds
// the sum of all before them, which it reads itself (64 workgroups unless the
// subsets alone take more buckets than 2^16; the counts stay in L2).
__global__ __launch_bounds__(kScan) void locality_scan(const unsigned *__restrict__ hist,
                                                       unsigned *__restrict__ first, int64_t n)
{
    const int64_t a = (int64_t)blockIdx.x * kScan;
    long long before = 0, total;
    for (int64_t i = threadIdx.x; i < a; i += kScan)
        before += hist[i];
    (void)block_scan<kScan>(before, total);
    const long long base = total;
    const int64_t i = a + threadIdx.x;
    const long long o = block_scan<kScan>(i < n ? (long long)hist[i] : 0ll, total);
    if (i < n)
        first[i] = (unsigned)(base + o);
}

__global__ __launch_bounds__(256) void locality_place(int64_t n, LocalityOrder o, int *place)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n)
        place[e] = (int)atomicAdd(&o.cursor[o.key[e]], 1u);
}

// Key bits of a subset: about eight events a bucket, at most 2^16 buckets in all
// unless the subsets alone take more.
int key_bits(int64_t n, int64_t K)
{
    int b = 0;
    while (b < kMaxBits && (K << (b + 1)) <= ((int64_t)1 << kMaxBits) &&
           (K << (b + 4)) <= n)
        b++;
    return b;
}

} // namespace

size_t locality_bytes(int64_t n, int64_t K)
{
    return align256(sizeof(LocalityState)) + align256(sizeof(float) * 2 * kDims * kRangeBlocks) +
           2 * align256(sizeof(unsigned) * (size_t)(K << key_bits(n, K))) +
           align256(sizeof(int) * (size_t)n);
}

int locality_order(const TorParams &p, int64_t K, LocalityOrder &order, char *ws, hipStream_t st)
{
    const int bits = key_bits(p.n, K);
    const int64_t nh = K << bits;
    auto *s = (LocalityState *)ws;
    auto *part = (float *)(ws + align256(sizeof(LocalityState)));
    auto *hist = (unsigned *)((char *)part + align256(sizeof(float) * 2 * kDims * kRangeBlocks));
    auto *first = (unsigned *)((char *)hist + align256(sizeof(unsigned) * (size_t)nh));
    auto *key = (int *)((char *)first + align256(sizeof(unsigned) * (size_t)nh));
    const dim3 eb(blocks_for(p.n, 256)), b(256);
    const int parts = (int)std::min(eb.x, (unsigned)kRangeBlocks);
    hipLaunchKernelGGL(locality_range, dim3(parts), b, 0, st, p, part, hist, nh);
    hipLaunchKernelGGL(locality_bits, dim3(1), dim3(kRangeBlocks), 0, st, part, parts, s, bits);
    hipLaunchKernelGGL(locality_count, eb, b, 0, st, p, K, bits, s, key, hist);
    hipLaunchKernelGGL(locality_scan, dim3((unsigned)((nh + kScan - 1) / kScan)), dim3(kScan), 0,
                       st, hist, first, nh);
    order = LocalityOrder{key, first};
    return launch_status();
}

int locality_places(const TorParams &p, int64_t K, int *place, char *ws, hipStream_t st)
{
    LocalityOrder o;
    const int rc = locality_order(p, K, o, ws, st);
    if (rc)
        return rc;
    hipLaunchKernelGGL(locality_place, dim3(blocks_for(p.n, 256)), dim3(256), 0, st, p.n, o, place);
    return launch_status();
}

} // namespace srfx
