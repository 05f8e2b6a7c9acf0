// Counting sort of one chunk of a tile's list by the length of its entries'
// walks, longest first (plan builds and the binned scatters).
#pragma once

#include "common.h"

namespace srfx {
namespace {

constexpr int kSortBuckets = 32;

// The lanes of the wave whose v (0 <= v < 64) equals this lane's: one ballot
// per bit of v.  Call with every lane of the wave active.
__device__ __forceinline__ uint64_t lanes_with(int v)
{
    uint64_t m = ~0ull;
#pragma unroll
    for (int b = 0; b < 6; b++) {
        const bool bit = (v >> b) & 1;
        const uint64_t bal = __ballot(bit);
        m &= bit ? bal : ~bal;
    }
    return m;
}

// Order list[0..count) by length(entry), longest first, lengths of 31 and more
// together.  Inside a bucket the entries keep their order within a wave and the
// waves their order of arrival, which with coalesced reads keeps roughly the
// given order.  The lanes of a wave with the same key count and take their
// positions together: one LDS atomic per key and wave, the lowest such lane's,
// instead of one per lane on a few shared counters.  One workgroup of 256
// threads; sh: kSortBuckets + 1 counters and count ints; count <= 16 * 256.
template <class F>
__device__ __forceinline__ void chunk_sort(int *__restrict__ list, int count, int *sh, F length)
{
    constexpr int kPer = 16;
    int *cnt = sh, *ord = sh + kSortBuckets + 1;
    const int lane = (int)threadIdx.x & 63;
    for (int i = threadIdx.x; i <= kSortBuckets; i += blockDim.x)
        cnt[i] = 0;
    __syncthreads();
    // per entry: its key (-1: no entry), value, and its rank among the wave's
    // lanes with the same key | the first such lane << 6 | their number << 12
    int key[kPer], ent[kPer], grp[kPer];
#pragma unroll
    for (int r = 0; r < kPer; r++) {
        key[r] = -1;
        ent[r] = 0;
        grp[r] = 0;
        if (r * (int)blockDim.x >= count)
            continue; // the same for every lane of the workgroup
        const int j = r * (int)blockDim.x + (int)threadIdx.x; // coalesced reads
        if (j < count) {
            ent[r] = list[j];
            // longest first: bucket 0 holds the longest walks
            key[r] = kSortBuckets - 1 - min(max(length(ent[r]), 0), kSortBuckets - 1);
        }
        const uint64_t m = lanes_with(key[r] + 1);
        const int rank = (int)__builtin_amdgcn_mbcnt_hi(
            (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
        const int n = __popcll(m);
        grp[r] = rank | (__builtin_ctzll(m) << 6) | (n << 12);
        if (key[r] >= 0 && rank == 0)
            atomicAdd(&cnt[key[r]], n);
    }
    __syncthreads();
    // exclusive prefix of the bucket counts, by the first wave
    if (threadIdx.x < 64) {
        const int c = lane < kSortBuckets ? cnt[lane] : 0;
        int v = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int u = __shfl_up(v, d, 64);
            v += lane >= d ? u : 0;
        }
        if (lane < kSortBuckets)
            cnt[lane] = v - c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPer; r++) {
        if (r * (int)blockDim.x >= count)
            continue;
        const int rank = grp[r] & 63;
        int base = 0;
        if (key[r] >= 0 && rank == 0)
            base = atomicAdd(&cnt[key[r]], grp[r] >> 12);
        base = __shfl(base, (grp[r] >> 6) & 63, 64);
        if (key[r] >= 0)
            ord[base + rank] = ent[r];
    }
    __syncthreads();
    for (int j = threadIdx.x; j < count; j += blockDim.x)
        list[j] = ord[j];
}

} // namespace
} // namespace srfx
