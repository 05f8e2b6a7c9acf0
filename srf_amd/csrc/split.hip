// LOR preprocessing on the device (srf_amd/preprocess.py): list-mode rows split
// into the TOR model's axis groups, and a group's events put in locality order.
//
// The split follows preprocess/function/on_tor_lors.py:70-77 (dominant axis),
// 137-166 (sigma2 factor), 175-193 (SwapPointsOrder), 196-229 (CutLoRs) and
// 243-262 (column orders) in FP64 with its order of operations, every product
// and sum rounded on its own, so that the results are those of the numpy
// restatement bit for bit.  As elementwise tensor operations it took ~90 passes
// over the rows and a host synchronisation per group and sign: 2.1 ms for 1M
// rows, 12.1 for 8M; here the rows are read twice and every output is written
// once, with one synchronisation for the group sizes: 0.063 and 0.35 ms.  The
// locality order of 1M events in 4 subsets, a stable sort per subset and a
// gather per column before, is one radix sort and one gather: 2.8 -> 0.57 ms.
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "common.h"

namespace srfx {
namespace {

constexpr int kSplitRows = 1024; // rows of a workgroup, in 4 rounds of 256
constexpr int kCats = 6;         // axis * 2 + swapped

struct SplitRows {
    const void *rows;
    int64_t n, rs, cs; // rows and their strides in elements
    int f64;
    __device__ __forceinline__ double at(int64_t e, int c) const
    {
        const int64_t i = e * rs + c * cs;
        return f64 ? ((const double *)rows)[i] : (double)((const float *)rows)[i];
    }
};

// Category of a row: its dominant axis (x on ties with y or z, y on ties with
// z; -1 for NaN differences), and whether its end points are swapped.
__device__ __forceinline__ int category(const double (&p)[6])
{
    const double dx = __dsub_rn(p[3], p[0]), dy = __dsub_rn(p[4], p[1]), dz = __dsub_rn(p[5], p[2]);
    const double ax = fabs(dx), ay = fabs(dy), az = fabs(dz);
    if (ax >= ay && ax >= az)
        return dx >= 0.0 ? 0 : 1;
    if (ay > ax && ay >= az)
        return dy >= 0.0 ? 2 : 3;
    if (az > ax && az > ay)
        return dz >= 0.0 ? 4 : 5;
    return -1;
}

// The workgroup's rows by category: counts of every (round, wave), and each of
// this thread's rows' category and rank among its wave's rows of it.
__device__ __forceinline__ void classify(const SplitRows &s, int (&cat)[4], int (&rank)[4],
                                         int (*cnt)[4][kCats])
{
    const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int64_t e = (int64_t)blockIdx.x * kSplitRows + r * 256 + threadIdx.x;
        cat[r] = -1;
        rank[r] = 0;
        if (e < s.n) {
            double p[6];
#pragma unroll
            for (int c = 0; c < 6; c++)
                p[c] = s.at(e, c);
            cat[r] = category(p);
        }
#pragma unroll
        for (int c = 0; c < kCats; c++) {
            const uint64_t m = __ballot(cat[r] == c);
            if (cat[r] == c)
                rank[r] = (int)__builtin_amdgcn_mbcnt_hi(
                    (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            if (lane == 0)
                cnt[r][wv][c] = __popcll(m);
        }
    }
    __syncthreads();
}

// work[c * nblocks + b] = rows of category c in workgroup b.
__global__ __launch_bounds__(256) void split_count(SplitRows s, int *work)
{
    __shared__ int cnt[4][4][kCats];
    int cat[4], rank[4];
    classify(s, cat, rank, cnt);
    if (threadIdx.x < kCats) {
        int t = 0;
        for (int r = 0; r < 4; r++)
            for (int w = 0; w < 4; w++)
                t += cnt[r][w][threadIdx.x];
        work[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = t;
    }
}

// Exclusive prefix of each category's counts over the workgroups, and the
// totals.  One workgroup per category.
__global__ __launch_bounds__(1024) void split_scan(int *work, int nblocks, int64_t *totals)
{
    int *w = work + (int64_t)blockIdx.x * nblocks;
    long long carry = 0;
    for (int b0 = 0; b0 < nblocks; b0 += 1024) {
        const int b = b0 + (int)threadIdx.x;
        long long total;
        const long long ex = carry + block_scan<1024>(b < nblocks ? w[b] : 0, total);
        if (b < nblocks)
            w[b] = (int)ex;
        carry += total;
    }
    if (threadIdx.x == 0)
        totals[blockIdx.x] = carry;
}

struct SplitOut {
    float *out[3];     // [ncols][ld] of each group
    int64_t ld[3];
    int64_t *order[3]; // input row of each output row (nullable)
};

// on_tor_lors.py:137-166 of the row as it came.
__device__ __forceinline__ double sigma2_factor(const double (&p)[6])
{
    const double dx = __dsub_rn(p[3], p[0]), dy = __dsub_rn(p[4], p[1]), dz = __dsub_rn(p[5], p[2]);
    const double xy = __dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy));
    const double d2 = __dadd_rn(xy, __dmul_rn(dz, dz));
    const double rsq =
        __dadd_rn(__dadd_rn(__dadd_rn(__dmul_rn(p[0], p[0]), __dmul_rn(p[3], p[3])),
                            __dmul_rn(p[1], p[1])),
                  __dmul_rn(p[4], p[4]));
    return __dmul_rn(__ddiv_rn(__ddiv_rn(__dmul_rn(xy, xy), rsq), d2), 0.5);
}

// TOF: seven input columns, ten output rows (end points cut to centre +- limit
// where cut and the centre lies further than that from p1); else six and seven.
template <bool TOF>
__global__ __launch_bounds__(256) void split_fill(SplitRows s, const int *__restrict__ work,
                                                  const int64_t *__restrict__ totals, int cut,
                                                  double limit, SplitOut o)
{
    __shared__ int cnt[4][4][kCats];
    int cat[4], rank[4];
    classify(s, cat, rank, cnt);
    if (threadIdx.x < kCats) { // counts -> first output row of each (round, wave)
        int64_t t = work[(int64_t)threadIdx.x * gridDim.x + blockIdx.x];
        if (threadIdx.x & 1) // swapped rows follow the group's others
            t += totals[threadIdx.x - 1];
        for (int r = 0; r < 4; r++)
            for (int w = 0; w < 4; w++) {
                const int c = cnt[r][w][threadIdx.x];
                cnt[r][w][threadIdx.x] = (int)t;
                t += c;
            }
    }
    __syncthreads();
    const int wv = (int)threadIdx.x >> 6;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (cat[r] < 0)
            continue;
        const int64_t e = (int64_t)blockIdx.x * kSplitRows + r * 256 + threadIdx.x;
        const int a = cat[r] >> 1;
        const bool swap = cat[r] & 1;
        const int64_t q = cnt[r][wv][cat[r]] + rank[r];
        double p[6];
#pragma unroll
        for (int c = 0; c < 6; c++)
            p[c] = s.at(e, c);
        const double f = sigma2_factor(p);
        double p0[3], p1[3], ctr[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            p0[c] = swap ? p[3 + c] : p[c];
            p1[c] = swap ? p[c] : p[3 + c];
        }
        if (TOF) {
            double t = s.at(e, 6);
            t = swap ? __dsub_rn(0.0, t) : t;
            double d[3];
#pragma unroll
            for (int c = 0; c < 3; c++)
                d[c] = __dsub_rn(p1[c], p0[c]);
            const double L = __dsqrt_rn(
                __dadd_rn(__dadd_rn(__dmul_rn(d[0], d[0]), __dmul_rn(d[1], d[1])),
                          __dmul_rn(d[2], d[2])));
            const double ratio = __dsub_rn(0.5, __ddiv_rn(t, L));
            double g[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                ctr[c] = __dadd_rn(__dmul_rn(ratio, d[c]), p0[c]);
                g[c] = __dsub_rn(ctr[c], p0[c]);
            }
            const double far = __dsqrt_rn(
                __dadd_rn(__dadd_rn(__dmul_rn(g[0], g[0]), __dmul_rn(g[1], g[1])),
                          __dmul_rn(g[2], g[2])));
            if (cut && far > limit) {
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const double u = __dmul_rn(limit, __ddiv_rn(d[c], L));
                    p0[c] = __dsub_rn(ctr[c], u);
                    p1[c] = __dadd_rn(ctr[c], u);
                }
            }
        }
        // op x, y, z of the group: world y, z, x for x; x, z, y for y; x, y, z
        const int ox = a == 0 ? 1 : 0, oy = a == 2 ? 1 : 2, oz = a == 0 ? 0 : (a == 1 ? 1 : 2);
        auto pick = [](const double (&v)[3], int c) {
            return (float)(c == 0 ? v[0] : (c == 1 ? v[1] : v[2]));
        };
        float *out = (a == 0 ? o.out[0] : (a == 1 ? o.out[1] : o.out[2])) + q;
        const int64_t ld = a == 0 ? o.ld[0] : (a == 1 ? o.ld[1] : o.ld[2]);
        out[0] = pick(p0, ox);
        out[ld] = pick(p0, oy);
        out[2 * ld] = pick(p0, oz);
        out[3 * ld] = pick(p1, ox);
        out[4 * ld] = pick(p1, oy);
        out[5 * ld] = pick(p1, oz);
        if (TOF) {
            out[6 * ld] = pick(ctr, ox);
            out[7 * ld] = pick(ctr, oy);
            out[8 * ld] = pick(ctr, oz);
            out[9 * ld] = (float)f;
        } else {
            out[6 * ld] = (float)f;
        }
        int64_t *ord = a == 0 ? o.order[0] : (a == 1 ? o.order[1] : o.order[2]);
        if (ord)
            ord[q] = e;
    }
}

// -------------------------------------------------------- locality order ---

// Bit i of the low 8 bits of v to bit 4 i.
__device__ __forceinline__ unsigned spread8(unsigned v)
{
    v = (v | (v << 12)) & 0x000f000fu;
    v = (v | (v << 6)) & 0x03030303u;
    return (v | (v << 3)) & 0x11111111u;
}

// floor(v inv) + 128 within 0 .. 255 (NaN: 0), v / step as v times 1 / step.
__device__ __forceinline__ unsigned quantum(double v, double inv, double off, double top)
{
    const double q = __dadd_rn(floor(__dmul_rn(v, inv)), off);
    return q >= 0.0 ? (unsigned)fmin(q, top) : 0u;
}

// Sort key of event i of a [>= 9, n] group: OSEM subset, then coarse TOF-centre
// position along the slice axis, then the Morton interleave of the two slopes
// and the crossing with the plane z = center_z.
__global__ __launch_bounds__(256) void locality_keys(const float *__restrict__ soa, int64_t n,
                                                     int64_t ld, int64_t K, double cz,
                                                     double zc_inv, double slope_inv,
                                                     double pos_inv, unsigned long long *keys,
                                                     int *idx)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const double x1 = soa[i], y1 = soa[ld + i], z1 = soa[2 * ld + i];
    const double dx = __dsub_rn((double)soa[3 * ld + i], x1);
    const double dy = __dsub_rn((double)soa[4 * ld + i], y1);
    double dz = __dsub_rn((double)soa[5 * ld + i], z1);
    dz = dz == 0.0 ? 1e-12 : dz;
    const double sx = __ddiv_rn(dx, dz), sy = __ddiv_rn(dy, dz), w = __dsub_rn(cz, z1);
    const double X0 = __dadd_rn(x1, __dmul_rn(sx, w)), Y0 = __dadd_rn(y1, __dmul_rn(sy, w));
    const unsigned zc = quantum((double)soa[8 * ld + i], zc_inv, 64.0, 127.0);
    const unsigned m = spread8(quantum(sx, slope_inv, 128.0, 255.0)) |
                       (spread8(quantum(sy, slope_inv, 128.0, 255.0)) << 1) |
                       (spread8(quantum(X0, pos_inv, 128.0, 255.0)) << 2) |
                       (spread8(quantum(Y0, pos_inv, 128.0, 255.0)) << 3);
    // the subset of row i: the k with (k n) / K <= i < ((k + 1) n) / K
    int64_t k = i * K / n;
    while (k + 1 < K && (k + 1) * n / K <= i)
        k++;
    while (k > 0 && k * n / K > i)
        k--;
    keys[i] = ((unsigned long long)k << 39) | ((unsigned long long)zc << 32) | m;
    idx[i] = (int)i;
}

__global__ __launch_bounds__(256) void take_columns(const float *__restrict__ soa, int64_t n,
                                                    int64_t ld, int ncols,
                                                    const int *__restrict__ idx,
                                                    float *__restrict__ out, int64_t *order)
{
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n)
        return;
    const int64_t i = idx[j];
    order[j] = i;
    if (out)
        for (int c = 0; c < ncols; c++)
            out[c * n + j] = soa[c * ld + i];
}

} // namespace
} // namespace srfx

using namespace srfx;

extern "C" int srfx_split_lors_count(const void *rows, int64_t n, int64_t row_stride,
                                     int64_t col_stride, int32_t f64, int32_t *work,
                                     int64_t *totals, void *stream)
{
    if (n < 1 || n > (int64_t)INT32_MAX || !rows || !work || !totals || row_stride < 0 ||
        col_stride < 0)
        return SRFX_EINVAL;
    const SplitRows s{rows, n, row_stride, col_stride, f64 ? 1 : 0};
    const int nb = (int)((n + kSplitRows - 1) / kSplitRows);
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(split_count, dim3(nb), dim3(256), 0, st, s, work);
    hipLaunchKernelGGL(split_scan, dim3(kCats), dim3(1024), 0, st, work, nb, totals);
    return launch_status();
}

extern "C" int srfx_split_lors_fill(const void *rows, int64_t n, int64_t row_stride,
                                    int64_t col_stride, int32_t f64, int32_t ncols, int32_t cut,
                                    double limit, const int32_t *work, const int64_t *totals,
                                    float *const *out, const int64_t *ld, int64_t *const *order,
                                    void *stream)
{
    if (n < 1 || n > (int64_t)INT32_MAX || !rows || !work || !totals || !out || !ld ||
        row_stride < 0 || col_stride < 0 || (ncols != 6 && ncols != 7))
        return SRFX_EINVAL;
    const SplitRows s{rows, n, row_stride, col_stride, f64 ? 1 : 0};
    SplitOut o{};
    for (int a = 0; a < 3; a++) {
        o.out[a] = out[a];
        o.ld[a] = ld[a];
        o.order[a] = order ? order[a] : nullptr;
    }
    const dim3 grid((unsigned)((n + kSplitRows - 1) / kSplitRows));
    hipStream_t st = (hipStream_t)stream;
    if (ncols == 7)
        hipLaunchKernelGGL(split_fill<true>, grid, dim3(256), 0, st, s, work, totals, cut, limit,
                           o);
    else
        hipLaunchKernelGGL(split_fill<false>, grid, dim3(256), 0, st, s, work, totals, 0, 0.0, o);
    return launch_status();
}

extern "C" int srfx_locality_sort(const float *soa, int64_t n, int64_t ld, int32_t ncols,
                                  int32_t nb_subsets, double center_z, double zc_bin,
                                  double slope_bin, double pos_bin, float *out, int64_t *order,
                                  void *stream)
{
    if (n < 1 || n > (int64_t)INT32_MAX - 1 || ld < n || ncols < 9 || nb_subsets < 1 ||
        nb_subsets > (1 << 24) || !soa || !order)
        return SRFX_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    const int bits = 39 + std::max(1, 32 - __builtin_clz((unsigned)nb_subsets));
    size_t tmp = 0;
    if (hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, (unsigned long long *)nullptr,
                                           (unsigned long long *)nullptr, (int *)nullptr,
                                           (int *)nullptr, (int)n, 0, bits, st) != hipSuccess)
        return SRFX_ELAUNCH;
    const size_t kb = align256(sizeof(unsigned long long) * (size_t)n);
    const size_t ib = align256(sizeof(int) * (size_t)n);
    char *ws = nullptr;
    int rc = ws_alloc((void **)&ws, 2 * kb + 2 * ib + tmp, st);
    if (rc)
        return rc;
    auto *k0 = (unsigned long long *)ws, *k1 = (unsigned long long *)(ws + kb);
    auto *i0 = (int *)(ws + 2 * kb), *i1 = (int *)(ws + 2 * kb + ib);
    const dim3 grid(blocks_for(n, 256)), block(256);
    hipLaunchKernelGGL(locality_keys, grid, block, 0, st, soa, n, ld, (int64_t)nb_subsets,
                       center_z, 1.0 / zc_bin, 1.0 / slope_bin, 1.0 / pos_bin, k0, i0);
    rc = launch_status();
    if (!rc && hipcub::DeviceRadixSort::SortPairs(ws + 2 * kb + 2 * ib, tmp, k0, k1, i0, i1,
                                                  (int)n, 0, bits, st) != hipSuccess)
        rc = SRFX_ELAUNCH;
    if (!rc) {
        hipLaunchKernelGGL(take_columns, grid, block, 0, st, soa, n, ld, ncols, i1, out, order);
        rc = launch_status();
    }
    const int rf = ws_free(ws, st);
    return rc ? rc : rf;
}
