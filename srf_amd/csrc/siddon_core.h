// Siddon ray setup and walk shared by the untiled kernels (siddon.hip) and
// the tiled backprojection (siddon_tile.hip).
//
// Semantics follow the reference CUDA op src/cpp/tf_custom_ops/siddon.cu.cc
// (CreateRay 61-81, ClipRay / IsThroughImage 118-183, SetupRayCast 196-284,
// RayTracing / BackRayTracing / Map 293-415).  Ray geometry (clip, start voxel,
// first crossings) is formed in FP64 with explicitly rounded operations in the
// reference's source order, so a ray enters through the voxel of the FP64
// restatement, also where it lies exactly on a voxel face.  The count follows the
// reference's traversal step by step (nextT updates, argmin); the other walks form
// crossing k of an axis as n + k t (spans, below), whose segments are the
// traversal's up to the rounding of that product.  Segment lengths, TOF distance and
// variance are FP64; weights (1/L^2, the TOF Gaussian) and the accumulation are
// FP32.
#pragma once

#include <float.h>
#include <math.h>

#include "common.h"

namespace srfx {
namespace {

enum SidMode { kProj = 0, kBack = 1, kMap = 2, kAdj = 3, kCount = 4, kOsem = 5 };

} // namespace

struct SidParams {
    const float *__restrict__ lors;
    int64_t n, ld;
    const float *__restrict__ val;
    const float *__restrict__ img;
    float *out;
    int32_t *nnz;
    unsigned long long *nnz_total;
    int g[3];
    float size[3], center[3];
    int s[3]; // read-image strides
    int o[3]; // written-image strides
    float tof_bin, tof_sigma2;
    int use_tof;
};

namespace {

struct Walk {
    double nextT[3], deltaT[3];
    int inBuf[3], step[3];
    int pos[3];
    float weight;
    double t_tof;
    bool ok;
};

// Ray setup: CreateRay, IsThroughImage, SetupRayCast and the weight / TOF
// origin of project() (siddon.cu.cc:450-460).
template <int MODE>
__device__ __forceinline__ void setup_walk(const SidParams &p, int64_t e, Walk &w)
{
    const float *L = p.lors;
    const int64_t ld = p.ld;
    double P0[3], D[3];
    P0[0] = __builtin_nontemporal_load(L + 0 * ld + e);
    P0[1] = __builtin_nontemporal_load(L + 1 * ld + e);
    P0[2] = __builtin_nontemporal_load(L + 2 * ld + e);
    double x2 = __builtin_nontemporal_load(L + 3 * ld + e);
    double y2 = __builtin_nontemporal_load(L + 4 * ld + e);
    double z2 = __builtin_nontemporal_load(L + 5 * ld + e);
    double dx = x2 - P0[0], dy = y2 - P0[1], dz = z2 - P0[2]; // exact
    double length =
        __dsqrt_rn(__dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz)));
    D[0] = __ddiv_rn(dx, length);
    D[1] = __ddiv_rn(dy, length);
    D[2] = __ddiv_rn(dz, length);
    if (MODE == kMap)
        w.weight = (float)(1.0 / (length * length));
    else
        w.weight = (float)(1.0 / length / length);
    w.ok = false;
    // IsThroughImage / ClipRay
    double tmin = 0.0, tmax = length;
    for (int c = 0; c < 3; c++) {
        double half = (double)p.size[c] / 2;
        double top = __dadd_rn((double)p.center[c], half);
        double bot = __dsub_rn((double)p.center[c], half);
        double p0 = P0[c], dp = D[c];
        if (dp > 0.0) {
            double t = __ddiv_rn(__dsub_rn(top, p0), dp);
            if (t < tmax)
                tmax = t;
            t = __ddiv_rn(__dsub_rn(bot, p0), dp);
            if (t > tmin)
                tmin = t;
        } else if (dp < 0.0) {
            double t = __ddiv_rn(__dsub_rn(bot, p0), dp);
            if (t < tmax)
                tmax = t;
            t = __ddiv_rn(__dsub_rn(top, p0), dp);
            if (t > tmin)
                tmin = t;
        } else {
            if ((p0 < bot) || (p0 > top))
                return;
        }
        if (!(tmin < tmax))
            return;
    }
    // SetupRayCast: origin at the box corner, per-axis start voxel.
    for (int c = 0; c < 3; c++) {
        double p0 =
            __dsub_rn(P0[c], __dsub_rn((double)p.center[c], (double)p.size[c] / 2));
        double dir = D[c];
        double pt = __dadd_rn(__dmul_rn(tmin, dir), p0);
        double v_res = __ddiv_rn((double)p.size[c], (double)p.g[c]);
        int vc = p.g[c];
        int pos;
        if (dir > 0.0) {
            pos = (int)__ddiv_rn(pt, v_res);
            w.nextT[c] = __ddiv_rn(__dsub_rn(__dmul_rn((double)(pos + 1), v_res), pt), dir);
            w.deltaT[c] = __ddiv_rn(v_res, dir);
            w.step[c] = 1;
            w.inBuf[c] = vc - pos;
        } else if (dir < 0.0) {
            pos = vc - 1 - (int)__dsub_rn((double)vc, __ddiv_rn(pt, v_res));
            w.nextT[c] = __ddiv_rn(__dsub_rn(__dmul_rn((double)pos, v_res), pt), dir);
            w.deltaT[c] = __ddiv_rn(-v_res, dir);
            w.step[c] = -1;
            w.inBuf[c] = pos + 1;
        } else {
            pos = (int)__ddiv_rn(pt, v_res);
            w.nextT[c] = DBL_MAX;
            w.deltaT[c] = DBL_MAX;
            w.step[c] = 0;
            w.inBuf[c] = 1;
        }
        if (pos < 0 || pos >= vc)
            return;
        w.pos[c] = pos;
    }
    if (MODE != kMap) {
        double tof = __builtin_nontemporal_load(L + 6 * ld + e);
        w.t_tof = __dsub_rn(__dsub_rn(__dmul_rn(length, 0.5), tmin), tof);
    } else {
        w.t_tof = 0.0;
    }
    w.ok = true;
}

// Value of the segment (last_t, nt] of a ray, the reference's per-voxel
// factor of RayTracing / BackRayTracing (siddon.cu.cc:303-322): l / L^2,
// times the TOF Gaussian when TOF is on.  Returns false when the TOF test
// (t^2 / sigma^2 < 9) drops the segment.
template <bool TOF>
__device__ __forceinline__ bool seg_value(const SidParams &p, float weight, double t_tof,
                                          double nt, double last_t, float &g)
{
    const double l_d = __dsub_rn(nt, last_t);
    const float l_len = (float)l_d;
    if (TOF) {
        const double bs2 = (double)p.tof_bin * (double)p.tof_bin;
        double t = __dsub_rn(t_tof, __dmul_rn(0.5, __dadd_rn(nt, last_t)));
        double sigma2 = __dadd_rn((double)p.tof_sigma2,
                                  __ddiv_rn(__dadd_rn(__dmul_rn(l_d, l_d), bs2), 12.0));
        double tt = __ddiv_rn(__dmul_rn(t, t), sigma2);
        if (!(tt < 9.0))
            return false;
        // bin * exp(-t2/2) / sqrt(2 pi sigma2)
        g = weight * l_len * p.tof_bin * __expf(-0.5f * (float)tt) *
            __frsqrt_rn(6.283185307179586f * (float)sigma2);
        return true;
    }
    g = weight * l_len;
    return true;
}

// The number of non-zero segments of a ray: the reference's walk step by step
// (RayTracing, siddon.cu.cc:293-331).
template <bool TOF>
__device__ __forceinline__ int count_segments(const SidParams &p, const Walk &w)
{
    double n0 = w.nextT[0], n1 = w.nextT[1], n2 = w.nextT[2];
    const double t0 = w.deltaT[0], t1 = w.deltaT[1], t2 = w.deltaT[2];
    int b0 = w.inBuf[0], b1 = w.inBuf[1], b2 = w.inBuf[2];
    double last_t = 0.0;
    int count = 0;
    int stillin = b0 * b1 * b2;
    int cap = p.g[0] + p.g[1] + p.g[2] + 3;
    while (stillin && cap-- > 0) {
        int i = (n0 <= n1) ? ((n0 <= n2) ? 0 : 2) : ((n1 <= n2) ? 1 : 2);
        double nt = i == 0 ? n0 : (i == 1 ? n1 : n2);
        float g;
        if (seg_value<TOF>(p, w.weight, w.t_tof, nt, last_t, g))
            count += (__dsub_rn(nt, last_t) > 0.0);
        last_t = nt;
        if (i == 0) {
            n0 = __dadd_rn(nt, t0);
            stillin = --b0;
        } else if (i == 1) {
            n1 = __dadd_rn(nt, t1);
            stillin = --b1;
        } else {
            n2 = __dadd_rn(nt, t2);
            stillin = --b2;
        }
    }
    return count;
}

// ------------------------------------------------------------------- spans ---
//
// The walks of the ops.  The reference's walk is a chain: every step picks the
// nearest of three crossings, and its 171 dependent, divergent steps a ray (62
// VALU instructions each) left the chip waiting.  The k-th crossing of an axis
// is at n + k t, so a walk can start anywhere.  A span walk goes from plane to
// plane of the ray's dominant axis (the smallest t): between two of its planes
// every other axis is crossed at most once, so a slab holds at most three
// segments, cut by the two crossings in order.  That is 43 branch-free
// instructions for 2.1 segments on average, and a ray can be shared by several
// lanes and started at a tile's face.  The segments are those of the
// reference's walk up to the rounding of n + k t (the reference adds t k times;
// both stay within ~1e-13 of the exact crossing), which moves less than 1e-12
// of a segment's length to its neighbour.

// A ray by its crossings: time (length along the ray from its entry) n[c] + k
// t[c] of the k-th crossing of axis c, start voxel, step signs, exit time.
struct SidRay {
    double n[3], t[3];
    double tend, t_tof; // tend <= 0: the ray misses the image
    int pos[3], step[3];
    float weight;
};

__device__ __forceinline__ double cross_time(double n, double t, double k)
{
    return fma(k, t, n);
}

__device__ __forceinline__ void make_ray(const Walk &w, SidRay &r)
{
    double tend = DBL_MAX;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        r.n[c] = w.nextT[c];
        r.t[c] = w.deltaT[c];
        r.pos[c] = w.pos[c];
        r.step[c] = w.step[c];
        // the crossing that leaves the image: inBuf[c] - 1 more before it
        tend = fmin(tend, cross_time(w.nextT[c], w.deltaT[c], (double)(w.inBuf[c] - 1)));
    }
    r.tend = w.ok ? tend : -1.0;
    r.t_tof = w.t_tof;
    r.weight = w.weight;
}

// A ray's axes ordered for a span walk: d the dominant one, y and z the others
// in their own order.
struct SidAxes {
    double nd, td, ny, ty, nz, tz;
    int d;
};

__device__ __forceinline__ SidAxes ray_axes(const SidRay &r)
{
    SidAxes a;
    a.d = r.t[1] < r.t[0] ? 1 : 0;
    a.d = r.t[2] < (a.d ? r.t[1] : r.t[0]) ? 2 : a.d;
    const bool d0 = a.d == 0, d2 = a.d == 2;
    a.nd = d0 ? r.n[0] : (d2 ? r.n[2] : r.n[1]);
    a.td = d0 ? r.t[0] : (d2 ? r.t[2] : r.t[1]);
    a.ny = d0 ? r.n[1] : r.n[0];
    a.ty = d0 ? r.t[1] : r.t[0];
    a.nz = d2 ? r.n[1] : r.n[2];
    a.tz = d2 ? r.t[1] : r.t[2];
    return a;
}

// v[d], v[y], v[z] of a per-axis value.
__device__ __forceinline__ void by_axes(const SidAxes &a, const int (&v)[3], int &vd, int &vy,
                                        int &vz)
{
    vd = a.d == 0 ? v[0] : (a.d == 2 ? v[2] : v[1]);
    vy = a.d == 0 ? v[1] : v[0];
    vz = a.d == 2 ? v[1] : v[2];
}

// Elements of the voxels a walk visits, in a strided image or LDS tile: element
// of the current slab's first voxel and the signed strides of one crossing.
struct SpanIndex {
    int off, sd, sy, sz;

    // s: strides; base: element of the ray's start voxel; kd, ky, kz: crossings
    // before the walk
    __device__ __forceinline__ SpanIndex(const SidRay &r, const SidAxes &a, const int (&s)[3],
                                           int base, int kd, int ky, int kz)
    {
        const int q[3] = {r.step[0] * s[0], r.step[1] * s[1], r.step[2] * s[2]};
        by_axes(a, q, sd, sy, sz);
        off = base + kd * sd + ky * sy + kz * sz;
    }
    // the slab's three voxels: crossed y / z (cy, cz), y first (yf)
    __device__ __forceinline__ void slab(bool cy, bool cz, bool yf, int &o0, int &o1, int &o2)
    {
        const int da = cy ? sy : 0, db = cz ? sz : 0;
        o0 = off;
        o1 = off + (yf ? da : db);
        o2 = off + da + db;
        off = o2 + sd;
    }
};

// a / b to ~2^-48 relative: v_rcp_f64 (below 2^-24) and one Newton step, a sixth of a
// division's instructions.
__device__ __forceinline__ double quotient(double a, double b)
{
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    return a * r;
}

// Crossings of an axis before time T, within [lo, hi].  A crossing at T itself
// may fall on either side: the segment it would cut has no length.  The
// quotient's relative error matters as little: it can only misplace a crossing
// that close to T, by that much.
__device__ __forceinline__ int crossings(double n, double t, double T, int lo, int hi)
{
    const double k = ceil(quotient(T - n, t));
    return k >= (double)hi ? hi : max(lo, (int)fmax(k, -1.0));
}

// Value of the segment [ta, tb] as seg_value's: distance, variance and their
// quotient in FP64, rounded once; the division itself where the quotient lies at
// the TOF test's bound.  (In FP32 the values are 1.56e-7 from 64 bits, root mean
// square, instead of 1.08e-7; a projection and a backprojection of 100k TOF rays,
// 128 x 128 x 64, take 200 us in FP32 and 204.5 here.)  Without TOF the ray's
// weight is left to the caller.
template <bool TOF>
__device__ __forceinline__ float span_value(const SidParams &p, const SidRay &r, double ta,
                                            double tb)
{
    const double ld = tb - ta;
    const float l = (float)ld;
    if (!TOF)
        return l;
    // the fused steps written out: every kernel forms the same bits
    const double t = fma(-0.5, ta + tb, r.t_tof);
    const double bs2 = (double)p.tof_bin * (double)p.tof_bin;
    const double s2 = fma(fma(ld, ld, bs2), 1.0 / 12.0, (double)p.tof_sigma2);
    const double tt = quotient(t * t, s2);
    bool in = tt < 9.0;
    if (fabs(tt - 9.0) < 1.0e-10) {
        float g;
        in = seg_value<true>(p, r.weight, r.t_tof, tb, ta, g);
    }
    return in ? l * (__expf(-0.5f * (float)tt) * __frsqrt_rn(6.283185307179586f * (float)s2)) : 0.0f;
}

// What a span walk's values are to be multiplied by.
template <bool TOF>
__device__ __forceinline__ float span_factor(const SidParams &p, const SidRay &r)
{
    return TOF ? r.weight * p.tof_bin : r.weight;
}

// Walk the ray from time ta to tb (times of crossings, or its ends), kd, ky and
// kz crossings of the axes lying before ta; ix is the index of the voxel there.
// f is called once a slab with the elements and values of its three segments, a
// value <= 0 for one that does not exist (its element is then still one the
// walk visits).  A crossing is taken only before tb, so the elements stay
// inside whatever the crossings at or after tb leave.
template <bool TOF, class F>
__device__ __forceinline__ void walk_span(const SidParams &p, const SidRay &r, const SidAxes &a,
                                          SpanIndex ix, int kd, int ky, int kz, double ta, double tb,
                                          F &&f)
{
    double kdd = (double)kd, kyd = (double)ky, kzd = (double)kz;
    double T = ta, Tn = cross_time(a.nd, a.td, kdd);
    double Ny = cross_time(a.ny, a.ty, kyd), Nz = cross_time(a.nz, a.tz, kzd);
    while (T < tb) {
        const double To = fmin(Tn, tb);
        const bool cy = Ny < To, cz = Nz < To;
        const double qy = fmin(Ny, To), qz = fmin(Nz, To);
        const double lo = fmin(qy, qz), hi = fmax(qy, qz);
        int o0, o1, o2;
        ix.slab(cy, cz, Ny <= Nz, o0, o1, o2);
        f(o0, span_value<TOF>(p, r, T, lo), o1, span_value<TOF>(p, r, lo, hi), o2,
          span_value<TOF>(p, r, hi, To));
        kyd += cy ? 1.0 : 0.0;
        kzd += cz ? 1.0 : 0.0;
        kdd += 1.0;
        Ny = cross_time(a.ny, a.ty, kyd);
        Nz = cross_time(a.nz, a.tz, kzd);
        T = To;
        Tn = cross_time(a.nd, a.td, kdd);
    }
}

// The times outside which the TOF test drops every segment of the ray (segments
// are at most one dominant spacing long).
__device__ __forceinline__ void tof_window(const SidParams &p, const SidRay &r, double td,
                                           double &wa, double &wb)
{
    const double s2 = (double)p.tof_sigma2 +
                      (td * td + (double)p.tof_bin * (double)p.tof_bin) * (1.0 / 12.0);
    const double R = s2 > 0.0 ? 3.0001 * sqrt(s2) + td : 1.0e300;
    wa = r.t_tof - R;
    wb = r.t_tof + R;
}

// Lane `sub` of the L lanes that share a ray walks its part of the ray's
// dominant slabs over the image with strides s (contiguous shares; with TOF of
// the slabs the window leaves).
template <bool TOF, int L, class F>
__device__ __forceinline__ void walk_ray(const SidParams &p, const SidRay &r, const int (&s)[3],
                                         int sub, F &&f)
{
    if (!(r.tend > 0.0))
        return;
    const SidAxes a = ray_axes(r);
    int b[3], bd, by, bz;
#pragma unroll
    for (int c = 0; c < 3; c++)
        b[c] = r.step[c] > 0 ? p.g[c] - r.pos[c] : (r.step[c] < 0 ? r.pos[c] + 1 : 1);
    by_axes(a, b, bd, by, bz);
    // slab k lies between crossings k - 1 and k of the dominant axis
    int k0 = 0, k1 = crossings(a.nd, a.td, r.tend, 0, bd - 1) + 1;
    if (TOF) {
        double wa, wb;
        tof_window(p, r, a.td, wa, wb);
        k0 = max(0, crossings(a.nd, a.td, wa, 0, bd - 1) - 1);
        k1 = min(k1, crossings(a.nd, a.td, wb, 0, bd - 1) + 1);
    }
    if (k0 >= k1)
        return;
    const int n = k1 - k0;
    const int ka = k0 + (int)((unsigned)(n * sub) / (unsigned)L);
    const int kb = k0 + (int)((unsigned)(n * (sub + 1)) / (unsigned)L);
    if (ka >= kb)
        return;
    const double ta = ka == 0 ? 0.0 : cross_time(a.nd, a.td, (double)(ka - 1));
    const double tb = fmin(r.tend, cross_time(a.nd, a.td, (double)(kb - 1)));
    const int ky = ka == 0 ? 0 : crossings(a.ny, a.ty, ta, 0, by - 1);
    const int kz = ka == 0 ? 0 : crossings(a.nz, a.tz, ta, 0, bz - 1);
    const int base = r.pos[0] * s[0] + r.pos[1] * s[1] + r.pos[2] * s[2];
    walk_span<TOF>(p, r, a, SpanIndex(r, a, s, base, ka, ky, kz), ka, ky, kz, ta, tb, f);
}

// Projection part of lane `sub`.  A segment without length adds nothing,
// whatever the voxel holds; it is not loaded either (the gathers of rays that
// are no neighbours cost a cache line per active lane).
template <bool TOF, int L>
__device__ __forceinline__ float gather_ray(const SidParams &p, const SidRay &r, int sub)
{
    float acc = 0.0f;
    walk_ray<TOF, L>(p, r, p.s, sub,
                     [&](int o0, float g0, int o1, float g1, int o2, float g2) {
                         float v0 = 0.0f, v1 = 0.0f, v2 = 0.0f;
                         if (g0 > 0.0f)
                             v0 = p.img[o0];
                         if (g1 > 0.0f)
                             v1 = p.img[o1];
                         if (g2 > 0.0f)
                             v2 = p.img[o2];
                         acc = fmaf(g0, v0, acc);
                         acc = fmaf(g1, v1, acc);
                         acc = fmaf(g2, v2, acc);
                     });
    return acc * span_factor<TOF>(p, r);
}

// Scatter of scale times the ray's weights with FP32 global atomics.
template <bool TOF, int L>
__device__ __forceinline__ void scatter_ray(const SidParams &p, const SidRay &r, int sub,
                                            float scale)
{
    const float w = span_factor<TOF>(p, r) * scale;
    walk_ray<TOF, L>(p, r, p.o, sub,
                     [&](int o0, float g0, int o1, float g1, int o2, float g2) {
                         if (g0 > 0.0f)
                             unsafeAtomicAdd(p.out + o0, g0 * w);
                         if (g1 > 0.0f)
                             unsafeAtomicAdd(p.out + o1, g1 * w);
                         if (g2 > 0.0f)
                             unsafeAtomicAdd(p.out + o2, g2 * w);
                     });
}

// A workgroup of 256 threads takes 256 / L consecutive rays, thread i on ray i
// mod (256 / L): the lanes of a wave walk neighbouring rays (neighbouring
// voxels, for LORs in a locality order) over the same share of their slabs.
// ray_sum adds the L parts of each ray in order; every thread of the workgroup
// calls it and receives its ray's sum.
template <int L>
__device__ __forceinline__ float ray_sum(float v)
{
    if (L == 1)
        return v;
    constexpr int R = 256 / L;
    __shared__ float part[256];
    part[threadIdx.x] = v;
    __syncthreads();
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < L; k++)
        s += part[(int)threadIdx.x % R + k * R];
    return s;
}

// Lanes per ray: as many as leave the chip about six waves per SIMD.
inline int lanes_per_ray(int64_t n)
{
    return n <= 24576 ? 16 : (n <= 131072 ? 4 : 1);
}

} // namespace
} // namespace srfx
