// PSF blur of an image around the projector (the reference's PSFReconStep,
// model/recon_step.py:56-115): the image seen as a matrix X of nxy = nx * ny
// rows (voxel columns) by nz columns (slices), blurred across columns by a
// sparse nxy x nxy matrix S (CSR) and along z by a dense nz x nz matrix:
//   out[r, z] = sum_z' (sum_k S[r, c_k] X[c_k, z']) M[z', z]
// Forward (recon_step.py:79-90, S psf_xy and X psf_z^T): M = psf_z^T.
// Backward (recon_step.py:103-110, S^T psf_xy and X psf_z): M = psf_z, with
// S^T passed as its own CSR.  The reference forms X M first and then S (X M);
// the product is associative, so the sums here differ from its order by FP32
// rounding only.
#include <algorithm>

#include "common.h"

namespace srfx {
namespace {

constexpr int kPsfRowsPerBlock = 4; // one wave of 64 lanes per row
constexpr int kPsfMaxNz = 2048;     // 4 rows x nz floats of LDS

// One wave per output row.  Lanes stride over z: first the sparse sum of the
// neighbour rows (each a contiguous run of nz floats, so the lanes' reads are
// coalesced) into the wave's LDS row t, then out[r, z] = sum_z' t[z'] M[z', z]
// with t from LDS and M read along z (coalesced, cached), z' over the band
// z - below .. z + above outside which M is zero (an axial blur is banded;
// the skipped terms are exact zeros).
__global__ __launch_bounds__(256) void psf_apply_kernel(const int *__restrict__ row_ptr,
                                                        const int *__restrict__ col,
                                                        const float *__restrict__ val, int nrows,
                                                        const float *__restrict__ m, int nz,
                                                        int below, int above,
                                                        const float *__restrict__ img,
                                                        float *__restrict__ out)
{
    extern __shared__ float t_lds[];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // wave-uniform row: the CSR entries come through scalar loads
    const int r = __builtin_amdgcn_readfirstlane((int)blockIdx.x * kPsfRowsPerBlock + w);
    float *t = t_lds + w * nz;
    if (r < nrows) {
        const int k0 = row_ptr[r], k1 = row_ptr[r + 1];
        // 256 columns per pass, 4 per lane, so that each CSR entry issues up
        // to 4 independent row loads
        for (int zb = 0; zb < nz; zb += 256) {
            float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
            for (int k = k0; k < k1; k++) {
                const float v = val[k];
                const float *src = img + (int64_t)col[k] * nz + zb + lane;
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (zb + lane + 64 * j < nz)
                        acc[j] = fmaf(v, src[64 * j], acc[j]);
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (zb + lane + 64 * j < nz)
                    t[zb + lane + 64 * j] = acc[j];
        }
    }
    __syncthreads();
    if (r < nrows) {
        for (int z = lane; z < nz; z += 64) {
            float acc = 0.0f;
            const int z0 = max(0, z - below), z1 = min(nz - 1, z + above);
            for (int zp = z0; zp <= z1; zp++)
                acc = fmaf(t[zp], m[(int64_t)zp * nz + z], acc);
            out[(int64_t)r * nz + z] = acc;
        }
    }
}

// Four consecutive floats at any float's address (one 16-byte load).
struct __attribute__((packed, aligned(4))) Vec4 {
    float x, y, z, w;
};

// The blur of 4 <= nz <= 512 columns, G lanes (16 up to 64 columns, else 32) per
// row: a lane holds four consecutive columns of a chunk of 4 G (NC chunks; the
// last lane of a row is moved back to end on it and repeats a few columns), so a
// neighbour's row is one 16-byte load a lane, two or four rows a wave.  One wave
// per row with one column a lane (psf_apply_kernel) needed 42 loads of 4 bytes
// for 21 entries of 100 columns and re-read M for every row: 91 us at 200 x 200
// x 100, bound by load latency; 28 us here, 12 TB/s of neighbour rows from the
// L1s and L2s.  Entries are staged in LDS G at a time and broadcast from
// there; M's band stays in LDS for the workgroup's rows where it fits
// (mlds), the sparse sum goes to LDS between zeros so that the band needs no
// bounds.  The workgroups of an XCD take a contiguous eighth of the rows: what
// neighbouring rows share stays in its L2.  Sums in psf_apply_kernel's order
// (entries ascending, z' ascending), the same bits.
template <int G, int NC>
__global__ __launch_bounds__(256) void psf_rows_kernel(const int *__restrict__ row_ptr,
                                                       const int *__restrict__ col,
                                                       const float *__restrict__ val, int nrows,
                                                       const float *__restrict__ m, int nz,
                                                       int below, int above, int mlds,
                                                       int rows_per_block,
                                                       const float *__restrict__ img,
                                                       float *__restrict__ out)
{
    extern __shared__ float sh[];
    constexpr int N = 256 / G; // rows of a pass
    const int row = (int)threadIdx.x / G, l = (int)threadIdx.x % G;
    const int W = below + above + 1, tw = nz + below + above;
    float *const t = sh + row * tw;                      // columns -below .. nz + above - 1
    float *const mb = sh + N * tw;                       // M's band: [tap][z]
    int2 *const ent = (int2 *)(sh + ((N * tw + (mlds ? W * nz : 0) + 1) & ~1)) + row * G;
    for (int i = l; i < tw; i += G)
        t[i] = 0.0f;
    if (mlds) {
        for (int i = threadIdx.x; i < W * nz; i += 256) {
            const int j = i / nz, z = i - j * nz, zp = z - below + j;
            mb[i] = zp >= 0 && zp < nz ? m[(int64_t)zp * nz + z] : 0.0f;
        }
    }
    __syncthreads();
    // this workgroup's rows: XCD b mod 8 takes a contiguous eighth of the blocks
    const int nb = (int)gridDim.x, b = (int)blockIdx.x;
    const int blk = (b & 7) * (nb >> 3) + min(b & 7, nb & 7) + (b >> 3);
    const int r1 = min(nrows, (blk + 1) * rows_per_block);
    for (int r0 = blk * rows_per_block; r0 < r1; r0 += N) {
        const int r = r0 + row;
        const bool live = r < r1;
        const int k0 = live ? row_ptr[r] : 0, k1 = live ? row_ptr[r + 1] : 0;
        float acc[4 * NC];
        int z0[NC]; // first column of the lane's vector (-1: none)
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int z = 4 * (G * c + l);
            z0[c] = live && z < nz ? min(z, nz - 4) : -1;
            acc[4 * c] = acc[4 * c + 1] = acc[4 * c + 2] = acc[4 * c + 3] = 0.0f;
        }
        for (int kb = k0; kb < k1; kb += G) {
            const int n = min(G, k1 - kb);
            if (l < n)
                ent[l] = make_int2(col[kb + l], __float_as_int(val[kb + l]));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 4
            for (int i = 0; i < n; i++) {
                const int2 e = ent[i];
                const float v = __int_as_float(e.y);
                const float *src = img + (int64_t)e.x * nz;
#pragma unroll
                for (int c = 0; c < NC; c++)
                    if (z0[c] >= 0) {
                        const Vec4 x = *reinterpret_cast<const Vec4 *>(src + z0[c]);
                        acc[4 * c] = fmaf(v, x.x, acc[4 * c]);
                        acc[4 * c + 1] = fmaf(v, x.y, acc[4 * c + 1]);
                        acc[4 * c + 2] = fmaf(v, x.z, acc[4 * c + 2]);
                        acc[4 * c + 3] = fmaf(v, x.w, acc[4 * c + 3]);
                    }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
#pragma unroll
        for (int c = 0; c < NC; c++)
            if (z0[c] >= 0)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    t[below + z0[c] + q] = acc[4 * c + q];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int c = 0; c < NC; c++) {
            if (z0[c] < 0)
                continue;
            const int z = z0[c];
            float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (mlds) {
#pragma unroll 4
                for (int j = 0; j < W; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        o[q] = fmaf(t[z + j + q], mb[j * nz + z + q], o[q]);
            } else {
                // z' from the first to the last of the four columns' bands
                const int a = max(0, z - below), e = min(nz - 1, z + 3 + above);
                for (int zp = a; zp <= e; zp++) {
                    const float x = t[below + zp];
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        if (zp >= z + q - below && zp <= z + q + above)
                            o[q] = fmaf(x, m[(int64_t)zp * nz + z + q], o[q]);
                }
            }
            *reinterpret_cast<Vec4 *>(out + (int64_t)r * nz + z) = Vec4{o[0], o[1], o[2], o[3]};
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// LDS of psf_rows_kernel<G>: a pass' rows of sums, M's band, their entries.
unsigned psf_rows_lds(int G, int nz, int below, int above, bool mlds)
{
    const int N = 256 / G, W = below + above + 1, tw = nz + below + above;
    return 4u * (unsigned)((N * tw + (mlds ? W * nz : 0) + 1) & ~1) + 256u * sizeof(int2);
}

template <int G, int NC>
int launch_rows(const int *row_ptr, const int *col, const float *val, int nrows, const float *m,
                int nz, int below, int above, const float *img, float *out, int cus,
                hipStream_t st)
{
    constexpr int N = 256 / G;
    // M's band in LDS where five workgroups still share a CU
    const bool mlds = psf_rows_lds(G, nz, below, above, true) <= 32u * 1024u;
    // eight workgroups a CU, each with whole passes of rows
    const int want = 8 * cus;
    const int per = std::max(1, ((nrows + want - 1) / want + N - 1) / N) * N;
    hipLaunchKernelGGL((psf_rows_kernel<G, NC>), dim3((nrows + per - 1) / per), dim3(256),
                       psf_rows_lds(G, nz, below, above, mlds), st, row_ptr, col, val, nrows, m,
                       nz, below, above, mlds ? 1 : 0, per, img, out);
    return launch_status();
}

} // namespace
} // namespace srfx

extern "C" int srfx_psf_apply(const int32_t *row_ptr, const int32_t *col, const float *val,
                              int32_t nrows, const float *m, int32_t nz, int32_t below,
                              int32_t above, const float *img, float *out, void *stream)
{
    using namespace srfx;
    if (nrows < 0 || nz < 1 || below < 0 || above < 0 ||
        (nrows > 0 && (!row_ptr || !col || !val || !m || !img || !out)))
        return SRFX_EINVAL;
    if (img == out)
        return SRFX_EINVAL; // rows read neighbours: no in-place blur
    if (nz > kPsfMaxNz)
        return SRFX_EUNSUPPORTED;
    if (nrows == 0)
        return SRFX_OK;
    hipStream_t st = (hipStream_t)stream;
    if (nz >= 4 && nz <= 512 && below < nz && above < nz) {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return SRFX_ELAUNCH;
        if (nz <= 64)
            return launch_rows<16, 1>(row_ptr, col, val, nrows, m, nz, below, above, img, out,
                                      cus, st);
        if (nz <= 128)
            return launch_rows<32, 1>(row_ptr, col, val, nrows, m, nz, below, above, img, out,
                                      cus, st);
        if (nz <= 256)
            return launch_rows<32, 2>(row_ptr, col, val, nrows, m, nz, below, above, img, out,
                                      cus, st);
        return launch_rows<32, 4>(row_ptr, col, val, nrows, m, nz, below, above, img, out, cus,
                                  st);
    }
    const int blocks = (nrows + kPsfRowsPerBlock - 1) / kPsfRowsPerBlock;
    hipLaunchKernelGGL(psf_apply_kernel, dim3(blocks), dim3(64 * kPsfRowsPerBlock),
                       sizeof(float) * kPsfRowsPerBlock * nz, st, row_ptr, col,
                       val, nrows, m, nz, below, above, img, out);
    return launch_status();
}
