// Elementwise kernels: output zeroing (a fill kernel, so the ops stay
// capturable in HIP graphs) and the MLEM image update.
#include <mutex>

#include "common.h"

namespace srfx {
namespace {

__global__ __launch_bounds__(256) void fill_contig(float *v, int64_t n, float value)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride)
        v[i] = value;
}

__global__ __launch_bounds__(256) void fill_strided(float *v, int gx, int gy, int gz, int sx,
                                                    int sy, int sz, float value)
{
    int64_t n = (int64_t)gx * gy * gz;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        int ix = (int)(i % gx);
        int iy = (int)((i / gx) % gy);
        int iz = (int)(i / ((int64_t)gx * gy));
        v[ix * sx + iy * sy + iz * sz] = value;
    }
}

// model/recon_step.py:48-49: d * efficiency_map * image_succ.
__global__ __launch_bounds__(256) void mlem_update_kernel(float *x, const float *__restrict__ e,
                                                          const float *__restrict__ b, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride)
        x[i] = (x[i] * e[i]) * b[i];
}

unsigned fill_blocks(int64_t n)
{
    int64_t b = (n + 255) / 256;
    if (b > 8192)
        b = 8192;
    return (unsigned)(b < 1 ? 1 : b);
}

} // namespace

int zero_vec(float *v, int64_t n, uint32_t flags, hipStream_t st)
{
    if (flags & SRFX_ACCUMULATE)
        return SRFX_OK;
    if (n <= 0)
        return SRFX_OK;
    hipLaunchKernelGGL(fill_contig, dim3(fill_blocks(n)), dim3(256), 0, st, v, n, 0.0f);
    return launch_status();
}

int zero_grid(float *img, const srfx_grid &g, uint32_t flags, hipStream_t st)
{
    if (flags & SRFX_ACCUMULATE)
        return SRFX_OK;
    Strides s = grid_strides(g);
    int64_t n = grid_nvox(g);
    if (s.x == 1 && s.y == g.shape[0] && s.z == (int64_t)g.shape[0] * g.shape[1])
        return zero_vec(img, n, flags, st);
    hipLaunchKernelGGL(fill_strided, dim3(fill_blocks(n)), dim3(256), 0, st, img, g.shape[0],
                       g.shape[1], g.shape[2], (int)s.x, (int)s.y, (int)s.z, 0.0f);
    return launch_status();
}

// The workspaces' memory pool of each device: one of its own, so that its release
// threshold concerns nobody else.  It keeps freed workspaces, up to kKeptBytes
// (three of the largest calls at once), instead of returning them to the driver
// at every synchronisation (a call that maps its memory again takes milliseconds);
// srfx_workspace_trim returns the rest.
constexpr uint64_t kKeptBytes = 1ull << 30;
constexpr int kMaxDevices = 64;

static std::mutex pool_mutex;
static hipMemPool_t pools[kMaxDevices];

// The current device's pool, or null.
static hipMemPool_t workspace_pool(bool create)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev >= kMaxDevices)
        return nullptr;
    std::lock_guard<std::mutex> lock(pool_mutex);
    if (!pools[dev] && create) {
        hipMemPoolProps props{};
        props.allocType = hipMemAllocationTypePinned;
        props.handleTypes = hipMemHandleTypeNone;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t pool = nullptr;
        uint64_t keep = kKeptBytes;
        if (hipMemPoolCreate(&pool, &props) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        if (hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipMemPoolDestroy(pool);
            return nullptr;
        }
        pools[dev] = pool;
    }
    return pools[dev];
}

int ws_alloc(void **ptr, size_t bytes, hipStream_t st)
{
    bytes = bytes ? bytes : 256;
    // under capture the allocation is the graph's own
    const hipMemPool_t pool = workspace_ok(st) ? workspace_pool(true) : nullptr;
    if ((pool ? hipMallocFromPoolAsync(ptr, bytes, pool, st) : hipMallocAsync(ptr, bytes, st)) !=
        hipSuccess) {
        (void)hipGetLastError();
        return SRFX_ENOMEM;
    }
    return SRFX_OK;
}

int ws_free(void *ptr, hipStream_t st)
{
    return hipFreeAsync(ptr, st) == hipSuccess ? SRFX_OK : SRFX_ELAUNCH;
}

bool workspace_ok(hipStream_t st)
{
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cap) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return cap == hipStreamCaptureStatusNone;
}

} // namespace srfx

using namespace srfx;

extern "C" int srfx_mlem_update(float *x, const float *emap, const float *bp, int64_t n,
                                void *stream)
{
    if (n < 0 || (n > 0 && (!x || !emap || !bp)))
        return SRFX_EINVAL;
    if (n == 0)
        return SRFX_OK;
    hipLaunchKernelGGL(mlem_update_kernel, dim3(fill_blocks(n)), dim3(256), 0,
                       (hipStream_t)stream, x, emap, bp, n);
    return launch_status();
}

extern "C" const char *srfx_strerror(int status)
{
    switch (status) {
    case SRFX_OK:
        return "ok";
    case SRFX_EINVAL:
        return "invalid argument";
    case SRFX_ELAUNCH:
        return "HIP launch failed";
    case SRFX_EUNSUPPORTED:
        return "unsupported configuration";
    case SRFX_ENOMEM:
        return "device workspace allocation failed";
    case SRFX_ETOOLARGE:
        return "input larger than the entry point's static scratch";
    default:
        return "unknown status";
    }
}

extern "C" int srfx_workspace_trim(void)
{
    const hipMemPool_t pool = workspace_pool(false);
    if (pool && hipMemPoolTrimTo(pool, 0) != hipSuccess) {
        (void)hipGetLastError();
        return SRFX_ELAUNCH;
    }
    return SRFX_OK;
}
