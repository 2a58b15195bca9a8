// fakehip.cpp -- the HIP runtime calls that the linears' host code makes, on host memory, for tests of that code without
// a GPU: allocations come from malloc, a launch is only recorded, and a test chooses what fails. Loaded with RTLD_GLOBAL
// before the library, its symbols take the place of the runtime's.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>

namespace {

struct Launch {
    const void *fn;
    void *stream;
    const void *arg1;   // the kernel's second argument, read as a pointer
    dim3 grid, block;
};
constexpr int kMax = 64;
Launch g_launch[kMax];
int g_launches, g_fail_launch = -1, g_fail_malloc, g_mallocs, g_live, g_device, g_capturing, g_arg1;
hipError_t g_last;
dim3 g_grid, g_block;
size_t g_shmem;
hipStream_t g_stream;

hipError_t set(hipError_t e)
{
    if (e != hipSuccess) g_last = e;
    return e;
}

}  // namespace

extern "C" {

void fake_reset() { g_launches = 0, g_fail_launch = -1, g_fail_malloc = 0, g_last = hipSuccess; }
int fake_launches() { return g_launches; }
void *fake_launch_arg1(int i) { return const_cast<void *>(g_launch[i].arg1); }
void *fake_launch_stream(int i) { return g_launch[i].stream; }
int fake_launch_grid(int i) { return (int)g_launch[i].grid.x; }
int fake_launch_block(int i) { return (int)g_launch[i].block.x; }
void fake_read_arg1(int on) { g_arg1 = on; }   // only where every launched kernel has a second argument
void fake_fail_launch(int i) { g_fail_launch = i; }
void fake_fail_malloc(int on) { g_fail_malloc = on; }
int fake_mallocs() { return g_mallocs; }
int fake_live() { return g_live; }
void fake_device(int d) { g_device = d; }
void fake_capturing(int on) { g_capturing = on; }

hipError_t hipMalloc(void **p, size_t n)
{
    ++g_mallocs;
    if (g_fail_malloc || !(*p = calloc(1, n))) return set(hipErrorOutOfMemory);
    ++g_live;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (p) --g_live;
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s)
{
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipStreamGetId(hipStream_t s, unsigned long long *id)
{
    *id = (unsigned long long)(size_t)s;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = g_device;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 160 << 10 : 0;
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t st)
{
    g_grid = grid, g_block = block, g_shmem = shmem, g_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shmem, hipStream_t *st)
{
    *grid = g_grid, *block = g_block, *shmem = g_shmem, *st = g_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **args, size_t, hipStream_t st)
{
    const int i = g_launches++;
    if (i < kMax) {
        g_launch[i] = {fn, st, nullptr, grid, block};
        if (g_arg1) memcpy(&g_launch[i].arg1, args[1], sizeof(void *));
    }
    return set(i == g_fail_launch ? hipErrorLaunchFailure : hipSuccess);
}

}  // extern "C"
