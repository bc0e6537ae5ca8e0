/* Host stand-ins for the HIP calls of og_runtime.c, and og_runtime.c itself,
 * for CPU tests of its memory handling: "device" memory is malloc'ed and
 * remembered with the device that was the calling thread's, errors are kept as
 * the runtime keeps them. */
#include <stdlib.h>
#include <string.h>

#include "../opengraph_amd/csrc/og_runtime.c"

#define STUB_MAX 4096
static struct { void *p; size_t bytes; int device; } g_blocks[STUB_MAX];
static size_t g_limit = (size_t)1 << 40, g_used = 0;
static int g_known = 1;   /* hipPointerGetAttributes succeeds for ordinary memory */
static __thread int t_device = 0;
static __thread hipError_t t_last = hipSuccess;

static hipError_t fail(hipError_t e) { return t_last = e; }

hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = t_device; return hipSuccess; }
hipError_t hipGetLastError(void) { hipError_t e = t_last; t_last = hipSuccess; return e; }
hipError_t hipPeekAtLastError(void) { return t_last; }
const char *hipGetErrorString(hipError_t e) { (void)e; return "stub error"; }
#undef hipGetDeviceProperties
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d)
{
    (void)d;
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 4;
    p->totalGlobalMem = (size_t)64 << 20;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n)
{
    if (g_used + n > g_limit) return fail(hipErrorOutOfMemory);
    for (int i = 0; i < STUB_MAX; i++)
        if (!g_blocks[i].p)
        {
            *p = g_blocks[i].p = malloc(n);
            g_blocks[i].bytes = n;
            g_blocks[i].device = t_device;
            g_used += n;
            return hipSuccess;
        }
    return fail(hipErrorOutOfMemory);
}
hipError_t hipFree(void *p)
{
    for (int i = 0; i < STUB_MAX; i++)
        if (g_blocks[i].p == p)
        {
            g_used -= g_blocks[i].bytes;
            g_blocks[i].p = NULL;
            free(p);
            return hipSuccess;
        }
    return fail(hipErrorInvalidValue);
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    (void)k; (void)st;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    (void)p;
    if (!g_known) return fail(hipErrorInvalidValue);
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; *s = NULL; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { (void)f; *e = NULL; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
int og_learn_noalloc_setup(int device) { (void)device; return 0; }
int og_launch_copy(const void *s, void *d, uint64_t n, hipStream_t st) { (void)st; memcpy(d, s, n); return 0; }

/* what the tests look at */
void stub_limit(size_t n) { g_limit = n; }
void stub_known(int k) { g_known = k; }
size_t stub_used(void) { return g_used; }
int stub_device_of(const void *p)
{
    for (int i = 0; i < STUB_MAX; i++) if (g_blocks[i].p == p) return g_blocks[i].device;
    return -1;
}
size_t stub_size_of(const void *p)
{
    for (int i = 0; i < STUB_MAX; i++) if (g_blocks[i].p == p) return g_blocks[i].bytes;
    return 0;
}
int stub_last(void) { return (int)t_last; }
int stub_current(void) { return t_device; }
void stub_set(int device, int error) { t_device = device; t_last = (hipError_t)error; }
