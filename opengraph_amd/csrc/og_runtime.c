/*
 * og_runtime.c -- device context, error text and allocation helpers of
 * libopengraph_amd (host C over the HIP runtime C API).
 */
#include <pthread.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#include "og_internal.h"
#include "og_learn.h"
#include "opengraph_amd_ext.h"

static __thread char g_err[512];
static int g_ready = 0;
static int g_device = 0;
static int g_cus = 0;
static hipStream_t g_stream = NULL;
/* second stream and its fork / join events: the pull's long-row chains run
 * there beside the persistent kernel (og_pr.hip) */
static hipStream_t g_side = NULL;
static hipEvent_t g_fork = NULL, g_join = NULL;
static pthread_mutex_t g_ctx_lock = PTHREAD_MUTEX_INITIALIZER;
static size_t g_pool_cap = 0;   /* bytes of freed device memory kept */

void og_set_error(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

const char *og_get_error(void) { return g_err; }

int og_hip_check(hipError_t e, const char *what)
{
    if (e == hipSuccess) return 0;
    og_set_error("%s: %s (%d)", what, hipGetErrorString(e), (int)e);
    return -1;
}

static __thread hipError_t g_launch_err = hipSuccess;

void og_launch_note(hipError_t e)
{
    if (e != hipSuccess && g_launch_err == hipSuccess) g_launch_err = e;
}

hipError_t og_launch_status(void)
{
    hipError_t e = g_launch_err;
    g_launch_err = hipSuccess;
    return e;
}

static void og_ctx_release(void)
{
    if (g_join) (void)hipEventDestroy(g_join);
    if (g_fork) (void)hipEventDestroy(g_fork);
    if (g_side) (void)hipStreamDestroy(g_side);
    if (g_stream) (void)hipStreamDestroy(g_stream);
    g_join = g_fork = NULL;
    g_side = g_stream = NULL;
}

/* The device, its streams (both non-blocking, default priority) and events,
 * created together once per process under a lock; on a failure nothing
 * made so far is kept and the next call starts again. */
static int og_ctx_create(void)
{
    int n = 0;
    if (og_hip_check(hipGetDeviceCount(&n), "hipGetDeviceCount")) return -1;
    if (n <= 0)
    {
        og_set_error("no HIP device is visible");
        return -1;
    }
    if (g_device >= n) g_device = 0;
    if (og_hip_check(hipSetDevice(g_device), "hipSetDevice")) return -1;
    hipDeviceProp_t prop;
    if (og_hip_check(hipGetDeviceProperties(&prop, g_device), "hipGetDeviceProperties")) return -1;
    g_cus = prop.multiProcessorCount;
    g_pool_cap = prop.totalGlobalMem / 64;
    if (og_hip_check(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking), "hipStreamCreate") ||
        og_hip_check(hipStreamCreateWithFlags(&g_side, hipStreamNonBlocking), "hipStreamCreate (side)") ||
        og_hip_check(hipEventCreateWithFlags(&g_fork, hipEventDisableTiming), "hipEventCreate (fork)") ||
        og_hip_check(hipEventCreateWithFlags(&g_join, hipEventDisableTiming), "hipEventCreate (join)") ||
        og_learn_noalloc_setup(g_device))
    {
        og_ctx_release();
        return -1;
    }
    return 0;
}

int og_device(void) { return g_device; }

int og_ctx_ensure(void)
{
    if (__atomic_load_n(&g_ready, __ATOMIC_ACQUIRE)) return 0;
    pthread_mutex_lock(&g_ctx_lock);
    int rc = 0;
    if (!g_ready)
    {
        rc = og_ctx_create();
        if (!rc) __atomic_store_n(&g_ready, 1, __ATOMIC_RELEASE);
    }
    pthread_mutex_unlock(&g_ctx_lock);
    return rc;
}

hipStream_t og_side_stream(void) { return g_side; }
hipEvent_t og_side_fork(void) { return g_fork; }
hipEvent_t og_side_join(void) { return g_join; }

hipStream_t og_stream(void) { return g_stream; }

hipError_t og_copy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind)
{
    hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, g_stream);
    if (e != hipSuccess) return e;
    return hipStreamSynchronize(g_stream);
}
int og_num_cus(void) { return g_cus; }

/* With OGPU_TRACE set (any value), each drop-in entry point names itself,
 * the device and the graph on stderr: a host program linked against the
 * library can show which definition it called.  Output only. */
void og_trace_entry(const char *fn, uint32_t n_vertices, uint32_t n_edges)
{
    if (!getenv("OGPU_TRACE")) return;
    fprintf(stderr, "opengraph_amd: %s on HIP device %d (%d CUs), %u vertices, %u edges\n", fn, g_device,
            g_cus, n_vertices, n_edges);
}

/* With OGPU_TRACE, the plans the drop-in entry points build (a later call on the
 * same graph uses them again). */
void og_trace_plan(const char *kind)
{
    if (getenv("OGPU_TRACE")) fprintf(stderr, "opengraph_amd: plan built (%s)\n", kind);
}

/* ---- device memory ----
 * A graph's build and a run's setup take dozens of short-lived buffers, and
 * hipMalloc and hipFree (which waits for the device) of the large ones cost
 * more than the kernels between them: 10 of 21 ms from a 67 M-edge list to its
 * ranks.  Freed blocks are kept by size and handed out again.  All the
 * library's work is on one stream (its side stream is joined to it), so what
 * a block's next owner enqueues runs after what its last one did, and none of
 * these pointers leaves the library.  Kept blocks are bounded by a 64th of the
 * device's memory, the longest unused given back first, and all of them are
 * given back before an allocation is allowed to fail, or when the caller says so
 * (ogpu_release_memory).  Every block is the library's device's, whichever the
 * calling thread has chosen: another thread may get it next. */
typedef struct og_block
{
    void *p;
    size_t bytes;
    struct og_block *next;
} og_block;

#define OG_POOL_SLOTS 4096u
static pthread_mutex_t g_pool_lock = PTHREAD_MUTEX_INITIALIZER;
static og_block *g_pool_live[OG_POOL_SLOTS];   /* handed out, by address */
static og_block *g_pool_free = NULL;           /* kept, the last freed first */
static size_t g_pool_bytes = 0;

static unsigned og_pool_slot(const void *p)
{
    return (unsigned)(((uintptr_t)p >> 8) * 0x9E3779B97F4A7C15ull >> 40) & (OG_POOL_SLOTS - 1);
}

/* Sizes are rounded up by at most an eighth, so that similar ones meet; a
 * block that is never kept is not. */
static size_t og_pool_size(size_t bytes)
{
    if (bytes <= 4096) return 4096;
    if (bytes > g_pool_cap) return bytes;
    size_t step = 512;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

/* Frees the kept blocks past `most` bytes, the longest unused first. */
static void og_pool_trim(size_t most)
{
    while (g_pool_bytes > most && g_pool_free)
    {
        og_block **q = &g_pool_free;
        while ((*q)->next) q = &(*q)->next;
        og_block *b = *q;
        *q = NULL;
        g_pool_bytes -= b->bytes;
        (void)hipFree(b->p);
        free(b);
    }
}

static hipError_t og_device_malloc(void **p, size_t bytes)
{
    int was = g_device;
    (void)hipGetDevice(&was);
    hipError_t e = was == g_device ? hipSuccess : hipSetDevice(g_device);
    if (e == hipSuccess) e = hipMalloc(p, bytes);
    if (e != hipSuccess) (void)hipGetLastError();   /* reported by og_dalloc */
    if (was != g_device) (void)hipSetDevice(was);
    return e;
}

void *og_dalloc(size_t bytes)
{
    const size_t size = og_pool_size(bytes);
    pthread_mutex_lock(&g_pool_lock);
    og_block *b = NULL;
    for (og_block **q = &g_pool_free; *q; q = &(*q)->next)
        if ((*q)->bytes == size)
        {
            b = *q;
            *q = b->next;
            g_pool_bytes -= size;
            break;
        }
    if (!b)
    {
        hipError_t e = hipErrorOutOfMemory;
        b = (og_block *)malloc(sizeof(og_block));
        if (b)
        {
            b->bytes = size;
            e = og_device_malloc(&b->p, size);
            if (e != hipSuccess)
            {
                og_pool_trim(0);
                b->bytes = bytes ? bytes : 256;
                e = og_device_malloc(&b->p, b->bytes);
            }
        }
        if (e != hipSuccess)
        {
            free(b);
            pthread_mutex_unlock(&g_pool_lock);
            og_set_error("hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
            return NULL;
        }
    }
    const unsigned k = og_pool_slot(b->p);
    b->next = g_pool_live[k];
    g_pool_live[k] = b;
    pthread_mutex_unlock(&g_pool_lock);
    return b->p;
}

void og_dfree(void *p)
{
    if (!p) return;
    pthread_mutex_lock(&g_pool_lock);
    og_block **q = &g_pool_live[og_pool_slot(p)];
    while (*q && (*q)->p != p) q = &(*q)->next;
    og_block *b = *q;
    if (b)
    {
        *q = b->next;
        if (b->bytes <= g_pool_cap)
        {
            b->next = g_pool_free;
            g_pool_free = b;
            g_pool_bytes += b->bytes;
            og_pool_trim(g_pool_cap);
            p = NULL;
        }
        else free(b);
    }
    pthread_mutex_unlock(&g_pool_lock);
    if (p) (void)hipFree(p);
}

/* ---- large results to the caller's memory ----
 * The caller's buffer is ordinary, usually fresh memory: a plain copy into it
 * stages and faults its pages on one thread (64 MB: 6 ms, 11 GB/s).  Here
 * each of a few threads takes every n-th piece through a pinned buffer of its
 * own, so that the copy engine serves one thread while the others move their
 * pieces on (64 MB: 2 ms).  Below OG_STAGE_MIN a thread costs more than it
 * saves. */
#define OG_STAGE_BYTES ((size_t)1 << 20)
#define OG_STAGE_THREADS 8u
#define OG_STAGE_MIN ((size_t)4 << 20)
static pthread_mutex_t g_stage_lock = PTHREAD_MUTEX_INITIALIZER;
static char *g_stage = NULL;                    /* a piece per thread */
static hipEvent_t g_stage_ev[OG_STAGE_THREADS];

typedef struct og_stage_job
{
    char *dst;
    const char *src;
    size_t bytes;
    uint32_t self, threads;
    hipError_t err;
} og_stage_job;

static int og_stage_make(void **p)
{
    if (hipHostMalloc(p, OG_STAGE_THREADS * OG_STAGE_BYTES, hipHostMallocDefault) != hipSuccess)
    {
        (void)hipGetLastError();
        return 0;
    }
    for (uint32_t i = 0; i < OG_STAGE_THREADS; i++)
        if (hipEventCreateWithFlags(&g_stage_ev[i], hipEventDisableTiming) != hipSuccess)
        {
            (void)hipGetLastError();
            while (i-- > 0) (void)hipEventDestroy(g_stage_ev[i]);
            (void)hipHostFree(*p);
            return 0;
        }
    return 1;
}

static int og_stage_ready(void)
{
    if (g_stage) return 1;
    void *p = NULL;
    int was = g_device;
    (void)hipGetDevice(&was);
    if (was != g_device && hipSetDevice(g_device) != hipSuccess) return 0;
    const int ok = og_stage_make(&p);
    if (was != g_device) (void)hipSetDevice(was);   /* the caller's choice stays */
    if (ok) g_stage = (char *)p;
    return ok;
}

static void *og_stage_run(void *arg)
{
    og_stage_job *j = (og_stage_job *)arg;
    char *buf = g_stage + j->self * OG_STAGE_BYTES;
    /* (thread 0 is the caller's, whose current device stays) */
    j->err = j->self ? hipSetDevice(g_device) : hipSuccess;
    for (size_t o = j->self * OG_STAGE_BYTES; o < j->bytes && j->err == hipSuccess; o += j->threads * OG_STAGE_BYTES)
    {
        const size_t k = j->bytes - o < OG_STAGE_BYTES ? j->bytes - o : OG_STAGE_BYTES;
        j->err = hipMemcpyAsync(buf, j->src + o, k, hipMemcpyDeviceToHost, g_stream);
        if (j->err == hipSuccess) j->err = hipEventRecord(g_stage_ev[j->self], g_stream);
        if (j->err == hipSuccess) j->err = hipEventSynchronize(g_stage_ev[j->self]);
        if (j->err == hipSuccess) memcpy(j->dst + o, buf, k);
    }
    return NULL;
}

hipError_t og_download(void *dst, const void *src, size_t bytes)
{
    /* the caller's own pinned (or device) memory takes the copy directly; so does
     * a thread with an error pending, which asking about an unknown pointer
     * could replace */
    int plain = bytes < OG_STAGE_MIN || hipPeekAtLastError() != hipSuccess;
    if (!plain)
    {
        hipPointerAttribute_t at;
        memset(&at, 0, sizeof(at));
        if (hipPointerGetAttributes(&at, dst) == hipSuccess) plain = at.type != hipMemoryTypeUnregistered;
        else (void)hipGetLastError();
    }
    if (plain) return og_copy(dst, src, bytes, hipMemcpyDeviceToHost);
    pthread_mutex_lock(&g_stage_lock);
    if (!og_stage_ready())
    {
        pthread_mutex_unlock(&g_stage_lock);
        return og_copy(dst, src, bytes, hipMemcpyDeviceToHost);
    }
    const long cpus = sysconf(_SC_NPROCESSORS_ONLN);
    const uint32_t n = cpus > 0 && cpus < (long)OG_STAGE_THREADS ? (uint32_t)cpus : OG_STAGE_THREADS;
    og_stage_job job[OG_STAGE_THREADS];
    pthread_t th[OG_STAGE_THREADS];
    int started[OG_STAGE_THREADS] = {0};
    for (uint32_t i = 0; i < n; i++) job[i] = (og_stage_job){(char *)dst, (const char *)src, bytes, i, n, hipSuccess};
    for (uint32_t i = 1; i < n; i++) started[i] = !pthread_create(&th[i], NULL, og_stage_run, &job[i]);
    og_stage_run(&job[0]);
    hipError_t e = job[0].err;
    for (uint32_t i = 1; i < n; i++)
    {
        if (started[i]) pthread_join(th[i], NULL);
        else
        {
            int was = g_device;
            (void)hipGetDevice(&was);
            og_stage_run(&job[i]);
            if (was != g_device) (void)hipSetDevice(was);
        }
        if (e == hipSuccess) e = job[i].err;
    }
    pthread_mutex_unlock(&g_stage_lock);
    return e;
}

void *og_host_alloc(size_t bytes)
{
    void *p = NULL;
    if (bytes == 0) bytes = 1;
    if (posix_memalign(&p, 128, bytes) != 0)
    {
        fprintf(stderr, "Error, aligned_alloc of %zu bytes failed\n", bytes);
        exit(EXIT_FAILURE);
    }
    return p;
}

/* ------------------------- public helpers ------------------------- */

int ogpu_init(int device)
{
    if (g_ready && device != g_device)
    {
        og_set_error("ogpu_init: already initialised on device %d", g_device);
        return -1;
    }
    g_device = device < 0 ? 0 : device;
    return og_ctx_ensure();
}

const char *ogpu_last_error(void) { return g_err; }

int ogpu_device_info(char *name, size_t name_len, int *num_cus, size_t *total_mem)
{
    if (og_ctx_ensure()) return -1;
    hipDeviceProp_t prop;
    if (og_hip_check(hipGetDeviceProperties(&prop, g_device), "hipGetDeviceProperties")) return -1;
    if (name && name_len)
    {
        snprintf(name, name_len, "%s (%s)", prop.name, prop.gcnArchName);
    }
    if (num_cus) *num_cus = prop.multiProcessorCount;
    if (total_mem) *total_mem = prop.totalGlobalMem;
    return 0;
}

int ogpu_malloc(void **ptr, size_t bytes)
{
    /* (the caller's: not from the pool, whose reuse follows the library stream) */
    if (og_ctx_ensure()) return -1;
    *ptr = NULL;
    hipError_t e = hipMalloc(ptr, bytes ? bytes : 256);
    if (e != hipSuccess)
    {
        (void)hipGetLastError();
        pthread_mutex_lock(&g_pool_lock);
        og_pool_trim(0);
        pthread_mutex_unlock(&g_pool_lock);
        e = hipMalloc(ptr, bytes ? bytes : 256);
    }
    if (e == hipSuccess) return 0;
    *ptr = NULL;
    og_set_error("hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
    return -1;
}

int ogpu_release_memory(void)
{
    pthread_mutex_lock(&g_pool_lock);
    og_pool_trim(0);
    pthread_mutex_unlock(&g_pool_lock);
    return 0;
}

int ogpu_free(void *ptr)
{
    if (!ptr) return 0;
    return og_hip_check(hipFree(ptr), "hipFree");
}

int ogpu_memcpy_h2d(void *dst, const void *src, size_t bytes)
{
    if (og_ctx_ensure()) return -1;
    if (og_hip_check(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g_stream), "hipMemcpy H2D"))
        return -1;
    return og_hip_check(hipStreamSynchronize(g_stream), "hipStreamSynchronize");
}

int ogpu_memcpy_d2h(void *dst, const void *src, size_t bytes)
{
    if (og_ctx_ensure()) return -1;
    if (og_hip_check(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g_stream), "hipMemcpy D2H"))
        return -1;
    return og_hip_check(hipStreamSynchronize(g_stream), "hipStreamSynchronize");
}

int og_launch_copy(const void *src, void *dst, uint64_t bytes, hipStream_t s);

int ogpu_device_copy(void *d_dst, const void *d_src, size_t bytes)
{
    if (og_ctx_ensure()) return -1;
    if (bytes % 16)
    {
        og_set_error("ogpu_device_copy: size %zu is not a multiple of 16", bytes);
        return -1;
    }
    if (og_launch_copy(d_src, d_dst, bytes, g_stream)) return -1;
    return og_hip_check(hipStreamSynchronize(g_stream), "hipStreamSynchronize");
}

int ogpu_synchronize(void)
{
    if (og_ctx_ensure()) return -1;
    if (og_hip_check(hipStreamSynchronize(g_stream), "hipStreamSynchronize")) return -1;
    return og_hip_check(hipDeviceSynchronize(), "hipDeviceSynchronize");
}
