/*
 * fake_hip.c -- the HIP runtime calls of libbp_amd.so, on host memory, for
 * tests of the library's host side where there is no GPU.  Memory is host
 * memory, copies are copies, kernels do nothing; every call is counted or
 * logged.  Loaded with RTLD_GLOBAL before the library, it takes the calls'
 * names first (tests/test_host_runtime.py).
 *
 * A resident run whose kernel does nothing never says that it went through:
 * to the library it is one that was given up.
 */
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#define LOG_BYTES (1u << 20)
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static char log_text[LOG_BYTES];
static size_t log_at, most_bytes = (size_t)-1;
static unsigned long long heap_calls; /* operator new of the library and libstdc++ */
static int fail_at = -1;
static void (*on_capture)(void);
static void (*on_launch)(void);

struct stream {
    int capturing;
};
static int captures, spoilt; /* streams in capture; a call that HIP forbids then has been made */

static void note(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    pthread_mutex_lock(&mu);
    if (log_at + 128 < LOG_BYTES)
        log_at += (size_t)vsnprintf(log_text + log_at, 128, fmt, ap);
    pthread_mutex_unlock(&mu);
    va_end(ap);
}

/* ---- for the tests -------------------------------------------------------- */

const char *fake_log(void) { return log_text; }
unsigned long long fake_heap_calls(void) { return heap_calls; }
void fake_clear(void)
{
    pthread_mutex_lock(&mu);
    log_at = 0;
    log_text[0] = 0;
    heap_calls = 0;
    pthread_mutex_unlock(&mu);
}
void fake_fail_at(int n) { fail_at = n; } /* the n-th allocation from now on fails, 0: the next */
void fake_most_bytes(size_t bytes) { most_bytes = bytes; } /* larger allocations fail from now on */
void fake_on_capture(void (*f)(void)) { on_capture = f; }  /* called while a stream is in capture */
void fake_on_launch(void (*f)(void)) { on_launch = f; }

void *_Znwm(size_t n) /* operator new */
{
    void *p = malloc(n ? n : 1);
    __atomic_fetch_add(&heap_calls, 1, __ATOMIC_RELAXED);
    if (!p)
        abort();
    return p;
}

/* ---- memory --------------------------------------------------------------- */

/* the last error of the calling thread, as the runtime keeps it */
static __thread hipError_t last_error;

static hipError_t allocate(void **p, size_t n)
{
    int fails = n > most_bytes;
    if (fail_at >= 0)
        fails |= fail_at-- == 0;
    *p = fails ? NULL : aligned_alloc(256, (n + 511) / 256 * 256);
    if (!*p)
        return last_error = hipErrorOutOfMemory;
    memset(*p, 0, n);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n)
{
    note("malloc %zu\n", n);
    return allocate(p, n);
}
hipError_t hipFree(void *p)
{
    note("free\n");
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags)
{
    (void)flags;
    note("hostmalloc %zu\n", n);
    return allocate(p, n);
}
hipError_t hipHostFree(void *p)
{
    note("hostfree\n");
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    (void)k, (void)st;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
    (void)st;
    memset(d, v, n);
    return hipSuccess;
}
/* what waits on the null stream or the device: a capture on any thread does
 * not survive it */
static hipError_t not_in_capture(const char *name)
{
    if (!captures)
        return hipSuccess;
    note("%s captured\n", name);
    spoilt = 1;
    return hipErrorStreamCaptureImplicit;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
    hipError_t e = not_in_capture("memcpy");
    return e == hipSuccess ? hipMemcpyAsync(d, s, n, k, NULL) : e;
}
hipError_t hipMemset(void *d, int v, size_t n)
{
    hipError_t e = not_in_capture("memset");
    return e == hipSuccess ? hipMemsetAsync(d, v, n, NULL) : e;
}
hipError_t hipGetSymbolAddress(void **p, const void *symbol)
{
    static double array[1u << 19];
    (void)symbol;
    *p = array;
    return hipSuccess;
}

/* ---- device --------------------------------------------------------------- */

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int d) { return d == 0 ? hipSuccess : hipErrorInvalidDevice; }
hipError_t hipDeviceSynchronize(void) { return not_in_capture("devicesync"); }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d)
{
    (void)d;
    *v = a == hipDeviceAttributeWallClockRate ? 100000 : 256;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d)
{
    (void)d;
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}

hipError_t hipGetLastError(void)
{
    hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "an error"; }

/* ---- launches ------------------------------------------------------------- */

static __thread struct {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
} config;

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream)
{
    config.grid = grid;
    config.block = block;
    config.shared = shared;
    config.stream = stream;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream)
{
    *grid = config.grid;
    *block = config.block;
    *shared = config.shared;
    *stream = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t shared, hipStream_t st)
{
    (void)f, (void)args, (void)shared;
    if (!grid.x || !grid.y || !grid.z || !block.x)
        return last_error = hipErrorInvalidConfiguration;
    note("launch %p%s\n", (void *)st, st && ((struct stream *)st)->capturing ? " captured" : "");
    if (on_launch)
        on_launch();
    return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t shared, hipStream_t st,
                              hipEvent_t a, hipEvent_t b, int flags)
{
    (void)a, (void)b, (void)flags;
    return hipLaunchKernel(f, grid, block, args, shared, st);
}

/* ---- streams, events, graphs ---------------------------------------------- */

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned flags)
{
    (void)flags;
    *s = (hipStream_t)calloc(1, sizeof(struct stream));
    note("stream %p\n", (void *)*s);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    note("sync %p\n", (void *)s);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned flags)
{
    (void)flags;
    note("wait %p %p\n", (void *)s, (void *)e);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *status)
{
    *status = ((struct stream *)s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags)
{
    (void)flags;
    note("eventcreate\n");
    *e = (hipEvent_t)malloc(8);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    note("record %p %p%s\n", (void *)e, (void *)s, s && ((struct stream *)s)->capturing ? " captured" : "");
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { return (void)e, hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { return (void)a, (void)b, *ms = 1.0f, hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode mode)
{
    (void)mode;
    note("begincapture %p\n", (void *)s);
    ((struct stream *)s)->capturing = 1;
    ++captures;
    spoilt = 0;
    if (on_capture)
        on_capture();
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
    note("endcapture %p\n", (void *)s);
    ((struct stream *)s)->capturing = 0;
    --captures;
    if (spoilt)
        return hipErrorStreamCaptureInvalidated;
    *g = (hipGraph_t)malloc(8);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *n, char *log, size_t bytes)
{
    (void)g, (void)n, (void)log, (void)bytes;
    note("instantiate\n");
    *x = (hipGraphExec_t)malloc(8);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g)
{
    free(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x)
{
    note("graphdestroy\n");
    free(x);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s)
{
    (void)x;
    note("graphlaunch %p%s\n", (void *)s, s && ((struct stream *)s)->capturing ? " captured" : "");
    return hipSuccess;
}
