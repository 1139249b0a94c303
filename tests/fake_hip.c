/* A HIP runtime of host memory for tests of libytm's host code on the CPU: kernels do nothing,
 * copies are made at once, and a stream counts as busy from its last launch or copy until it is
 * waited for.  fake_fail makes one call of a function fail.  Loaded with RTLD_GLOBAL before
 * libytm.so, so that its HIP symbols resolve here. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#define DEVICES 2
#define BLOCKS 65536

typedef struct { void *p; size_t bytes; int device; } Block; /* device -1: pinned host memory */
struct ihipStream_t { int busy, used; };

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static Block blocks[BLOCKS];
static struct ihipStream_t streams[256], null_stream;
static __thread int device;
static char fail_name[64];
static int fail_after = -1, fail_count, fail_seen;
static __thread hipError_t last_error;
static long calls_malloc, calls_free, calls_host_malloc, calls_host_free, calls_large; /* large: of 1 MiB and more */

void fake_fail(const char *name, int after, int count) { /* calls `after` .. after + count - 1 of `name` fail */
    pthread_mutex_lock(&mu);
    strncpy(fail_name, name, sizeof fail_name - 1);
    fail_after = after;
    fail_count = count;
    fail_seen = 0;
    pthread_mutex_unlock(&mu);
}
int fake_failed(void) { return fail_seen > fail_after; } /* whether that call was reached */
int fake_busy(void) { /* streams with work that nothing has waited for */
    int n = null_stream.busy;
    for (int i = 0; i < 256; ++i) n += streams[i].busy;
    return n;
}
size_t fake_live(int dev) { /* bytes allocated on a device (-1: pinned) */
    size_t n = 0;
    pthread_mutex_lock(&mu);
    for (int i = 0; i < BLOCKS; ++i)
        if (blocks[i].p && blocks[i].device == dev) n += blocks[i].bytes;
    pthread_mutex_unlock(&mu);
    return n;
}
static int delay_ms;
void fake_delay_malloc(int ms) { delay_ms = ms; } /* each hipMalloc takes that long */
static size_t limit;
void fake_limit(size_t bytes) { limit = bytes; } /* what a device holds at most; 0: anything */
long fake_calls(int which) {
    const long c[] = {calls_malloc, calls_free, calls_host_malloc, calls_host_free, calls_large};
    return c[which];
}

static int failing(const char *name) {
    int f = 0;
    pthread_mutex_lock(&mu);
    if (strcmp(name, fail_name) == 0) f = fail_seen >= fail_after && fail_seen < fail_after + fail_count, ++fail_seen;
    pthread_mutex_unlock(&mu);
    return f;
}
#define MAY_FAIL if (failing(__func__)) return last_error = hipErrorOutOfMemory

static hipError_t get(void **p, size_t bytes, int dev) {
    *p = malloc(bytes ? bytes : 1);
    if (!*p) return hipErrorOutOfMemory;
    memset(*p, 0, bytes < 4096 ? bytes : 4096);
    pthread_mutex_lock(&mu);
    int i = 0;
    while (i < BLOCKS && blocks[i].p) ++i;
    if (i == BLOCKS) abort();
    blocks[i] = (Block){*p, bytes, dev};
    pthread_mutex_unlock(&mu);
    return hipSuccess;
}
static hipError_t drop(void *p, int host) {
    if (!p) return hipSuccess;
    pthread_mutex_lock(&mu);
    int i = 0;
    while (i < BLOCKS && !(blocks[i].p == p && (blocks[i].device < 0) == host)) ++i;
    if (i == BLOCKS) abort(); /* freed twice, or not its own */
    blocks[i].p = NULL;
    pthread_mutex_unlock(&mu);
    free(p);
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t bytes) {
    MAY_FAIL;
    __sync_fetch_and_add(&calls_malloc, 1);
    if (bytes >= 1 << 20) __sync_fetch_and_add(&calls_large, 1);
    if (delay_ms) usleep(1000 * delay_ms);
    if (limit && fake_live(device) + bytes > limit) return last_error = hipErrorOutOfMemory;
    return get(p, bytes, device);
}
hipError_t hipFree(void *p) {
    __sync_fetch_and_add(&calls_free, 1);
    return drop(p, 0);
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    MAY_FAIL;
    __sync_fetch_and_add(&calls_host_malloc, 1);
    return get(p, bytes, -1);
}
hipError_t hipHostFree(void *p) {
    __sync_fetch_and_add(&calls_host_free, 1);
    return drop(p, 1);
}

static struct ihipStream_t *of(hipStream_t s) { return s ? s : &null_stream; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned flags) {
    MAY_FAIL;
    pthread_mutex_lock(&mu);
    int i = 0;
    while (i < 256 && streams[i].used) ++i;
    if (i == 256) abort();
    streams[i].used = 1;
    *s = &streams[i];
    pthread_mutex_unlock(&mu);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    s->busy = s->used = 0;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    MAY_FAIL;
    of(s)->busy = 0;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) {
    for (int i = 0; i < 256; ++i) streams[i].busy = 0;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t s) {
    MAY_FAIL;
    memcpy(dst, src, n);
    of(s)->busy = 1;
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind kind) {
    MAY_FAIL;
    memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *dst, int v, size_t n, hipStream_t s) {
    MAY_FAIL;
    memset(dst, v, n);
    of(s)->busy = 1;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t s) {
    MAY_FAIL;
    of(s)->busy = 1;
    return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void *f, dim3 grid, dim3 block, void **args, unsigned lds, hipStream_t s) {
    MAY_FAIL;
    of(s)->busy = 1;
    return hipSuccess;
}
static __thread struct { dim3 grid, block; size_t lds; hipStream_t s; } config;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    config.grid = grid;
    config.block = block;
    config.lds = lds;
    config.s = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = config.grid;
    *block = config.block;
    *lds = config.lds;
    *s = config.s;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *data) {
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **h) {}
void __hipRegisterFunction(void **h, const void *f, char *name, const char *dev, unsigned n, void *a, void *b, void *c,
                           void *d, int *e) {}
void __hipRegisterVar(void **h, void *v, char *host, char *dev, int ext, size_t n, int konst, int global) {}
hipError_t hipGetSymbolAddress(void **p, const void *sym) {
    static void *scratch;
    MAY_FAIL;
    if (!scratch) scratch = malloc((size_t)32 << 20);
    *p = scratch;
    return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t *e) {
    MAY_FAIL;
    *e = malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    MAY_FAIL;
    of(s)->busy = 1;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    MAY_FAIL;
    return hipDeviceSynchronize();
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
    MAY_FAIL;
    *ms = 1.0f;
    return hipSuccess;
}

hipError_t hipGetDevice(int *d) {
    MAY_FAIL;
    *d = device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    if (d < 0 || d >= DEVICES) return hipErrorInvalidDevice;
    device = d;
    return hipSuccess;
}
#undef hipGetDeviceProperties
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d) {
    MAY_FAIL;
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->cooperativeLaunch = 1;
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return "made to fail"; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int threads, size_t lds) {
    MAY_FAIL;
    *n = 1;
    return hipSuccess;
}
