/* The HIP calls of libsassena_amd.so on host memory, for tests of its host side
 * without a GPU: allocations of a device of set size, copies in stream order at
 * the next synchronisation, kernels recorded by name and not run.  Loaded with
 * RTLD_GLOBAL before the library, whose undefined symbols then resolve here. */
#define _GNU_SOURCE
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

typedef struct { unsigned x, y, z; } dim3_t;
enum { kOk = 0, kInvalid = 1, kNoMemory = 2, kMax = 1 << 16 };

static size_t total = (size_t)8 << 30, used;
static int last_error;
static struct { void *p; size_t n; } blocks[4096];
static struct { const void *fn; const char *name; } kernels[1024];
static int nkernels, nlaunches, nqueue, stale;
static struct { const char *name; dim3_t grid; unsigned char arg[128]; } launches[kMax];
static struct { void *dst; const void *src; size_t n; uint64_t sum; int fill, byte; } queue[kMax];

static int err(int e) { if (e) last_error = e; return e; }

static uint64_t sum(const void *p, size_t n) {
    uint64_t h = 1469598103934665603ull;
    for (size_t i = 0; i < n; ++i) h = (h ^ ((const unsigned char *)p)[i]) * 1099511628211ull;
    return h;
}

static int on_device(const void *p) {
    for (int i = 0; i < 4096; ++i)
        if (blocks[i].p && (const char *)p >= (char *)blocks[i].p && (const char *)p < (char *)blocks[i].p + blocks[i].n)
            return 1;
    return 0;
}

static void drain(void) {
    for (int i = 0; i < nqueue; ++i) {
        if (queue[i].fill) {
            memset(queue[i].dst, queue[i].byte, queue[i].n);
        } else {
            /* a source on the host must still hold what it held when the copy was queued */
            if (!on_device(queue[i].src) && sum(queue[i].src, queue[i].n) != queue[i].sum) ++stale;
            memcpy(queue[i].dst, queue[i].src, queue[i].n);
        }
    }
    nqueue = 0;
}

/* what the tests set and read */
void fake_memory(size_t bytes) { total = bytes; }
size_t fake_used(void) { return used; }
void fake_forget(void) { nlaunches = 0; }
int fake_launches(void) { return nlaunches; }
const char *fake_name(int i) { return launches[i].name; }
unsigned fake_grid(int i, int k) { return k == 0 ? launches[i].grid.x : k == 1 ? launches[i].grid.y : launches[i].grid.z; }
const void *fake_arg(int i) { return launches[i].arg; }
int fake_stale(void) { return stale; }

void **__hipRegisterFatBinary(const void *d) { (void)d; static void *h; return &h; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t n, int c, int g) {
    (void)m, (void)v, (void)h, (void)d, (void)e, (void)n, (void)c, (void)g;
}
void __hipRegisterFunction(void **m, const void *fn, char *host, const char *name, unsigned t, void *a, void *b, void *c,
                           void *d, int *e) {
    (void)m, (void)host, (void)t, (void)a, (void)b, (void)c, (void)d, (void)e;
    if (nkernels < 1024) { kernels[nkernels].fn = fn; kernels[nkernels++].name = name; }
}
static struct { dim3_t grid, block; size_t lds; void *stream; } config;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void *s) {
    config.grid = g, config.block = b, config.lds = lds, config.stream = s;
    return kOk;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *lds, void **s) {
    *g = config.grid, *b = config.block, *lds = config.lds, *s = config.stream;
    return kOk;
}
int hipLaunchKernel(const void *fn, dim3_t grid, dim3_t block, void **args, size_t lds, void *s) {
    (void)block, (void)lds, (void)s;
    if (grid.x == 0 || grid.y == 0 || grid.z == 0 || grid.y > 65535 || grid.z > 65535) return err(kInvalid);
    if (nlaunches == kMax) abort();
    launches[nlaunches].name = "?";
    for (int i = 0; i < nkernels; ++i)
        if (kernels[i].fn == fn) launches[nlaunches].name = kernels[i].name;
    launches[nlaunches].grid = grid;
    memcpy(launches[nlaunches++].arg, args[0], 128);
    return kOk;
}

int hipMalloc(void **p, size_t n) {
    *p = NULL;
    if (used + n > total) return err(kNoMemory);
    for (int i = 0; i < 4096; ++i)
        if (!blocks[i].p) {
            void *q = mmap(NULL, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
            if (q == MAP_FAILED) return err(kNoMemory);
            blocks[i].p = *p = q;
            blocks[i].n = n;
            used += n;
            return kOk;
        }
    abort();
}
int hipFree(void *p) {
    if (!p) return kOk;
    drain();
    for (int i = 0; i < 4096; ++i)
        if (blocks[i].p == p) {
            munmap(p, blocks[i].n);
            used -= blocks[i].n;
            blocks[i].p = NULL;
            return kOk;
        }
    return err(kInvalid);
}
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; return (*p = calloc(1, n)) ? kOk : err(kNoMemory); }
int hipHostFree(void *p) { drain(); free(p); return kOk; }
int hipMemGetInfo(size_t *f, size_t *t) { *f = total > used ? total - used : 0; *t = total; return kOk; }
static int push(void *dst, const void *src, size_t n, int fill, int byte) {
    if (!dst || (!fill && !src)) return err(kInvalid);
    if (nqueue == kMax) abort();
    queue[nqueue].dst = dst, queue[nqueue].src = src, queue[nqueue].n = n;
    queue[nqueue].fill = fill, queue[nqueue].byte = byte;
    queue[nqueue++].sum = fill || on_device(src) ? 0 : sum(src, n);
    return kOk;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)k, (void)st; return push(d, s, n, 0, 0); }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; drain(); memcpy(d, s, n); return kOk; }
int hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int k, void *st) {
    (void)k, (void)st;
    drain();
    for (size_t i = 0; i < h; ++i) memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
    return kOk;
}
int hipMemsetAsync(void *d, int v, size_t n, void *s) { (void)s; return push(d, NULL, n, 1, v); }
int hipStreamSynchronize(void *s) { (void)s; drain(); return kOk; }
int hipEventSynchronize(void *e) { (void)e; drain(); return kOk; }
static int handle(void **h) { static char some; *h = &some; return kOk; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; return handle(s); }
int hipStreamDestroy(void *s) { (void)s; return kOk; }
int hipEventCreate(void **e) { return handle(e); }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; return handle(e); }
int hipEventDestroy(void *e) { (void)e; return kOk; }
int hipEventRecord(void *e, void *s) { (void)e, (void)s; return kOk; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a, (void)b; *ms = 1.0f; return kOk; }
int hipSetDevice(int d) { (void)d; return kOk; }
int hipGetDeviceCount(int *n) { *n = 1; return kOk; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a, (void)d; *v = 256; return kOk; }
int hipFuncSetAttribute(const void *f, int a, int v) { (void)f, (void)a, (void)v; return kOk; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l) {
    (void)f, (void)b, (void)l;
    *n = 2;
    return kOk;
}
int hipGetSymbolAddress(void **p, const void *s) {
    (void)s;
    *p = mmap(NULL, (size_t)8 << 30, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return *p == MAP_FAILED ? err(kNoMemory) : kOk;
}
int hipGetLastError(void) { const int e = last_error; last_error = kOk; return e; }
const char *hipGetErrorString(int e) { return e == kNoMemory ? "out of memory" : e ? "error" : "no error"; }
