/* A HIP runtime of host memory for tests of the engine's error paths: loaded
 * with RTLD_GLOBAL before libsteps_amd.so, its functions take the place of
 * libamdhip64's.  Kernels do not run, but their launches are counted by name.
 * While `busy` is set no event has happened yet.  hipMalloc fails above a limit for
 * one allocation or a capacity for all, and an
 * error stays the thread's last error until hipGetLastError reads it, past
 * later calls that succeed, as the HIP 7 documentation states. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

typedef struct { unsigned x, y, z; } dim3_t;

static _Thread_local int last_error;
static size_t limit = (size_t)-1, capacity = (size_t)-1, largest, live;
static int pinned_fails;
static volatile int busy;

void fake_set_limit(size_t bytes) { limit = bytes; }
void fake_set_capacity(size_t bytes) { capacity = bytes; }
void fake_set_pinned_fails(int on) { pinned_fails = on; }
void fake_set_busy(int on) { busy = on; }
size_t fake_largest(void) { size_t v = largest; largest = 0; return v; }  /* since the last call */
size_t fake_live(void) { return live; }

static int put(void **p, size_t n, int device) {
    size_t *b = malloc(n + 64);
    if (!b) abort();
    *b = n;
    *p = (char *)b + 64;
    if (device) {
        live += n;
        if (n > largest) largest = n;
    }
    return 0;
}
int hipMalloc(void **p, size_t n) {
    if (n > limit || n > capacity || live > capacity - n) {
        *p = NULL;
        return last_error = 2; /* hipErrorOutOfMemory */
    }
    return put(p, n, 1);
}
int hipFree(void *p) {
    if (p) {
        live -= *(size_t *)((char *)p - 64);
        free((char *)p - 64);
    }
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    (void)flags;
    if (pinned_fails) return last_error = 2;
    return put(p, n, 0);
}
int hipHostFree(void *p) { free((char *)p - 64); return 0; }
int hipGetLastError(void) { int e = last_error; last_error = 0; return e; }
const char *hipGetErrorString(int e) { return e == 2 ? "out of memory" : "error"; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipDeviceGetAttribute(int *v, int attr, int dev) { (void)attr; (void)dev; *v = 256; return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int kind) { (void)kind; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) { (void)kind; (void)st; memcpy(d, s, n); return 0; }
int hipMemset(void *d, int v, size_t n) { memset(d, v, n); return 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)st; memset(d, v, n); return 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = (void *)1; return 0; }
int hipStreamDestroy(void *s) { (void)s; return 0; }
int hipStreamSynchronize(void *s) { (void)s; return 0; }
int hipEventCreate(void **e) { *e = (void *)1; return 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = (void *)1; return 0; }
int hipEventDestroy(void *e) { (void)e; return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventQuery(void *e) { (void)e; return busy ? 600 : 0; } /* hipErrorNotReady */
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 0; return 0; }

/* device variables (the engine has one, its static scratch) */
static size_t var_size;
static void *var;
int hipGetSymbolAddress(void **p, const void *symbol) {
    (void)symbol;
    if (!var && !(var = malloc(var_size))) return last_error = 2;
    *p = var;
    return 0;
}

/* launches by kernel name */
#define MAX_KERNELS 4096
static struct { const void *f; const char *name; long launches, blocks; } kernels[MAX_KERNELS];
static int nkernels;
static _Thread_local struct { dim3_t g, b; size_t sh; void *st; } config;

void **__hipRegisterFatBinary(const void *data) { (void)data; return (void **)&nkernels; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *f, char *device_fun, const char *name, unsigned limit_, void *tid,
                           void *bid, dim3_t *bd, dim3_t *gd, int *ws) {
    (void)m; (void)device_fun; (void)limit_; (void)tid; (void)bid; (void)bd; (void)gd; (void)ws;
    if (nkernels == MAX_KERNELS) abort();
    kernels[nkernels].f = f;
    kernels[nkernels++].name = name;
}
void __hipRegisterVar(void **m, void *v, char *host, char *device, int ext, size_t size, int constant, int global) {
    (void)m; (void)v; (void)host; (void)device; (void)ext; (void)constant; (void)global;
    var_size = size;
}
/* launches (or, blocks != 0, workgroups) of the kernels whose names hold `part`, since the last reset */
long fake_launches(const char *part, int blocks) {
    long n = 0;
    for (int i = 0; i < nkernels; ++i)
        if (strstr(kernels[i].name, part)) n += blocks ? kernels[i].blocks : kernels[i].launches;
    return n;
}
void fake_reset_launches(void) {
    for (int i = 0; i < nkernels; ++i) kernels[i].launches = kernels[i].blocks = 0;
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t sh, void *st) {
    config.g = g;
    config.b = b;
    config.sh = sh;
    config.st = st;
    return 0;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *sh, void **st) {
    *g = config.g;
    *b = config.b;
    *sh = config.sh;
    *st = config.st;
    return 0;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t sh, void *st) {
    (void)b; (void)args; (void)sh; (void)st;
    for (int i = 0; i < nkernels; ++i)
        if (kernels[i].f == f) {
            kernels[i].launches++;
            kernels[i].blocks += (long)g.x * g.y * g.z;
            return 0;
        }
    return last_error = 98; /* hipErrorInvalidDeviceFunction */
}
