/* A HIP runtime of host memory for tests of the engine's error paths: loaded
 * with RTLD_GLOBAL before libsteps_amd.so, its functions take the place of
 * libamdhip64's.  Kernels do not run.  hipMalloc fails above a limit for
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

void fake_set_limit(size_t bytes) { limit = bytes; }
void fake_set_capacity(size_t bytes) { capacity = bytes; }
void fake_set_pinned_fails(int on) { pinned_fails = on; }
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
int hipEventQuery(void *e) { (void)e; return 0; }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 0; return 0; }
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t sh, void *st) { (void)g; (void)b; (void)sh; (void)st; return 0; }
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *sh, void **st) {
    g->x = g->y = g->z = b->x = b->y = b->z = 1;
    *sh = 0;
    *st = NULL;
    return 0;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t sh, void *st) {
    (void)f; (void)g; (void)b; (void)args; (void)sh; (void)st;
    return 0;
}
