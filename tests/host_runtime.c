/* Stand-in for the HIP runtime in tests of the library's host code: device
 * memory is host memory, kernels do not run. Loaded before libfesom_gpu.so, so
 * that the library's calls resolve to it. It counts what is enqueued on
 * another stream while a fill of the null stream may still run (hipMemset
 * returns before the fill has ended, and a non-blocking stream does not wait
 * for the null stream), and what the null stream reads or writes while a fill of
 * another stream may still run there. It can let the n-th allocation from now
 * fail. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

#define EXPORT __attribute__((visibility("default")))
typedef struct { unsigned x, y, z; } dim3_t;
enum { NOMEM = 2, D2D = 3 };

static int pending, hazards, fail_in = -1;
static size_t live;
static struct { char *p; size_t n; } fill[64];   /* fills of the other streams that may still run */
static int fills;

EXPORT int host_hazards(void) { return hazards; }
EXPORT void host_fail_in(int n) { fail_in = n; }   /* 0: the next allocation; < 0: none */
EXPORT int host_fail_left(void) { return fail_in; }
EXPORT size_t host_live_bytes(void) { return live; }

static int used(void *stream)
{
    if (stream && pending) ++hazards;
    return 0;
}
static int waited(void)
{
    pending = 0;
    return 0;
}
static void touched(const void *q, size_t n)
{
    for (int i = 0; i < fills; ++i)
        if ((const char *)q < fill[i].p + fill[i].n && fill[i].p < (const char *)q + n) ++hazards;
}

EXPORT int hipMalloc(void **p, size_t n)
{
    if (fail_in == 0) {
        fail_in = -1;
        return NOMEM;
    }
    if (fail_in > 0) --fail_in;
    size_t *q = calloc(1, n + 64);
    q[0] = n;
    live += n;
    *p = (char *)q + 64;
    return 0;
}
EXPORT int hipFree(void *p)
{
    if (p) {
        size_t *q = (size_t *)((char *)p - 64);
        live -= q[0];
        free(q);
    }
    fills = 0;   /* waits for the device */
    return waited();
}
EXPORT int hipHostMalloc(void **p, size_t n, unsigned flags) { (void)flags; *p = calloc(1, n); return 0; }
EXPORT int hipHostFree(void *p) { free(p); return waited(); }
EXPORT int hipMemset(void *p, int v, size_t n) { touched(p, n); memset(p, v, n); pending = 1; return 0; }
EXPORT int hipMemsetAsync(void *p, int v, size_t n, void *s)
{
    memset(p, v, n);
    if (!s) {
        touched(p, n);
        pending = 1;
    } else if (fills < 64) {
        fill[fills].p = p;
        fill[fills++].n = n;
    } else {
        abort();
    }
    return used(s);
}
EXPORT int hipMemcpy(void *d, const void *s, size_t n, int kind)
{
    touched(d, n);
    touched(s, n);
    memmove(d, s, n);
    if (kind == D2D) pending = 1;
    else waited();
    return 0;
}
EXPORT int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st)
{
    (void)kind;
    if (!st) {
        touched(d, n);
        touched(s, n);
    }
    memmove(d, s, n);
    return used(st);
}
EXPORT int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **a, size_t l, void *s)
{
    (void)f; (void)g; (void)b; (void)a; (void)l;
    return used(s);
}
EXPORT int hipGraphLaunch(void *g, void *s) { (void)g; return used(s); }
EXPORT int hipStreamSynchronize(void *s)
{
    if (!s) return waited();
    fills = 0;   /* one stream a context, one context at a time in the tests that fill */
    return 0;
}

EXPORT int hipGetDeviceCount(int *n) { *n = 1; return 0; }
EXPORT int hipSetDevice(int d) { (void)d; return 0; }
EXPORT int hipGetLastError(void) { return 0; }
EXPORT const char *hipGetErrorString(int e) { return e == NOMEM ? "out of memory" : "error"; }
EXPORT int hipGetSymbolAddress(void **p, const void *s) { (void)s; *p = 0; return 0; }
static char handle;
EXPORT int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = &handle; return 0; }
EXPORT int hipStreamDestroy(void *s) { (void)s; return 0; }
EXPORT int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return 0; }
EXPORT int hipStreamEndCapture(void *s, void **g) { (void)s; *g = &handle; return 0; }
EXPORT int hipGraphInstantiate(void **e, void *g, void *n, char *b, size_t l) { (void)g; (void)n; (void)b; (void)l; *e = &handle; return 0; }
EXPORT int hipGraphDestroy(void *g) { (void)g; return 0; }
EXPORT int hipGraphExecDestroy(void *g) { (void)g; return 0; }
EXPORT int hipEventCreate(void **e) { *e = &handle; return 0; }
EXPORT int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = &handle; return 0; }
EXPORT int hipEventDestroy(void *e) { (void)e; return 0; }
EXPORT int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
EXPORT int hipEventSynchronize(void *e) { (void)e; return 0; }
EXPORT int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return 0; }

static dim3_t grid, block;
static size_t shared;
static void *on;
EXPORT int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t l, void *s) { grid = g; block = b; shared = l; on = s; return 0; }
EXPORT int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *l, void **s) { *g = grid; *b = block; *l = shared; *s = on; return 0; }
EXPORT void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }
EXPORT void __hipRegisterFunction(void **m, const void *h, char *d, const char *n, unsigned t, void *a, void *b, void *c, void *e, int *w)
{
    (void)m; (void)h; (void)d; (void)n; (void)t; (void)a; (void)b; (void)c; (void)e; (void)w;
}
EXPORT void __hipRegisterVar(void **m, void *v, char *d, char *n, int e, size_t s, int c, int g)
{
    (void)m; (void)v; (void)d; (void)n; (void)e; (void)s; (void)c; (void)g;
}
EXPORT void __hipUnregisterFatBinary(void **m) { (void)m; }
