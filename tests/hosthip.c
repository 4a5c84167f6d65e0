/* The HIP runtime calls of libfd23.so on host memory, for tests of the code
 * around the kernels: device memory is calloc'ed, launches are counted and
 * nothing runs.  The hh_* variables set limits and count calls. */
#include <stdlib.h>
#include <string.h>

typedef struct {
    unsigned x, y, z;
} dim3_;

long hh_room = 1L << 40;   /* bytes hipMalloc may still give */
long hh_graphs, hh_held, hh_launches, hh_mallocs, hh_copied, hh_async;
int hh_error;              /* the error hipGetLastError returns next */

static int failed(int e) {
    if (e) hh_error = e;
    return e;
}

int hipMalloc(void **p, size_t n) {
    if ((long)n > hh_room) return failed(2);
    long *b = calloc(1, n + 64);
    b[0] = (long)n;
    hh_room -= (long)n;
    hh_mallocs++;
    *p = (char *)b + 64;
    return 0;
}
int hipFree(void *p) {
    if (!p) return 0;
    long *b = (long *)((char *)p - 64);
    hh_room += b[0];
    free(b);
    return 0;
}
int hipMemGetInfo(size_t *f, size_t *t) {
    *f = (size_t)hh_room;
    *t = (size_t)1 << 40;
    return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) {
    (void)kind;
    memcpy(d, s, n);
    hh_copied += (long)n;
    return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
    (void)st;
    hh_async++;
    return hipMemcpy(d, s, n, kind);
}
int hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int kind) {
    for (size_t i = 0; i < h; i++) hipMemcpy((char *)d + i * dp, (const char *)s + i * sp, w, kind);
    return 0;
}
int hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int kind, void *st) {
    return (void)st, hipMemcpy2D(d, dp, s, sp, w, h, kind);
}
int hipMemset(void *d, int v, size_t n) { return memset(d, v, n), 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { return (void)st, hipMemset(d, v, n); }

int hipLaunchKernel(const void *f, dim3_ g, dim3_ b, void **a, size_t n, void *st) {
    (void)f, (void)g, (void)b, (void)a, (void)n, (void)st;
    hh_launches++;
    return 0;
}
static dim3_ cfg_g, cfg_b;
static size_t cfg_n;
static void *cfg_s;
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t n, void *st) {
    cfg_g = g, cfg_b = b, cfg_n = n, cfg_s = st;
    return 0;
}
int __hipPopCallConfiguration(dim3_ *g, dim3_ *b, size_t *n, void **st) {
    *g = cfg_g, *b = cfg_b, *n = cfg_n, *st = cfg_s;
    return 0;
}
static void *module_[1];
void **__hipRegisterFatBinary(const void *d) { return (void)d, module_; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}
static char symbol_[64 << 20];
int hipGetSymbolAddress(void **p, const void *s) { return (void)s, *p = symbol_, 0; }

int hipGetLastError(void) {
    const int e = hh_error;
    hh_error = 0;
    return e;
}
const char *hipGetErrorString(int e) { return e == 2 ? "out of memory" : e ? "error" : "no error"; }
int hipGetDevice(int *d) { return *d = 0, 0; }
int hipSetDevice(int d) { return (void)d, 0; }
int hipDeviceSynchronize(void) { return 0; }

static int object_;
static int made(void **p) { return *p = &object_, 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) { return (void)f, made(s); }
int hipStreamDestroy(void *s) { return (void)s, 0; }
int hipStreamSynchronize(void *s) { return (void)s, 0; }
int hipStreamGetDevice(void *s, int *d) { return (void)s, *d = 0, 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { return (void)s, (void)e, (void)f, 0; }
int hipStreamBeginCapture(void *s, int m) { return (void)s, (void)m, 0; }
int hipStreamEndCapture(void *s, void **g) { return (void)s, made(g); }
int hipGraphInstantiate(void **x, void *g, void *n, char *l, size_t b) {
    (void)g, (void)n, (void)l, (void)b;
    hh_graphs++;
    hh_held++;
    return made(x);
}
int hipGraphDestroy(void *g) { return (void)g, 0; }
int hipGraphExecDestroy(void *x) { return (void)x, hh_held--, 0; }
int hipGraphLaunch(void *x, void *s) { return (void)x, (void)s, 0; }
int hipEventCreate(void **e) { return made(e); }
int hipEventCreateWithFlags(void **e, unsigned f) { return (void)f, made(e); }
int hipEventDestroy(void *e) { return (void)e, 0; }
int hipEventRecord(void *e, void *s) { return (void)e, (void)s, 0; }
int hipEventQuery(void *e) { return (void)e, 0; }
int hipEventSynchronize(void *e) { return (void)e, 0; }
int hipEventElapsedTime(float *t, void *a, void *b) { return (void)a, (void)b, *t = 1.0f, 0; }
