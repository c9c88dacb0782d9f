/* A HIP runtime of host memory for CPU tests of the library's host code: loaded before the library,
 * its functions stand in front of the real runtime's. Allocations come from the heap and copies are
 * copies; a kernel launch does nothing. fake_fail_at(n) makes the n-th following device allocation
 * (from 1) fail once. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, OUT_OF_MEMORY = 2 };

static long live, count, fail_at, graph_launches;
static int last_error;

void fake_fail_at(long n) { fail_at = n > 0 ? count + n : 0; }
long fake_live(void) { return live; }
long fake_allocations(void) { return count; }
long fake_graph_launches(void) { return graph_launches; }

static int done(int e) {
    if (e != OK) last_error = e;
    return e;
}

int hipMalloc(void **p, size_t n) {
    *p = NULL;
    if (++count == fail_at) return done(OUT_OF_MEMORY);
    *p = calloc(1, n + 512);
    if (!*p) return done(OUT_OF_MEMORY);
    /* 256-byte aligned, the block's start kept in front */
    char *a = (char *)(((size_t)*p + sizeof(void *) + 255) & ~(size_t)255);
    memcpy(a - sizeof(void *), p, sizeof(void *));
    *p = a;
    ++live;
    return OK;
}
int hipFree(void *p) {
    if (p) {
        void *b;
        memcpy(&b, (char *)p - sizeof(void *), sizeof b);
        free(b);
        --live;
    }
    return OK;
}
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = calloc(1, n); return *p ? OK : done(OUT_OF_MEMORY); }
int hipHostFree(void *p) { free(p); return OK; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memcpy(d, s, n); return OK; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)k; (void)st; memcpy(d, s, n); return OK; }
int hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int k) {
    (void)k;
    for (size_t i = 0; i < h; ++i) memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
    return OK;
}
int hipMemset(void *d, int v, size_t n) { memset(d, v, n); return OK; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)st; memset(d, v, n); return OK; }
int hipMemsetD32Async(void *d, int v, size_t n, void *st) {
    (void)st;
    for (size_t i = 0; i < n; ++i) ((int *)d)[i] = v;
    return OK;
}
int hipGetDevice(int *d) { *d = 0; return OK; }
int hipSetDevice(int d) { (void)d; return OK; }
int hipGetDeviceCount(int *n) { *n = 1; return OK; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return OK; }
int hipDeviceSynchronize(void) { return OK; }
int hipGetLastError(void) { int e = last_error; last_error = OK; return e; }
const char *hipGetErrorString(int e) { return e == OK ? "no error" : "out of memory"; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int t, size_t l) {
    (void)f; (void)t; (void)l;
    *n = 2;
    return OK;
}

static int object;                        /* streams, events and graphs have no state */
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = &object; return OK; }
int hipStreamDestroy(void *s) { (void)s; return OK; }
int hipStreamSynchronize(void *s) { (void)s; return OK; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return OK; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = &object; return OK; }
int hipEventCreate(void **e) { *e = &object; return OK; }
int hipEventDestroy(void *e) { (void)e; return OK; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return OK; }
int hipEventSynchronize(void *e) { (void)e; return OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return OK; }
int hipGraphInstantiate(void **x, void *g, void *n, char *l, size_t z) {
    (void)g; (void)n; (void)l; (void)z;
    *x = &object;
    return OK;
}
int hipGraphLaunch(void *x, void *s) { (void)x; (void)s; ++graph_launches; return OK; }
int hipGraphDestroy(void *g) { (void)g; return OK; }
int hipGraphExecDestroy(void *x) { (void)x; return OK; }

/* dim3 arguments are passed as the compiler's launch stubs pass them: by value, 12 bytes each */
typedef struct { unsigned x, y, z; } dim3_t;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t l, void *s) { (void)g; (void)b; (void)l; (void)s; return OK; }
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *l, void **s) {
    g->x = g->y = g->z = b->x = b->y = b->z = 1;
    *l = 0;
    *s = NULL;
    return OK;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **a, size_t l, void *s) {
    (void)f; (void)g; (void)b; (void)a; (void)l; (void)s;
    return OK;
}
