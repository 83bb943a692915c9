/* A HIP runtime of host memory for CPU tests of the library's host code, preloaded in place of the
 * real one: memory is malloc's, kernels do nothing, and every asynchronous call leaves its stream
 * busy until that stream (or an event after the call, or the device) is waited for.  After
 * fake_arm(k), the k-th kernel launch fails (0: none). */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, FAILED = 719 /* hipErrorLaunchFailure */, STREAMS = 64 };
static int busy[STREAMS], nstream = 1, launches, fail_at, capturing;
static int overlaps; /* launches on other streams while the null stream has work, since fake_arm() */
static int live; /* allocations not freed */
static size_t watched; /* allocations of exactly this size are counted */
static int seen;
static uintptr_t last_error;

static int idx(void* s) { return (int)(uintptr_t)s; } /* stream 0: the null stream */

void fake_arm(int k) { launches = 0, fail_at = k, overlaps = 0; }
int fake_overlaps(void) { return overlaps; }
int fake_live(void) { return live; }
void fake_watch(size_t n) { watched = n, seen = 0; }
int fake_seen(void) { return seen; }
int fake_launches(void) { return launches; }
int fake_busy(void) { /* operations not waited for */
    int n = 0;
    for (int i = 0; i < nstream; ++i) n += busy[i];
    return n;
}

int hipMalloc(void** p, size_t n) { return ++live, seen += n == watched, *p = calloc(1, n ? n : 1), OK; }
int hipExtMallocWithFlags(void** p, size_t n, unsigned f) { return (void)f, hipMalloc(p, n); }
int hipFree(void* p) { return live -= p != NULL, free(p), OK; }
int hipMemcpy(void* d, const void* s, size_t n, int k) { return (void)k, memmove(d, s, n), busy[0] = 0, OK; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { return (void)k, memmove(d, s, n), ++busy[idx(st)], OK; }
int hipMemcpyWithStream(void* d, const void* s, size_t n, int k, void* st) { return (void)k, memmove(d, s, n), busy[idx(st)] = 0, OK; }
int hipMemcpy2D(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int k) {
    (void)k;
    for (size_t i = 0; i < h; ++i) memmove((char*)d + i * dp, (const char*)s + i * sp, w);
    return busy[0] = 0, OK;
}
int hipMemset(void* d, int v, size_t n) { return memset(d, v, n), ++busy[0], OK; } /* returns before it is done */
int hipMemsetAsync(void* d, int v, size_t n, void* st) { return memset(d, v, n), ++busy[idx(st)], OK; }
int hipStreamCreateWithFlags(void** s, unsigned f) { return (void)f, *s = (void*)(uintptr_t)nstream++, OK; }
int hipStreamDestroy(void* s) { return (void)s, OK; }
int hipStreamSynchronize(void* s) { return busy[idx(s)] = 0, OK; }
int hipDeviceSynchronize(void) { return memset(busy, 0, sizeof busy), OK; }
int hipEventCreate(void** e) { return *e = calloc(1, sizeof(int)), OK; }
int hipEventDestroy(void* e) { return free(e), OK; }
int hipEventRecord(void* e, void* s) { return *(int*)e = idx(s), OK; }
int hipEventSynchronize(void* e) { return busy[*(int*)e] = 0, OK; }
int hipEventElapsedTime(float* ms, void* a, void* b) { return (void)a, (void)b, *ms = 0.f, OK; }
int hipGetDevice(int* d) { return *d = 0, OK; }
int hipDeviceGetAttribute(int* v, int a, int d) { return (void)a, (void)d, *v = 0, OK; }
int hipGetLastError(void) { int e = (int)last_error; return last_error = 0, e; }
const char* hipGetErrorString(int e) { return e ? "failed on request" : "no error"; }
int hipPointerGetAttributes(void* a, const void* p) { return (void)a, (void)p, last_error = 1; } /* no pinned memory */
int hipFuncSetAttribute(const void* f, int a, int v) { return (void)f, (void)a, (void)v, OK; }
int hipGetSymbolAddress(void** p, const void* s) { return *p = (void*)s, OK; }
int hipStreamBeginCapture(void* s, int m) { return (void)s, (void)m, capturing = 1, OK; }
int hipStreamEndCapture(void* s, void** g) { return (void)s, *g = NULL, capturing = 0, OK; }
int hipGraphInstantiate(void** x, void* g, void** n, char* l, size_t b) { return (void)g, (void)n, (void)l, (void)b, *x = calloc(1, 1), OK; }
int hipGraphDestroy(void* g) { return (void)g, OK; }
int hipGraphExecDestroy(void* x) { return free(x), OK; }
int hipGraphLaunch(void* x, void* s) { return (void)x, ++busy[idx(s)], OK; }
typedef struct { unsigned x, y, z; } dim3_;
int hipLaunchKernel(const void* f, dim3_ g, dim3_ b, void** a, size_t l, void* st) {
    (void)f, (void)g, (void)b, (void)a, (void)l;
    overlaps += st && busy[0];
    if (++launches == fail_at) return last_error = FAILED;
    return busy[idx(st)] += !capturing, OK;
}
static struct { dim3_ g, b; size_t l; void* s; } call;
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t l, void* s) { return call.g = g, call.b = b, call.l = l, call.s = s, OK; }
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* l, void** s) { return *g = call.g, *b = call.b, *l = call.l, *s = call.s, OK; }
void** __hipRegisterFatBinary(const void* d) { static void* h; return (void)d, &h; }
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** h, const void* f, char* d, const char* n, unsigned t, void* a, void* b, void* c, void* e, int* w) {
    (void)h, (void)f, (void)d, (void)n, (void)t, (void)a, (void)b, (void)c, (void)e, (void)w;
}
void __hipRegisterVar(void** h, void* v, char* a, const char* n, int e, size_t s, int c, int g) {
    (void)h, (void)v, (void)a, (void)n, (void)e, (void)s, (void)c, (void)g;
}
