/* A HIP runtime without a device, for tests of the host side on a machine without a GPU: device memory is
   host memory, copies and fills happen at once, kernels are counted and do nothing.  Loaded with
   RTLD_GLOBAL before libsrx.so, it answers the library's calls into the runtime.
   host_fail_launch(k): the k-th launch from now (0: the next) fails, -1: none;
   host_launches(): launches since the last host_fail_launch.
   host_device_blocks(): device allocations not yet freed;
   host_pinned_bytes(): pinned memory handed out so far;
   host_stop_after(k): increments from now on stop after k outer iterations (host_control.cpp answers for
   the control and reduction kernels);
   host_watch_pointer(i): from now on, note the pointer every launch passes as its argument i (-1: none);
   host_pointer_offsets(): the bits set in any of their distances from the first. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;
static long launches, fail_at = -1;
static int last_error;

void host_fail_launch(long k) { launches = 0; fail_at = k; last_error = 0; }
long host_launches(void) { return launches; }

static int watched = -1;
static uintptr_t first_pointer, offsets;
void host_watch_pointer(int i) { watched = i; first_pointer = offsets = 0; }
long host_pointer_offsets(void) { return (long)offsets; }

static const void *control, *reduce;
static int stop_after = 1;
void host_stop_after(int k) { stop_after = k; }
void host_control(void *block, int stop);
void host_reduce(int nvals, double *out);
int __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned t, void *a, void *b, void *c,
                          void *d, int *w) {
    (void)m; (void)dev; (void)t; (void)a; (void)b; (void)c; (void)d; (void)w;
    if (strstr(name, "9k_controlE")) control = host;
    if (strstr(name, "8k_reduceE")) reduce = host;
    return 0;
}

static int launch(const void *f, void **args) {
    if (f == control) host_control(*(void **)args[4], stop_after);
    if (f == reduce) host_reduce(*(int *)args[2], *(double **)args[4]);
    if (watched >= 0) {
        const uintptr_t p = *(uintptr_t *)args[watched];
        if (!first_pointer) first_pointer = p;
        offsets |= p - first_pointer;
    }
    if (launches++ == fail_at) last_error = 701; /* hipErrorLaunchOutOfResources */
    else return 0;
    return last_error;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **a, size_t m, void *s) {
    (void)g; (void)b; (void)m; (void)s;
    return launch(f, a);
}
int hipExtLaunchKernel(const void *f, dim3_t g, dim3_t b, void **a, size_t m, void *s, void *e0, void *e1, int fl) {
    (void)g; (void)b; (void)m; (void)s; (void)e0; (void)e1; (void)fl;
    return launch(f, a);
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t m, void *s) { (void)g; (void)b; (void)m; (void)s; return 0; }
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *m, void **s) {
    dim3_t one = {1, 1, 1};
    *g = *b = one; *m = 0; *s = 0;
    return 0;
}
int hipGetLastError(void) { int e = last_error; last_error = 0; return e; }
const char *hipGetErrorString(int e) { return e ? "launch refused by the test" : "no error"; }
static int get(void **p, size_t n) { *p = calloc(1, n ? n : 1); return *p ? 0 : 2; }
/* numbers in [1, 2) that follow no pattern, so that matrices left uncomputed in it are regular */
static long blocks;
long host_device_blocks(void) { return blocks; }
int hipMalloc(void **p, size_t n) {
    uint64_t r = 88172645463325252u;
    if (get(p, n)) return 2;
    ++blocks;
    for (size_t i = 0; i < n / 8; ++i) {
        r ^= r << 13; r ^= r >> 7; r ^= r << 17;
        ((uint64_t *)*p)[i] = (r >> 12) | 0x3ff0000000000000u;
    }
    return 0;
}
static size_t pinned;
long host_pinned_bytes(void) { return (long)pinned; }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; pinned += n; return get(p, n); }
int hipFree(void *p) { blocks -= p != 0; free(p); return 0; }
int hipHostFree(void *p) { free(p); return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memmove(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)k; (void)st; memmove(d, s, n); return 0; }
int hipMemset(void *d, int v, size_t n) { memset(d, v, n); return 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)st; memset(d, v, n); return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipGetSymbolAddress(void **p, const void *sym) { (void)sym; return get(p, 32u << 20); }
static int handle;
static int make(void **p) { *p = &handle; return 0; }
int hipStreamCreate(void **s) { return make(s); }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; return make(s); }
int hipStreamDestroy(void *s) { (void)s; return 0; }
int hipStreamSynchronize(void *s) { (void)s; return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { (void)s; (void)e; (void)f; return 0; }
int hipEventCreate(void **e) { return make(e); }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; return make(e); }
int hipEventDestroy(void *e) { (void)e; return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return 0; }
