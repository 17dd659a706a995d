/* The HIP calls that libspz makes, on host memory and without a device, for
 * tests/test_host_allocations.py (preloaded before the HIP runtime).  Device
 * and pinned memory are host memory, kernels are counted and do not run.
 * fake_fail makes allocations fail; fake_count and fake_bytes tell what the
 * library asked for. */
#include <hip/hip_runtime_api.h>

#include <stdlib.h>
#include <string.h>

enum { DEVICE = 0, PINNED = 1, LAUNCHES = 2, KINDS = 3 };
static long counts[KINDS], bytes_held[KINDS], fail_after[KINDS] = {-1, -1, -1};
static struct { void *p; size_t n; int kind; } held[4096];

/* the first `after` allocations of the kind (0 device, 1 pinned) from now on
 * succeed, the ones after them fail; -1: none fails */
void fake_fail(int kind, long after) { fail_after[kind] = after; }
/* allocations (0 device, 1 pinned) or kernel launches (2) so far */
long fake_count(int kind) { return counts[kind]; }
long fake_bytes(int kind) { return bytes_held[kind]; }

static hipError_t allocate(int kind, void **out, size_t n) {
    int i;
    *out = NULL;
    if (fail_after[kind] == 0) return hipErrorOutOfMemory;
    if (fail_after[kind] > 0) --fail_after[kind];
    for (i = 0; i < 4096 && held[i].p; ++i) {}
    if (i == 4096 || !(held[i].p = calloc(1, n ? n : 1))) return hipErrorOutOfMemory;
    held[i].n = n;
    held[i].kind = kind;
    ++counts[kind];
    bytes_held[kind] += (long)n;
    *out = held[i].p;
    return hipSuccess;
}
static hipError_t give_back(int kind, void *p) {
    int i;
    if (!p) return hipSuccess;
    for (i = 0; i < 4096; ++i)
        if (held[i].p == p && held[i].kind == kind) {
            bytes_held[kind] -= (long)held[i].n;
            free(p);
            held[i].p = NULL;
            return hipSuccess;
        }
    abort(); /* freed twice, or never allocated */
}

hipError_t hipMalloc(void **p, size_t n) { return allocate(DEVICE, p, n); }
hipError_t hipFree(void *p) { return give_back(DEVICE, p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) { (void)flags; return allocate(PINNED, p, n); }
hipError_t hipHostFree(void *p) { return give_back(PINNED, p); }

hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) {
    (void)d;
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 4;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) { (void)a; (void)d; *v = 100000; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l) {
    (void)f; (void)b; (void)l;
    *n = 2;
    return hipSuccess;
}
static char symbol[4 << 20];
hipError_t hipGetSymbolAddress(void **p, const void *s) { (void)s; *p = symbol; return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "an error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; *s = (hipStream_t)symbol; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { (void)s; (void)m; return hipErrorNotSupported; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)symbol; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { (void)f; return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }

hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { (void)k; memmove(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t t) { (void)t; return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t t) { (void)t; memset(d, v, n); return hipSuccess; }

hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) { (void)g; (void)b; (void)l; (void)s; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, hipStream_t *s) {
    g->x = g->y = g->z = b->x = b->y = b->z = 1;
    *l = 0;
    *s = (hipStream_t)symbol;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t l, hipStream_t s) {
    (void)f; (void)g; (void)b; (void)a; (void)l; (void)s;
    ++counts[LAUNCHES];
    return hipSuccess;
}
