/* A HIP runtime without a GPU, for tests of the library's host code: device memory is
 * host memory, copies run at once, kernel launches are only counted by name, and
 * allocations of chosen sizes are refused. As in the real runtime, a failed call stays
 * the last error, through later calls that succeed, until hipGetLastError reads it.
 * Loaded with RTLD_GLOBAL before libvoxhip.so, its symbols take the place of
 * libamdhip64's. Only what the tests reach is here. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

static hipError_t last = hipSuccess;
static size_t refuse_lo, refuse_hi, largest;
static struct { const void *fn; const char *name; int launches; } fns[4096];
static int n_fns;

void fake_refuse(size_t lo, size_t hi) { refuse_lo = lo; refuse_hi = hi; }
size_t fake_largest(void) { size_t n = largest; largest = 0; return n; }
/* Launches so far of the kernels whose (mangled) name contains `part`. */
int fake_launches(const char *part) {
    int n = 0;
    for (int i = 0; i < n_fns; ++i)
        if (strstr(fns[i].name, part)) n += fns[i].launches;
    return n;
}

void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t s, int c, int g) {
    (void)m, (void)v, (void)h, (void)d, (void)e, (void)s, (void)c, (void)g;
}
void __hipRegisterFunction(void **m, const void *fn, char *dev, const char *name, unsigned l, void *t, void *b,
                           void *bd, void *gd, int *w) {
    (void)m, (void)dev, (void)l, (void)t, (void)b, (void)bd, (void)gd, (void)w;
    if (n_fns < 4096) fns[n_fns].fn = fn, fns[n_fns++].name = name;
}
static struct { dim3 g, b; size_t s; hipStream_t st; } cfg;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
    cfg.g = g, cfg.b = b, cfg.s = s, cfg.st = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) {
    *g = cfg.g, *b = cfg.b, *s = cfg.s, *st = cfg.st;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **a, size_t s, hipStream_t st) {
    (void)g, (void)b, (void)a, (void)s, (void)st;
    for (int i = 0; i < n_fns; ++i)
        if (fns[i].fn == fn) ++fns[i].launches;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipMalloc(void **p, size_t n) {
    *p = NULL;
    if (n > largest) largest = n;
    if (n >= refuse_lo && n <= refuse_hi) return last = hipErrorOutOfMemory;
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    return hipSuccess;
}
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
    (void)k, (void)st;
    memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind k,
                            hipStream_t st) {
    (void)k, (void)st;
    for (size_t i = 0; i < h; ++i) memmove((char *)d + i * dp, (const char *)s + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) { (void)st; memset(d, v, n); return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) {
    (void)a, (void)d;
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) {   /* the header maps the name to its version */
    (void)d;
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s) { static char mem[1 << 20]; (void)s; *p = mem; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; *s = (hipStream_t)&cfg; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
