/* Stand-in for the HIP runtime, so that the host side of libcmf_hip.so runs on a CPU:
 * device and pinned memory come from malloc, copies are done at once, kernels are
 * counted and not run. Loaded before the library (RTLD_GLOBAL), its symbols come
 * first. stub_fail makes single allocations fail. */
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

static long n_dev, n_pin, n_launch, n_live, fail_dev_from, fail_dev_to, fail_pin_from, fail_pin_to;

/* fail device allocations number from..to and pinned ones (counted from 1 after this
 * call; 0, 0: none) */
void stub_fail(long dev_from, long dev_to, long pin_from, long pin_to) {
    n_dev = n_pin = n_launch = 0;
    fail_dev_from = dev_from; fail_dev_to = dev_to;
    fail_pin_from = pin_from; fail_pin_to = pin_to;
}
long stub_device_allocs(void) { return n_dev; }
long stub_pinned_allocs(void) { return n_pin; }
long stub_launches(void) { return n_launch; }
long stub_live(void) { return n_live; }       /* allocations not yet freed */
/* milliseconds that a cooperative launch and a graph take */
static unsigned slow_ms;
void stub_slow(unsigned ms) { slow_ms = ms; }

enum { OK = 0, ENOMEM_HIP = 2 };
static int take(void **p, size_t n, int fails) {
    *p = NULL;
    if (fails) return ENOMEM_HIP;
    *p = calloc(1, n ? n : 1);
    if (*p) ++n_live;
    return *p ? OK : ENOMEM_HIP;
}
int hipMalloc(void **p, size_t n) { ++n_dev; return take(p, n, n_dev >= fail_dev_from && n_dev <= fail_dev_to); }
int hipHostMalloc(void **p, size_t n, unsigned f) {
    (void)f;
    ++n_pin;
    return take(p, n, n_pin >= fail_pin_from && n_pin <= fail_pin_to);
}
int hipFree(void *p) { if (p) { --n_live; free(p); } return OK; }
int hipHostFree(void *p) { return hipFree(p); }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memmove(d, s, n); return OK; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)st; return hipMemcpy(d, s, n, k); }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)st; memset(d, v, n); return OK; }
int hipLaunchKernel(const void *f, ...) { (void)f; ++n_launch; return OK; }
int hipLaunchCooperativeKernel(const void *f, ...) { (void)f; ++n_launch; usleep(1000u * slow_ms); return OK; }
int hipGetLastError(void) { return OK; }
const char *hipGetErrorString(int e) { return e == OK ? "success" : "out of memory (stand-in)"; }
int hipGetDevice(int *d) { *d = 0; return OK; }
int hipSetDevice(int d) { (void)d; return OK; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return OK; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t m) {
    (void)f; (void)b; (void)m;
    *n = 1;
    return OK;
}
int hipGetSymbolAddress(void **p, const void *s) {
    static double there[64];
    (void)s;
    *p = there;
    return OK;
}
static int handle_of(void **h) { static int any; *h = &any; return OK; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; return handle_of(s); }
int hipStreamDestroy(void *s) { (void)s; return OK; }
int hipStreamSynchronize(void *s) { (void)s; return OK; }
int hipEventCreate(void **e) { return handle_of(e); }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; return handle_of(e); }
int hipEventDestroy(void *e) { (void)e; return OK; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return OK; }
int hipEventSynchronize(void *e) { (void)e; return OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return OK; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return OK; }
int hipStreamEndCapture(void *s, void **g) { (void)s; return handle_of(g); }
int hipGraphInstantiate(void **x, void *g, void *n, char *log, size_t z) { (void)g; (void)n; (void)log; (void)z; return handle_of(x); }
int hipGraphLaunch(void *x, void *s) { (void)x; (void)s; ++n_launch; usleep(1000u * slow_ms); return OK; }
int hipGraphDestroy(void *g) { (void)g; return OK; }
int hipGraphExecDestroy(void *x) { (void)x; return OK; }
