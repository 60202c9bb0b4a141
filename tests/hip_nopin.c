/* hipHostMalloc that can be told to find no memory; everything else is the HIP
 * runtime's. Loaded before the library (RTLD_GLOBAL), so its symbol comes first. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

static int none, refused;
int stub_refused(void) { return refused; }
void stub_fail(long unused0, long unused1, long from, long to) {
    (void)unused0; (void)unused1; (void)to;
    none = from > 0;
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    static int (*real)(void **, size_t, unsigned);
    if (none) { *p = NULL; ++refused; return 2; }
    if (!real) {
        void *hip = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD);
        if (hip) real = (int (*)(void **, size_t, unsigned))dlsym(hip, "hipHostMalloc");
        if (!real) return 2;
    }
    return real(p, n, flags);
}
