/* hipMalloc and hipHostMalloc that answer out-of-memory for sizes in (lo, hi], as a
 * full device, or a host without pinned memory left, would.
 * Loaded with RTLD_GLOBAL before the library, so that the library's calls find it. */
#include <dlfcn.h>
#include <stddef.h>

typedef int (*malloc_fn)(void **, size_t);
typedef int (*host_malloc_fn)(void **, size_t, unsigned);

static size_t dev_lo, dev_hi, host_lo, host_hi;
static int count;

void refuse_device(size_t lo, size_t hi) { dev_lo = lo; dev_hi = hi; }
void refuse_pinned(size_t lo, size_t hi) { host_lo = lo; host_hi = hi; }
int refusals(void) { int c = count; count = 0; return c; }

static void *real(const char *name)
{
    void *h = dlopen("libamdhip64.so.7", RTLD_LAZY);
    return h ? dlsym(h, name) : 0;
}

int hipMalloc(void **p, size_t n)
{
    static malloc_fn f;
    if (n > dev_lo && n <= dev_hi) {
        ++count;
        *p = 0;
        return 2;
    }
    if (!f) f = (malloc_fn)real("hipMalloc");
    return f(p, n);
}

int hipHostMalloc(void **p, size_t n, unsigned flags)
{
    static host_malloc_fn f;
    if (n > host_lo && n <= host_hi) {
        ++count;
        *p = 0;
        return 2;
    }
    if (!f) f = (host_malloc_fn)real("hipHostMalloc");
    return f(p, n, flags);
}
