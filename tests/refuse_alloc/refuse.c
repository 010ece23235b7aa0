/* hipMalloc that answers out-of-memory for sizes in (lo, hi], as a full device would.
 * Loaded with RTLD_GLOBAL before the library, so that the library's calls find it. */
#include <dlfcn.h>
#include <stddef.h>

typedef int (*malloc_fn)(void **, size_t);

static size_t dev_lo, dev_hi;
static int count;

void refuse_device(size_t lo, size_t hi) { dev_lo = lo; dev_hi = hi; }
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
