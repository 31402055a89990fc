/* alloc_limit.c -- test infrastructure: device allocations of at least
 * alloc_limit_bytes are refused as the runtime refuses them when memory is
 * short, and streams that are made are counted.  Loaded with RTLD_GLOBAL ahead of the engine, whose calls then bind
 * here (tests/test_gpu_no_memory.py, tests/test_gpu_serve_streams.py). */
#include <dlfcn.h>
#include <stddef.h>

size_t alloc_limit_bytes = (size_t)-1;
int    alloc_refused = 0;
int    streams_made = 0;

static void *real(const char *name) { return dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), name); }

static int refuse(size_t n)
{
    if (n < alloc_limit_bytes) return 0;
    alloc_refused++;
    return 2; /* hipErrorOutOfMemory */
}

int hipMallocAsync(void **p, size_t n, void *stream)
{
    const int e = refuse(n);
    return e ? e : ((int (*)(void **, size_t, void *))real("hipMallocAsync"))(p, n, stream);
}

int hipMalloc(void **p, size_t n)
{
    const int e = refuse(n);
    return e ? e : ((int (*)(void **, size_t))real("hipMalloc"))(p, n);
}

int hipStreamCreateWithFlags(void **st, unsigned flags)
{
    streams_made++;
    return ((int (*)(void **, unsigned))real("hipStreamCreateWithFlags"))(st, flags);
}
