/* The HIP allocation calls with a limit on what they hand out, for a test process: loaded with
 * RTLD_GLOBAL before libselas_gpu, so that the library's calls come here first. Nothing is really
 * exhausted: a request past alloc_limit_set's bytes gets hipErrorOutOfMemory, every other goes on to the
 * runtime. A refusal stays the thread's last error until it is asked for, as the runtime's do. Memory
 * freed to the stream-ordered pool counts until the pool is trimmed. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stddef.h>

enum { kOutOfMemory = 2, kMax = 1 << 16 };

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static struct {
    void* p;
    size_t n;
} block[kMax];
static size_t count, plain, pooled, pool_size, limit = (size_t)-1, refused;
static __thread int last;

static void* real(const char* name)
{
    void* lib = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    return lib ? dlsym(lib, name) : NULL;
}

static void note(void* p, size_t n)
{
    if (count < kMax) {
        block[count].p = p;
        block[count++].n = n;
    }
}

static size_t forget(void* p)
{
    for (size_t k = 0; k < count; ++k)
        if (block[k].p == p) {
            const size_t n = block[k].n;
            block[k] = block[--count];
            return n;
        }
    return 0;
}

size_t alloc_limit_used(void) { return plain + pool_size; }
size_t alloc_limit_refused(void) { return refused; }
void alloc_limit_set(size_t bytes) { limit = bytes; }

int hipMalloc(void** p, size_t n)
{
    int (*f)(void**, size_t) = (int (*)(void**, size_t))real("hipMalloc");
    pthread_mutex_lock(&mu);
    int e = kOutOfMemory;
    if (plain + pool_size + n > limit)
        ++refused, last = e;
    else if ((e = f(p, n)) == 0) {
        note(*p, n);
        plain += n;
    }
    pthread_mutex_unlock(&mu);
    return e;
}

int hipFree(void* p)
{
    int (*f)(void*) = (int (*)(void*))real("hipFree");
    pthread_mutex_lock(&mu);
    plain -= forget(p);
    pthread_mutex_unlock(&mu);
    return f(p);
}

int hipMallocAsync(void** p, size_t n, void* stream)
{
    int (*f)(void**, size_t, void*) = (int (*)(void**, size_t, void*))real("hipMallocAsync");
    pthread_mutex_lock(&mu);
    const size_t size = pooled + n > pool_size ? pooled + n : pool_size;
    int e = kOutOfMemory;
    if (plain + size > limit)
        ++refused, last = e;
    else if ((e = f(p, n, stream)) == 0) {
        note(*p, n);
        pooled += n;
        pool_size = size;
    }
    pthread_mutex_unlock(&mu);
    return e;
}

int hipFreeAsync(void* p, void* stream)
{
    int (*f)(void*, void*) = (int (*)(void*, void*))real("hipFreeAsync");
    pthread_mutex_lock(&mu);
    pooled -= forget(p);
    pthread_mutex_unlock(&mu);
    return f(p, stream);
}

int hipMemPoolTrimTo(void* pool, size_t keep)
{
    int (*f)(void*, size_t) = (int (*)(void*, size_t))real("hipMemPoolTrimTo");
    pthread_mutex_lock(&mu);
    pool_size = pooled > keep ? pooled : keep;
    pthread_mutex_unlock(&mu);
    return f(pool, keep);
}

int hipGetLastError(void)
{
    int (*f)(void) = (int (*)(void))real("hipGetLastError");
    const int e = f(), mine = last;
    last = 0;
    return mine ? mine : e;
}
