/* hipMalloc, hipFree and hipHostMalloc with limits, for the tests of what happens
 * at the end of memory.  Loaded with global symbols before libimpec_hip.so, whose
 * calls then come here; the calls within the limits go on to the HIP runtime. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stddef.h>

enum { N_MAX = 4096, OUT_OF_MEMORY = 2 /* hipErrorOutOfMemory */ };

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static struct { void *p; size_t n; } blocks[N_MAX];
static size_t live, limit = (size_t)-1, host_limit = (size_t)-1;
static int host_calls;

void alloc_limit(size_t device_bytes, size_t host_block_bytes) {
    pthread_mutex_lock(&lock);
    limit = device_bytes;
    host_limit = host_block_bytes;
    pthread_mutex_unlock(&lock);
}
size_t alloc_live(void) { return live; }
/* successful host allocations of at least 1 MiB */
int alloc_host_calls(void) { return host_calls; }

static void *next(const char *name) {
    static void *hip;
    if (!hip) hip = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
    return hip ? dlsym(hip, name) : NULL;
}

int hipMalloc(void **p, size_t n) {
    int (*f)(void **, size_t) = (int (*)(void **, size_t))next("hipMalloc");
    int e;
    pthread_mutex_lock(&lock);
    if (!f || live + n > limit) {
        pthread_mutex_unlock(&lock);
        *p = NULL;
        return OUT_OF_MEMORY;
    }
    e = f(p, n);
    if (e == 0) {
        int k;
        for (k = 0; k < N_MAX; k++)
            if (!blocks[k].p) {
                blocks[k].p = *p;
                blocks[k].n = n;
                break;
            }
        live += n;
    }
    pthread_mutex_unlock(&lock);
    return e;
}

int hipFree(void *p) {
    int (*f)(void *) = (int (*)(void *))next("hipFree");
    int k;
    pthread_mutex_lock(&lock);
    for (k = 0; p && k < N_MAX; k++)
        if (blocks[k].p == p) {
            live -= blocks[k].n;
            blocks[k].p = NULL;
            break;
        }
    pthread_mutex_unlock(&lock);
    return f ? f(p) : OUT_OF_MEMORY;
}

int hipHostMalloc(void **p, size_t n, unsigned flags) {
    int (*f)(void **, size_t, unsigned) = (int (*)(void **, size_t, unsigned))next("hipHostMalloc");
    int e;
    if (!f || n >= host_limit) {
        *p = NULL;
        return OUT_OF_MEMORY;
    }
    e = f(p, n, flags);
    if (e == 0 && n >= (size_t)1 << 20) {
        pthread_mutex_lock(&lock);
        host_calls++;
        pthread_mutex_unlock(&lock);
    }
    return e;
}
