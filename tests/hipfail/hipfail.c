/* Calls of the HIP runtime that fail when a test asks for it.  Loaded with
 * RTLD_GLOBAL before the engine's library, whose calls then come here; each goes
 * on to the runtime unless it is the one that is to fail, which does nothing. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
#include <stdio.h>
#include <stdlib.h>

enum { MALLOC, HOST_MALLOC, MEMCPY_ASYNC, KINDS };
static struct {
    long calls, failed;    /* since armed */
    long skip, times;      /* let `skip` matching calls through, then fail `times` */
    size_t least, most;    /* bytes that match */
} rule[KINDS];

static void *runtime(const char *name) {
    static void *lib;
    if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_NOW);
    void *f = lib ? dlsym(lib, name) : NULL;
    if (!f) {
        fprintf(stderr, "hipfail: %s\n", dlerror());
        abort();
    }
    return f;
}

void hipfail_arm(int kind, long skip, long times, size_t least, size_t most) {
    rule[kind].calls = rule[kind].failed = 0;
    rule[kind].skip = skip;
    rule[kind].times = times;
    rule[kind].least = least;
    rule[kind].most = most;
}
long hipfail_calls(int kind) { return rule[kind].calls; }
long hipfail_failed(int kind) { return rule[kind].failed; }

static int fails(int kind, size_t bytes) {
    if (bytes < rule[kind].least || bytes > rule[kind].most) return 0;
    const long i = rule[kind].calls++ - rule[kind].skip;
    if (i < 0 || i >= rule[kind].times) return 0;
    rule[kind].failed++;
    return 1;
}

/* Device memory: bytes that the engine's library holds, and may hold. */
static size_t held, limit = (size_t)-1;
static struct {
    void *p;
    size_t n;
} block[4096];
void hipfail_limit(size_t bytes) { limit = bytes; }
size_t hipfail_held(void) { return held; }

/* hipErrorOutOfMemory is 2, hipErrorUnknown 999 */
int hipMalloc(void **p, size_t n) {
    if (fails(MALLOC, n) || n > limit || held > limit - n) return 2;
    const int e = ((int (*)(void **, size_t))runtime("hipMalloc"))(p, n);
    int i = 0;
    while (!e && block[i].p) i++;
    if (!e) {
        block[i].p = *p;
        block[i].n = n;
        held += n;
    }
    return e;
}
int hipFree(void *p) {
    for (int i = 0; p && i < 4096; i++)
        if (block[i].p == p) {
            block[i].p = NULL;
            held -= block[i].n;
            break;
        }
    return ((int (*)(void *))runtime("hipFree"))(p);
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    if (fails(HOST_MALLOC, n)) return 2;
    return ((int (*)(void **, size_t, unsigned))runtime("hipHostMalloc"))(p, n, flags);
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream) {
    if (fails(MEMCPY_ASYNC, n)) return 999;
    return ((int (*)(void *, const void *, size_t, int, void *))runtime("hipMemcpyAsync"))(d, s, n, kind, stream);
}
