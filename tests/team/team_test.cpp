// ResultHelpers where threads, or memory for them, cannot be had: argv[1] calls
// of "thread" (pthread_create) or "memory" (operator new) succeed, later ones fail.
#include <errno.h>
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>

#include <new>

#include "../../lighttraffic_amd/csrc/lt_team.h"

static std::atomic<long> left_threads{1L << 40}, left_news{1L << 40};
static std::atomic<bool> armed{false};

void *operator new(size_t n) {
    if (armed && left_news.fetch_sub(1) <= 0) throw std::bad_alloc();
    void *p = malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

extern "C" int __real_pthread_create(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
extern "C" int __wrap_pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) {
    if (armed && left_threads.fetch_sub(1) <= 0) return EAGAIN;
    return __real_pthread_create(t, a, f, x);
}

int main(int argc, char **argv) {
    if (argc != 3) return 2;
    const long ok = atol(argv[2]);
    (argv[1][0] == 't' ? left_threads : left_news) = ok;
    const size_t words = (6u << 20) + 77;
    std::vector<uint32_t> src(words), dst(words, 0);
    for (size_t i = 0; i < words; i++) src[i] = (uint32_t)(i * 2654435761u);
    std::vector<lt::OutSeg> outs{{dst.data(), nullptr, words}};
    std::vector<uint8_t> fresh(1 << 20, 1);
    armed = true;
    {
        lt::ResultHelpers help;
        help.most = 4;
        help.fresh = fresh.data();
        help.fresh_bytes = fresh.size();
        help.start(outs);
        for (size_t at = 0, n; at < words; at += n) {  // pieces of every size
            n = words - at < 500009 ? words - at : 500009 - at % 4097;
            help.copiers().copy(dst.data() + at, src.data() + at, 4 * n);
        }
    }
    armed = false;
    if (dst != src) {
        puts("copies differ");
        return 1;
    }
    puts("done");
    return 0;
}
