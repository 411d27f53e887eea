// The host loops of grotor_amd/csrc/gr_parallel.hpp where threads cannot be
// started: pthread_create below lets the first `argv[1]` calls through and
// fails the others as a process limit does.
#include "gr_parallel.hpp"

#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <stdexcept>

static std::atomic<int> allowed{0};

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* p) {
    if (allowed.fetch_sub(1) <= 0) return EAGAIN;
    using Create = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    static const Create create = reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"));
    return create(t, a, f, p);
}

int main(int, char** argv) {
    const int limit = std::atoi(argv[1]);
    for (int n : {1, 7, 4095, 4096, 70001}) {
        std::vector<std::atomic<int>> items(n), tasks(n);
        allowed = limit;
        grotor::parallel_items(n, [&](int k) { ++items[k]; });
        allowed = limit;
        grotor::parallel_tasks(n, [&](int k) { ++tasks[k]; });
        for (int k = 0; k < n; ++k)
            if (items[k] != 1 || tasks[k] != 1) return std::printf("item %d of %d: %d %d\n", k, n, int(items[k]), int(tasks[k])), 1;
        allowed = limit;
        try {
            grotor::parallel_items(n, [&](int k) {
                if (k == n / 2) throw std::runtime_error("item");
            });
            return std::printf("no exception from %d items\n", n), 1;
        } catch (const std::runtime_error&) {
        }
    }
    std::puts("ok");
    return 0;
}
