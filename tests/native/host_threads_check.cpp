// The host work that is shared among threads (the potential's tables, the
// model's bridge polynomials, the electron mesh's tile schedules) in a process
// that has no thread to give, or no memory inside one.
//   host_threads_check threads|none|memory
// "threads" and "none" print a hash of everything made; "memory" lets every
// allocation outside the main thread fail and expects the failure in the caller.
#include "sld_dte_plan.h"
#include "sld_model.h"
#include "sld_tables.h"

#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

using namespace sld;

static bool no_threads = false, no_memory = false;
static thread_local bool in_main = false;

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
    using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
    return no_threads ? EAGAIN : real(t, a, f, arg);
}

void* operator new(std::size_t n) {
    void* p = no_memory && !in_main ? nullptr : std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

static unsigned long long hash = 1469598103934665603ull;
template <class T>
static void add(const std::vector<T>& v) {
    const unsigned char* b = reinterpret_cast<const unsigned char*>(v.data());
    for (std::size_t k = 0; k < v.size() * sizeof(T); ++k) hash = (hash ^ b[k]) * 1099511628211ull;
}

static bool schedule(DteSchedule& s) {
    const int n = 24;  // 216 tiles
    std::vector<int> group(n * n * n);
    for (int c = 0; c < n * n * n; ++c) group[c] = (c % n % 2) + 2 * (c / n % n % 2) + 4 * (c / (n * n) % 2);
    return dte_schedule(n, n, n, group, kDteBoth, 4, 4, 4, kDteMaxLev, s);
}

int main(int argc, char** argv) {
    in_main = true;
    const char* mode = argc > 1 ? argv[1] : "";
    DteSchedule s;
    if (!std::strcmp(mode, "memory")) {
        no_memory = true;
        try {
            schedule(s);
        } catch (const std::bad_alloc&) {
            std::printf("bad_alloc in the caller\n");
            return 0;
        }
        std::printf("no failure\n");
        return 0;
    }
    no_threads = !std::strcmp(mode, "none");
    if (!schedule(s)) return 1;
    add(s.tile);
    add(s.upd);
    add(s.slot);
    add(s.lev);
    std::printf("schedule %016llx\n", hash);
    add(model_bridge(4.1)->q);
    std::printf("bridge %016llx\n", hash);
    const auto t = shared_tables(4.1, false);
    add(t->prow);
    add(t->jtab);
    add(t->sftab);
    add(t->rhotab);
    std::printf("tables %016llx\n", hash);
    return 0;
}
