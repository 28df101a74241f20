// Every host allocation of a sweep schedule failed in turn, in whichever
// thread it falls: the builders return T2_ERR_NOMEM or, where nothing failed,
// T2_OK, and the process goes on.  argv: mesh arrays (written by the test).
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>

#include "t2_common.hpp"

static std::atomic<long> g_left{-1};

void *operator new(std::size_t n)
{
    if (g_left.load() > 0 && --g_left == 0)
        throw std::bad_alloc();
    if (void *p = std::malloc(n))
        return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

template <typename T>
static std::vector<T> take(FILE *f, size_t n)
{
    std::vector<T> v(n);
    if (std::fread(v.data(), sizeof(T), n, f) != n)
        std::exit(2);
    return v;
}

int main(int, char **argv)
{
    FILE *f = std::fopen(argv[1], "rb");
    const auto size = take<int64_t>(f, 2);
    t2::HostMesh m;
    m.nc = size[0];
    const int64_t na = size[1];
    m.adj = take<int64_t>(f, 4 * m.nc);
    m.area = take<double>(f, 4 * m.nc);
    m.normal = take<double>(f, 12 * m.nc);
    const auto omega = take<double>(f, 3 * na);
    std::fclose(f);
    long failures = 0;
    auto each = [&](const char *name, auto build) {
        for (long nth = 1;; nth++) {
            g_left = nth;
            const int rc = build();
            const bool all_ran = g_left.load() > 0;
            g_left = -1;
            if (rc != T2_OK && rc != T2_ERR_NOMEM) {
                std::printf("%s %ld: %d\n", name, nth, rc);
                std::exit(1);
            }
            failures += rc != T2_OK;
            if (all_ran) {
                if (rc != T2_OK)
                    std::exit(1);
                return;
            }
        }
    };
    t2::Schedule s;
    each("schedule", [&]() {
        s = t2::Schedule();
        return t2::build_schedule(m, na, omega.data(), 1, T2_ORDER_FACES, s);
    });
    if (s.lagged.empty())   // the mesh is to reach the re-levelling
        return 3;
    each("slots", [&]() {
        std::vector<uint16_t> slot;
        int64_t n = 0;
        return t2::build_slots(m, na, omega.data(), s, slot, &n);
    });
    each("priorities", [&]() {
        t2::Schedule p;
        return t2::build_priority_schedule(m, na, omega.data(), 2, 2, 100,
                                           T2_ORDER_FACES, p);
    });
    std::printf("failures %ld\n", failures);
    return 0;
}
