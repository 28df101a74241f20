// Prints the level of every (angle, cell) of a level-set schedule and its
// lagged faces.  argv: mesh arrays (written by the test).
#include <cstdio>
#include <cstdlib>

#include "t2_common.hpp"

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
    t2::Schedule s;
    if (t2::build_schedule(m, na, omega.data(), 1, T2_ORDER_FACES, s))
        return 1;
    const uint32_t mask = (uint32_t(1) << s.cell_bits) - 1;
    for (int64_t st = 0; st < s.n_steps; st++)
        for (int64_t i = s.step_off[st]; i < s.step_off[st + 1]; i++)
            std::printf("level %d %d %lld\n", int(s.work[i] >> s.cell_bits),
                        int(s.work[i] & mask), (long long)st);
    for (const auto &l : s.lagged)
        std::printf("lagged %d %d %d\n", l.angle, l.cell, l.face);
    return 0;
}
