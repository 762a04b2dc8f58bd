// The first-hit order when memory or threads run out: operator new fails from the
// n-th allocation on, or only there, for every n a build reaches.  Each call returns
// CD_OK with the same order, or CD_ERR_OOM; none may end the process.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "cd_api.h"

namespace {
std::atomic<long> g_count{0};
long g_fail_at = -1;    // the allocation that fails (-1: none)
bool g_and_after = false;
}  // namespace

void* operator new(std::size_t n) {
    const long i = g_count++;
    if (g_fail_at >= 0 && (i == g_fail_at || (g_and_after && i > g_fail_at))) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

extern "C" int cd_bvh_first_hit_order(const double* xy, int mx, int my, int* order);

int main() {
    const int m = 200;  // 79202 triangles: threads on three levels
    std::vector<double> xy(2 * m * m);
    for (int i = 0; i < m * m; ++i) {
        xy[2 * i] = i % m + 0.3 * std::rand() / RAND_MAX;
        xy[2 * i + 1] = i / m + 0.3 * std::rand() / RAND_MAX;
    }
    std::vector<int> want(2 * (m - 1) * (m - 1)), got(want.size());
    g_count = 0;
    if (cd_bvh_first_hit_order(xy.data(), m, m, want.data()) != CD_OK) return 1;
    const long n = g_count;
    std::printf("%ld allocations\n", n);
    int oom = 0;
    for (int after = 0; after < 2; ++after)
        for (long k = 0; k < n; ++k) {
            std::fill(got.begin(), got.end(), -1);
            g_and_after = after != 0;
            g_count = 0;
            g_fail_at = k;
            const int rc = cd_bvh_first_hit_order(xy.data(), m, m, got.data());
            g_fail_at = -1;
            std::printf("fail at %ld%s: %d\n", k, after ? " and after" : "", rc);
            std::fflush(stdout);
            if (rc == CD_ERR_OOM) ++oom;
            else if (rc != CD_OK || got != want) return 1;
        }
    return n >= 2 && oom >= 1 ? 0 : 1;
}
