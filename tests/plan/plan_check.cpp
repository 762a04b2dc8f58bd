// Checks of the sweeps' layouts and plans (cd_plan.h) over many sizes, on the host.
// One check per argument; prints what fails and exits with 1.
#include <cstdio>
#include <cstring>

#include "cd_plan.h"

namespace {

int g_bad = 0;
#define CHECK(cond, ...)                                   \
    do {                                                   \
        if (!(cond) && ++g_bad <= 20) {                    \
            std::printf(__VA_ARGS__);                      \
            std::printf(": %s\n", #cond);                  \
        }                                                  \
    } while (0)

// Every row that a region loads or stores: the address parts lie in the plane by
// themselves (the instruction adds them without wrapping), and a row of the grid
// has its own address.
void rows_in_plane() {
    for (int w : {2, 180, 1000})
        for (int h = 2; h <= 300; ++h) {
            const Brick bk = make_brick(w, h);
            for (int rows = 4; rows <= 8; rows += 2)
                for (int Y = 0; Y < std::max(h, BK_NW * rows); Y += 2) {
                    const BrickRows br = brick_rows(bk, Y, h);
                    for (int k = 0; k < rows; ++k) {
                        const unsigned at = br.at(k), row = at - 64u * k;
                        // (with the row's last columns)
                        CHECK(row < bk.plane && at + (bk.nbx - 1) * (size_t)512 + 64 <= bk.plane,
                              "%d x %d, %d rows from %d, row %d", w, h, rows, Y, k);
                        if (Y + k < h) {
                            const size_t want =
                                (size_t)((Y + k) >> 3) * bk.nbx * 512 + (size_t)((Y + k) & 7) * 64;
                            CHECK(at == want, "%d x %d, row %d", w, h, Y + k);
                        }
                    }
                }
        }
}

}  // namespace

int main(int argc, char** argv) {
    const struct { const char* name; void (*fn)(); } checks[] = {
        {"rows_in_plane", rows_in_plane},
    };
    for (const auto& c : checks)
        if (argc == 2 && !std::strcmp(argv[1], c.name)) {
            c.fn();
            std::printf("%s: %d bad\n", c.name, g_bad);
            return g_bad ? 1 : 0;
        }
    std::printf("no such check\n");
    return 2;
}
