// Checks of the sweeps' layouts and plans (cd_plan.h) over many sizes, on the host.
// One check per argument; prints what fails and exits with 1.
#include <cstdio>
#include <cstring>
#include <utility>
#include <vector>

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

// Every tracking plan's words and maxima fit behind the partials' other use, on
// any shape, and its halo is whole waves (the cells that count are whole waves').
void tracking_room() {
    for (int h : {2, 3, 4, 5, 8, 60, 64, 65, 97, 300, 4000})
        for (double wd = 2; wd * h < 5e8; wd *= 1.07) {
            const int w = (int)wd;
            const size_t room = cd_partials_bytes((size_t)div_up(w, RED_BX) * div_up(h, RED_BY));
            for (int batch : {1, 4, 5, 7, 15, 92, 1000}) {
                const BlockedPlan p = blocked_plan(w, h, batch, true, room);
                CHECK(p.t.ntiles >= 1 && track_bytes(p.t.ntiles, p.sweeps) <= room,
                      "%d x %d, batch %d, blocked", w, h, batch);
                CHECK(p.t.ntiles == 1 || (p.t.halo % p.rows == 0 && p.t.halo >= 2 * p.sweeps),
                      "%d x %d, batch %d: halo %d, %d rows, %d sweeps", w, h, batch, p.t.halo,
                      p.rows, p.sweeps);
                for (bool fp64 : {false, true}) {
                    const SweepTiles t = natural_tiles(w, h, fp64, batch, true, room);
                    CHECK(track_bytes(t.ntiles, natural_sweeps(t, batch, true)) <= room,
                          "%d x %d, batch %d, natural", w, h, batch);
                }
            }
        }
}

// No plan puts more sweeps into a launch than a solve in one workgroup takes.
void launch_length() {
    for (int w : {2, 40, 128, 129, 500})
        for (int h : {2, 40, 64, 128, 129, 500})
            for (int batch : {1, 100, 16384, 16385, 100000, INT_MAX})
                for (bool track : {false, true}) {
                    const BlockedPlan p = blocked_plan(w, h, batch, track, 1u << 20);
                    CHECK(p.sweeps <= kRegionSweeps, "%d x %d, batch %d: %d", w, h, batch, p.sweeps);
                    const int n =
                        natural_sweeps(natural_tiles(w, h, true, batch, track, 1u << 20), batch, track);
                    CHECK(n <= kRegionSweeps, "%d x %d, batch %d: %d", w, h, batch, n);
                }
}

// No tracking launch writes what it reads, and each reads what the one before wrote.
void track_words() {
    for (int ntiles : {1, 7, 600})
        for (int slots : {2, 5, 15})
            for (int launches = 1; launches < 6; ++launches) {
                std::vector<unsigned> buf(track_bytes(ntiles, slots) / 4);
                TrackBatch b = track_batch(buf.data(), ntiles, slots, 5, 1.0);
                auto range = [&](const TrackOut& t) {  // [first, last) word of a TrackOut
                    const long lo = t.bits - buf.data();
                    const long hi = reinterpret_cast<unsigned*>(t.maxima) - buf.data() +
                                    (long)ntiles * slots;
                    return std::pair<long, long>(lo, hi);
                };
                unsigned* last = nullptr;
                for (int i = 0; i <= launches; ++i) {
                    const TrackArgs a = i < launches ? b.launch(i + 1, slots, slots * i)
                                                     : b.check(i + 1);
                    CHECK(a.prev.bits == last, "launch %d of %d", i, launches);
                    CHECK(a.check_only == (i == launches), "launch %d of %d", i, launches);
                    CHECK(i == 0 || (a.nprev == slots && a.first_prev == slots * (i - 1)),
                          "launch %d of %d", i, launches);
                    const auto out = range(a.out);
                    CHECK(out.first >= 0 && out.second <= (long)buf.size(), "launch %d", i);
                    if (last) {
                        const auto prev = range(a.prev);
                        CHECK(out.second <= prev.first || prev.second <= out.first,
                              "launch %d of %d writes what it reads", i, launches);
                    }
                    last = a.out.bits;
                }
            }
}

// The launch that goes out ahead of a batch is one launch, so that the batch goes on
// from its output.
void early_launch() {
    for (int w = 2; w <= 6000; w += w < 700 ? 1 : 37)
        for (int h = 2; h <= 6000; h += h < 300 ? 3 : 53) {
            const int ahead = std::min(8, blocked_plan(w, h, 8, false, 0).sweeps);
            const int per = blocked_plan(w, h, ahead, false, 0).sweeps;
            CHECK(per >= ahead, "%d x %d: %d sweeps in launches of %d", w, h, ahead, per);
        }
}

}  // namespace

int main(int argc, char** argv) {
    const struct { const char* name; void (*fn)(); } checks[] = {
        {"rows_in_plane", rows_in_plane},
        {"tracking_room", tracking_room},
        {"launch_length", launch_length},
        {"track_words", track_words},
        {"early_launch", early_launch},
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
