// Layouts, tiles and plans of the solver's sweeps: what its host code computes
// before a launch, and the address arithmetic that kernels share with it.  No HIP
// in here, so that a host program can check it over all sizes.
#pragma once

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstddef>

#ifdef __HIPCC__
#define CD_HD __host__ __device__ __forceinline__
#else
#define CD_HD inline
#endif

namespace {

inline int div_up(long long a, long long b) { return (int)((a + b - 1) / b); }

// cells of a workgroup of the reduction passes
constexpr int RED_BX = 64;
constexpr int RED_BY = 4;

// Bytes of the reduction partials: four doubles for each of nred workgroups,
// and room for the per-tile maxima of the max-update rule on small grids.
constexpr size_t cd_partials_bytes(size_t nred) { return sizeof(double) * 4 * nred + 32768; }

// Bricked checkerboard layout of the blocked sweeps.  Colour c = (x+y)&1 and
// packed column j = x>>1 split the grid into two planes of h x wp cells
// (wp = (w+1)/2); each plane is stored in bricks of 8 rows x 64 packed columns
// (2 KiB of FP32), bricks row-major.  A wave of the blocked kernel reads
// 8 consecutive rows of one brick as one contiguous 2 KiB stream.
struct Brick {
    int wpb;       // packed columns rounded up to 64
    int nbx;       // bricks per row of bricks
    size_t plane;  // elements per colour plane (rows rounded up to 8)
};

inline Brick make_brick(int w, int h) {
    Brick b;
    const int wp = (w + 1) / 2;
    b.wpb = (wp + 63) / 64 * 64;
    b.nbx = b.wpb / 64;
    b.plane = (size_t)((h + 7) / 8 * 8) * b.wpb;
    return b;
}

// Plane offsets (elements) of R <= 8 consecutive rows from Y on: they lie in at
// most two bricks, so that one select per row and a constant give each.  Rows
// beyond the plane's last brick get the offset of some row in it.  a and b are
// offsets in the plane by themselves: a kernel passes them as scalar offsets, to
// which the hardware adds the rest without wrapping.
struct BrickRows {
    unsigned a, b;  // offset of row k less 64 k, before and from the brick border on
    int split;
    CD_HD unsigned at(int k) const { return (k < split ? a : b) + 64u * k; }
};
CD_HD BrickRows brick_rows(const Brick& bk, int Y, int h) {
    const int nby = (h + 7) >> 3, by = (Y >> 3) < nby ? Y >> 3 : nby - 1;
    const unsigned brow = (unsigned)bk.nbx * 512u;
    BrickRows r;
    r.a = (unsigned)by * brow + (unsigned)(Y & 7) * 64u;
    const int b = (int)(r.a + (by + 1 < nby ? brow : 0u)) - 512;
    r.b = (unsigned)(b > 0 ? b : 0);  // (below 0 on a single row of bricks)
    r.split = 8 - (Y & 7);
    return r;
}

constexpr int SW_RX = 128;  // region columns (64 lanes, two cells each)

// Tiling of a w x h grid by regions of SW_RX x ry cells with `halo` overlap.
// Region (tx, ty) starts at (min(tx*ix, we - SW_RX), min(ty*iy, he - ry)), never
// below 0; we, he are w, h rounded up to even, so that a cell's colour is its
// lane slot's on every region.  It stores columns [tx*ix + halo, (tx+1)*ix +
// halo) (from 0 for the first region, to w for the last), and rows alike.
struct SweepTiles {
    int w, h, we, he;
    int ry, halo, ix, iy;
    int tiles_x, tiles_y, ntiles;
    unsigned inv_x;  // floor((2^32 - 1) / tiles_x): tile * inv_x >> 32 is tile / tiles_x or one less
};

inline SweepTiles sweep_tiles(int w, int h, int ry, int halo) {
    SweepTiles t;
    t.w = w;
    t.h = h;
    t.we = (w + 1) / 2 * 2;
    t.he = (h + 1) / 2 * 2;
    t.ry = ry;
    t.halo = halo;
    t.ix = SW_RX - 2 * halo;
    t.iy = ry - 2 * halo;
    t.tiles_x = t.we <= SW_RX ? 1 : 1 + (t.we - SW_RX + t.ix - 1) / t.ix;
    t.tiles_y = t.he <= ry ? 1 : 1 + (t.he - ry + t.iy - 1) / t.iy;
    t.ntiles = t.tiles_x * t.tiles_y;
    t.inv_x = UINT_MAX / (unsigned)t.tiles_x;
    return t;
}

// workgroups of a launch over ntiles tiles: a multiple of 8 (see tile_of_block)
inline int sweep_grid(int ntiles) { return (ntiles + 7) / 8 * 8; }

// natural-layout sweeps
constexpr int NAT_R = 4;    // rows per wave
constexpr int NAT_NW = 16;  // waves per workgroup
constexpr int NAT_RY = NAT_R * NAT_NW;

// blocked sweeps
constexpr int BK_NW = 16;  // waves per workgroup
constexpr int BK_THREADS = 64 * BK_NW;

// The most sweeps of any launch (about 6 ms on a grid of one region, 14 in FP64), but
// that a solve in one workgroup returns at its first check after this many.
constexpr int kRegionSweeps = 16384;

// A max-update stop of the blocked sweeps falls at the end of a group of this
// many sweeps, counted from the last check.
constexpr int kStopGroup = 5;

constexpr int kTrackSweeps = 15;  // most sweeps of a tracking launch

// A launch's words.  The maxima are as many a tile as the launch has sweeps, which
// writer and reader hold anyway (a stride of its own in the arguments spilled 5 more
// scalars at 6 rows).
struct TrackOut {
    unsigned* bits;  // [ntiles]
    float* maxima;   // [ntiles][sweeps of the launch]
};
// bytes of two TrackOut for ntiles tiles and launches of up to `slots` sweeps, and
// their placement in `base`
inline size_t track_bytes(int ntiles, int slots) { return 2 * (size_t)ntiles * 4 * (1 + slots); }
inline TrackOut track_out(void* base, int ntiles, int slots, int which) {
    unsigned* u = static_cast<unsigned*>(base) + (size_t)which * ntiles * (1 + slots);
    return {u, reinterpret_cast<float*>(u + ntiles)};
}

struct TrackArgs {
    TrackOut out;    // this launch's
    TrackOut prev;   // the previous launch's, null for a batch's first
    int nprev;       // sweeps of the previous launch
    int first_prev;  // sweeps of the solve before it
    int group;       // sweeps the stop is rounded up to
    int lid;         // launch number within the solve
    int check_only;  // after a batch's last launch: decide, at most repeat it
    double tol;
};

// The tracking launches of a batch: each reads the words of the one before and
// leaves its own in the other TrackOut, the one that only checks too (it may repeat
// a launch and leave words, while workgroups that start later still read).
struct TrackBatch {
    void* base;  // both TrackOut
    int ntiles, slots;
    TrackArgs a;
    int launches;
    // the next launch: nsweeps sweeps after the solve's first `first`
    TrackArgs launch(int lid, int nsweeps, int first) {
        a.lid = lid;
        a.out = track_out(base, ntiles, slots, launches++ & 1);
        const TrackArgs now = a;
        a.prev = a.out;
        a.nprev = nsweeps;
        a.first_prev = first;
        return now;
    }
    // after the last one
    TrackArgs check(int lid) {
        TrackArgs now = launch(lid, 0, 0);
        now.check_only = 1;
        return now;
    }
};
inline TrackBatch track_batch(void* base, int ntiles, int slots, int group, double tol) {
    TrackBatch t{base, ntiles, slots, {}, 0};
    t.a.group = group;
    t.a.tol = tol;
    return t;
}

// Sweeps of a launch of the natural-layout sweeps: a grid of one region takes any
// number up to kRegionSweeps.
inline int natural_sweeps(const SweepTiles& t, int batch, bool track) {
    return t.ntiles > 1 ? t.halo / 2 : track ? kTrackSweeps : std::min(batch, kRegionSweeps);
}

// Tiles of the natural-layout sweeps: the halo (twice the sweeps of a launch)
// that is cheapest per sweep by what launches measured: about 5 us of dispatch,
// loads and stores, and 0.43 us (FP64) or 0.28 us (FP32) per half-sweep and
// round of one workgroup per CU.  At 400 x 400 in FP64 halos of 8 / 16 / 24 / 28
// take 2.18 / 1.49 / 1.29 / 1.25 us per sweep; at 700 x 700 the 369 tiles of halo
// 24 need a second round and take 2.12, halo 20 1.41.  track_room: bytes for a
// tracking launch's two TrackOut; cd_partials_bytes has room for those of the
// smallest halo on every shape.
SweepTiles natural_tiles(int w, int h, bool fp64, int batch, bool track, size_t track_room) {
    const double half_us = fp64 ? 0.43 : 0.28, fixed_us = 5.0;
    SweepTiles best = sweep_tiles(w, h, NAT_RY, 4);
    double best_cost = INFINITY;
    for (int halo = 4; halo <= 28; halo += 4) {
        const SweepTiles t = sweep_tiles(w, h, NAT_RY, halo);
        if (track && track_bytes(t.ntiles, natural_sweeps(t, batch, true)) > track_room) continue;
        const int sweeps = std::min(halo / 2, std::max(batch, 1));
        const double cost = (fixed_us + 2 * sweeps * half_us * div_up(t.ntiles, 256)) / sweeps;
        if (cost < best_cost) {
            best_cost = cost;
            best = t;
        }
    }
    return best;
}

// How a batch of sweeps is cut into launches: sweeps per launch, rows per wave.
struct BlockedPlan {
    int rows, sweeps;
    SweepTiles t;
};

// Time of a launch of `sweeps` sweeps over ntiles regions of 16 waves x `rows`
// rows, in us: a first region per CU, a second (resident beside it, except
// tracked at 8 rows), then every further one.  Fitted to launches of 4 to 19
// sweeps on grids of 300 to 4096 squared, to 1 to 3 % (rows 4: 6.1 us for 5
// sweeps of up to 256 regions, 8.6 for 14; rows 8: 10.0 for 8, 14.0 with two
// regions per CU, 44.4 with nine); a half costs less than a launch's first ones
// because waves at the inner borders sit out the later ones.
double blocked_launch_us(int rows, int sweeps, int ntiles, bool track) {
    struct Cost { double first, first_half, second, second_half, next, next_half; };
    static constexpr Cost cost[2][3] = {{{4.7, 0.142, 1.9, 0.005, 2.5, 0.023},
                                         {5.1, 0.205, 1.7, 0.063, 4.0, 0.025},
                                         {5.6, 0.268, 2.4, 0.100, 5.3, 0.042}},
                                        {{6.9, 0.246, 3.2, 0.045, 3.5, 0.080},
                                         {7.1, 0.332, 3.1, 0.137, 4.0, 0.134},
                                         {7.4, 0.440, 8.0, 0.287, 6.4, 0.352}}};
    const Cost& c = cost[track][(rows - 4) / 2];
    const int halves = 2 * sweeps, rounds = div_up(ntiles, 256);
    return c.first + c.first_half * halves + (rounds > 1 ? c.second + c.second_half * halves : 0.0) +
           (c.next + c.next_half * halves) * std::max(rounds - 2, 0);
}

// The cut of a batch of `batch` sweeps on a w x h grid that blocked_launch_us
// finds cheapest.  Per sweep, measured: 2048 x 2048 1.70 us (8 rows, 9 sweeps;
// 2.78 with 4 rows, 5 sweeps), 1024 x 1024 0.87 (8, 17; 1.29), 400 x 400 0.62
// (4, 14; 1.28); tracked, 400 x 400 1.12 (6, 15; 1.85 with 4 rows, 5 sweeps).
// Tracking launches take whole groups, a halo of whole waves,
// and need room for two TrackOut in track_room bytes; cd_partials_bytes has room
// for those of 4 rows and one group on every shape (48 bytes a region of 104
// columns, where the partials of up to 4 rows have 32 per 64).
BlockedPlan blocked_plan(int w, int h, int batch, bool track, size_t track_room) {
    BlockedPlan best{};
    double best_us = INFINITY;
    batch = std::max(batch, 1);
    for (int rows = 4; rows <= 8; rows += 2) {
        const int ry = BK_NW * rows, unit = track ? kStopGroup : 1;
        const int most = track ? kTrackSweeps / unit * unit : 19;
        for (int sweeps = unit; sweeps <= most; sweeps += unit) {
            const int halo = track ? div_up(2 * sweeps, rows) * rows : 2 * sweeps;
            if (ry - 2 * halo < 8) break;
            SweepTiles t = sweep_tiles(w, h, ry, halo);
            // a grid of one region takes any number of sweeps up to kRegionSweeps
            const int per = t.ntiles > 1 ? sweeps : track ? most : std::min(batch, kRegionSweeps);
            if (track && track_bytes(t.ntiles, per) > track_room) continue;
            const int full = batch / per, rest = batch % per;
            const double us = full * blocked_launch_us(rows, per, t.ntiles, track) +
                              (rest ? blocked_launch_us(rows, rest, t.ntiles, track) : 0.0);
            if (us < best_us) {
                best_us = us;
                best = BlockedPlan{rows, per, t};
            }
        }
    }
    return best;
}

}  // namespace
