// Regions of the temporally blocked red-black sweeps, shared by the sweep
// kernels of cd_solver.hip.
//
// A workgroup of NW waves holds a region of NW*R rows x 128 columns: lane l of
// wave v keeps the cells 2l and 2l+1 (one per colour) of rows v*R .. v*R+R-1 in
// registers.  The regions of a grid overlap by `halo` cells on every inner
// side: after n <= halo half-sweeps the cells at distance >= halo from an inner
// region border equal n global half-sweeps, and those are stored.  Regions at
// the grid border end there (no halo on that side): what lies beyond reads as
// zero, so a border cell's neighbour sum needs no weights, and a grid that fits
// one region takes any number of sweeps in one launch.
#pragma once

#include <algorithm>
#include <climits>

#include "cd_internal.h"

namespace {

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
    return t;
}

// workgroups of a launch over ntiles tiles: a multiple of 8 (see tile_of)
inline int sweep_grid(int ntiles) { return (ntiles + 7) / 8 * 8; }

// One region: its origin, the half-open range of cells it stores, and which of
// its sides lie on the grid border.
struct Region {
    int X0, Y0;
    int xs0, xs1, ys0, ys1;
    bool left, right, top, bottom;
};

__device__ __forceinline__ Region region_of(const SweepTiles& t, int tile) {
    Region g;
    const int ty = tile / t.tiles_x, tx = tile - ty * t.tiles_x;
    g.X0 = max(min(tx * t.ix, t.we - SW_RX), 0);
    g.Y0 = max(min(ty * t.iy, t.he - t.ry), 0);
    g.left = tx == 0;
    g.right = tx == t.tiles_x - 1;
    g.top = ty == 0;
    g.bottom = ty == t.tiles_y - 1;
    g.xs0 = g.left ? 0 : tx * t.ix + t.halo;
    g.xs1 = g.right ? t.w : (tx + 1) * t.ix + t.halo;
    g.ys0 = g.top ? 0 : ty * t.iy + t.halo;
    g.ys1 = g.bottom ? t.h : (ty + 1) * t.iy + t.halo;
    return g;
}

// XCD-aware tile order: gridDim.x is a multiple of 8 and consecutive workgroups
// go round-robin to the 8 XCDs; each XCD gets a contiguous band of tiles so
// that halo re-reads hit its own L2.  May return a tile >= ntiles.
__device__ __forceinline__ int tile_of_block() {
    const int per = gridDim.x >> 3;
    return (blockIdx.x & 7) * per + (blockIdx.x >> 3);
}

// value of lane l-1 (0 in lane 0) / lane l+1 (0 in lane 63): DPP wave shifts
__device__ __forceinline__ float lane_prev(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_next(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_prev(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x138, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x138, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_next(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x130, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x130, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// ---------------------------------------------------------------------------
// Max-update stop rule (solver.cpp:142) over launches of several sweeps.
//
// A launch leaves the largest |update| of each of its sweeps over the cells it
// stores, per tile, in tmax (kTrackSweeps slots a tile; two such arrays,
// alternating).  The next launch of the batch first reduces the previous
// launch's array: the solve stops with the group of `group` sweeps that holds
// the first sweep below tol.  If that group ends the previous launch there is
// nothing left to do; otherwise the launch repeats the previous one from its
// input, which the ping-pong still holds, up to the end of that group.  Every
// workgroup reaches the same decision from the same array; the first one
// records it (stop_lid: the launch that found the stop; launches after it
// return at once, the workgroups of that launch itself do not look at it).
// ---------------------------------------------------------------------------
constexpr int kTrackSweeps = 16;  // most sweeps of a tracking launch

struct TrackArgs {
    float* tmax;        // this launch's array
    const float* prev;  // the previous launch's array, null for a batch's first
    int nprev;          // sweeps of the previous launch
    int first_prev;     // sweeps of the solve before it
    int group;          // sweeps the stop is rounded up to
    int lid;            // launch number within the solve
    int check_only;     // after a batch's last launch: decide, at most repeat it
    double tol;
};

// The sweep decision of a tracking launch, the same in every workgroup.
struct TrackPlan {
    int nsweeps;  // sweeps to take (0: nothing to do)
    bool redo;    // from the previous launch's input to its output
};

// red: LDS of NW * kTrackSweeps floats.  All threads of the workgroup (64*NW)
// must call it.
template <int NW>
__device__ __forceinline__ TrackPlan track_decide(const TrackArgs& a, SolveDev* st, int ntiles,
                                                  int nsweeps, float* red) {
    TrackPlan p{a.check_only ? 0 : nsweeps, false};
    if (!a.prev) return p;
    static_assert(kTrackSweeps == 16, "lane j of 16 takes sweep j");
    float m = 0.f;
    for (int i = threadIdx.x; i < ntiles * kTrackSweeps; i += 64 * NW) m = fmaxf(m, a.prev[i]);
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane < kTrackSweeps) red[wave * kTrackSweeps + lane] = m;
    __syncthreads();
    float mj = lane < kTrackSweeps ? red[lane] : 0.f;
    if (lane < kTrackSweeps)
        for (int v = 1; v < NW; ++v) mj = fmaxf(mj, red[v * kTrackSweeps + lane]);
    const unsigned long long below = __ballot(lane < a.nprev && (double)mj < a.tol);
    const int stop = below ? __ffsll((long long)below) - 1 : -1;
    const float last = __shfl(mj, stop >= 0 ? stop : a.nprev - 1, 64);
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (first) st->last_max_update = (double)last;
    if (stop >= 0) {
        const int end = min((stop / a.group + 1) * a.group, a.nprev);
        p.nsweeps = end < a.nprev ? end : 0;
        p.redo = true;
        if (first) {
            st->sweeps_at_done = a.first_prev + end;
            st->done = 1;
            __hip_atomic_store(&st->stop_lid, a.lid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    return p;
}

}  // namespace
