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
// one region takes up to kRegionSweeps sweeps in one launch.
#pragma once

#include "cd_internal.h"
#include "cd_plan.h"

namespace {

// One region: its origin, the half-open range of cells it stores, and which of
// its sides lie on the grid border.
struct Region {
    int X0, Y0;
    int xs0, xs1, ys0, ys1;
    bool left, right, top, bottom;
};

__device__ __forceinline__ Region region_of(const SweepTiles& t, int tile) {
    Region g;
    // (no division and no branch: the loads that follow wait for this)
    const int q = (int)__umulhi((unsigned)tile, t.inv_x), rem = tile - q * t.tiles_x;
    const bool more = rem >= t.tiles_x;
    const int ty = more ? q + 1 : q, tx = more ? rem - t.tiles_x : rem;
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

// Sweeps (from the first) that wave `wave` of a region takes part in.  After
// half-sweep s only rows at distance >= s from an inner border are exact, and
// only those are read by exact ones later, so a wave whose rows all lie nearer
// need not update them: of the (wave + 1) R rows up to its last (counted from the
// inner border), the last is still exact after (wave + 1) R - 1 half-sweeps, and
// read by the next.  After that the wave only meets the barriers.
template <int R, int NW>
__device__ __forceinline__ int live_sweeps(const Region& g, int wave) {
    static_assert(R % 2 == 0, "whole sweeps");
    return min(g.top ? INT_MAX : (wave + 1) * R / 2, g.bottom ? INT_MAX : (NW - wave) * R / 2);
}

// XCD-aware tile order: gridDim.x is a multiple of 8 and consecutive workgroups
// go round-robin to the 8 XCDs; each XCD gets a contiguous band of tiles so
// that halo re-reads hit its own L2.  May return a tile >= ntiles.
__device__ __forceinline__ int tile_of_block(int ntiles) {
    const int per = (ntiles + 7) >> 3;  // gridDim.x / 8
    return (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
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

// lane_prev(v) + b, and in lane 0 own + b; lane_next(v) + b, and in lane 63
// own + b: an add with a wave shift does not write the lane without a source.
// (DPP reads a register two wait states after it was written, at the earliest.)
__device__ __forceinline__ float add_prev(float v, float b, float own) {
    float s = own + b;
    asm("s_nop 1\n\tv_add_f32_dpp %0, %1, %2 wave_shr:1 row_mask:0xf bank_mask:0xf"
        : "+v"(s) : "v"(v), "v"(b));
    return s;
}
__device__ __forceinline__ float add_next(float v, float b, float own) {
    float s = own + b;
    asm("s_nop 1\n\tv_add_f32_dpp %0, %1, %2 wave_shl:1 row_mask:0xf bank_mask:0xf"
        : "+v"(s) : "v"(v), "v"(b));
    return s;
}

// ---------------------------------------------------------------------------
// Max-update stop rule (solver.cpp:142) over launches of several sweeps.
//
// A tile of a launch leaves a word with bit j set when some cell it stores moved
// by tol or more in the launch's sweep j, and the largest |update| of each sweep
// (TrackOut; two of them, alternating).  The next launch of the batch ORs the
// previous one's words: the solve stops with the group of `group` sweeps that
// holds the first sweep whose bit is clear.  If that group ends the previous
// launch there is nothing left to do; otherwise the launch repeats the previous
// one from its input, which the ping-pong still holds, up to the end of that
// group.  Every workgroup reaches the same decision from the same words; the
// first one records it (stop_lid: the launch that found the stop; launches
// after it return at once, the workgroups of that launch itself do not look at
// it) with the largest update of the sweep.  The words are read beside the
// region's loads, which the decision would otherwise hold back; a word shared
// by all tiles (atomicOr) cost 0.6 us of a launch at 50 tiles and 9 us at 1000.
// ---------------------------------------------------------------------------
// The decision of a tracking launch, the same in every workgroup.
struct TrackPlan {
    int nsweeps;  // sweeps to take (0: nothing to do)
    bool redo;    // from the previous launch's input to its output
};

// Reductions of a wave by DPP (row shifts, then row broadcasts): the result of
// lane 63, in every lane.
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned dpp_or0(unsigned v) {
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
template <typename Op>
__device__ __forceinline__ unsigned wave_reduce(unsigned v, Op op) {
    v = op(v, dpp_or0<0x111, 0xf>(v));
    v = op(v, dpp_or0<0x112, 0xf>(v));
    v = op(v, dpp_or0<0x114, 0xf>(v));
    v = op(v, dpp_or0<0x118, 0xf>(v));
    v = op(v, dpp_or0<0x142, 0xa>(v));
    v = op(v, dpp_or0<0x143, 0xc>(v));
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ unsigned wave_or(unsigned v) {
    return wave_reduce(v, [](unsigned a, unsigned b) { return a | b; });
}
// largest of non-negative floats, which order like their bit patterns
__device__ __forceinline__ float wave_max_pos(float v) {
    return __uint_as_float(
        wave_reduce(__float_as_uint(v), [](unsigned a, unsigned b) { return max(a, b); }));
}

// this thread's part of the previous launch's words
template <int NW>
__device__ __forceinline__ unsigned track_load(const TrackArgs& a, int ntiles) {
    if (!a.prev.bits) return 0u;
    // (the first load is unconditional, so that nothing waits for it here)
    unsigned w = a.prev.bits[min((int)threadIdx.x, ntiles - 1)];
    for (int i = threadIdx.x + 64 * NW; i < ntiles; i += 64 * NW) w |= a.prev.bits[i];
    return w;
}

// words: track_load's; red: LDS of NW (<= 16) words.  All threads of the
// workgroup (64*NW) must call it.
template <int NW>
__device__ __forceinline__ TrackPlan track_decide(const TrackArgs& a, SolveDev* st, int ntiles,
                                                  int nsweeps, unsigned words, unsigned* red) {
    static_assert(NW <= 16, "one row of lanes reads the waves' words");
    TrackPlan p{a.check_only ? 0 : nsweeps, false};
    if (st->stop_lid < a.lid) return TrackPlan{0, false};
    if (!a.prev.bits) return p;
    words = wave_or(words);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = words;
    __syncthreads();
    const unsigned over = wave_or(red[min((int)threadIdx.x & 15, NW - 1)]);
    const unsigned clear = ~over & ((1u << a.nprev) - 1u);
    const int stop = clear ? __ffs((int)clear) - 1 : -1;
    const int end = stop >= 0 ? min((stop / a.group + 1) * a.group, a.nprev) : 0;
    if (stop >= 0) {
        p.nsweeps = end < a.nprev ? end : 0;
        p.redo = true;
    }
    if (blockIdx.x == 0 && (stop >= 0 || a.check_only)) {
        const int j = stop >= 0 ? stop : a.nprev - 1;
        float m = 0.f;
        for (int i = threadIdx.x; i < ntiles; i += 64 * NW)
            m = fmaxf(m, a.prev.maxima[(size_t)i * a.nprev + j]);
        m = wave_max_pos(m);
        __syncthreads();  // red has been read
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = __float_as_uint(m);
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int v = 1; v < NW; ++v) m = fmaxf(m, __uint_as_float(red[v]));
            st->last_max_update = (double)m;
            if (stop >= 0) {
                st->sweeps_at_done = a.first_prev + end;
                st->done = 1;
                __hip_atomic_store(&st->stop_lid, a.lid, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    return p;
}

// The end of a tracking launch's workgroup: its tile's largest updates from
// those of the lanes, one wave per sweep, and the tile's word.
template <int NW>
__device__ __forceinline__ void track_store(const TrackArgs& a, const float (*smax)[NW][64],
                                            unsigned* red, int tile, int nsweeps, int wave,
                                            int lane) {
    __syncthreads();
    unsigned over = 0u;
    for (int j = wave; j < nsweeps; j += NW) {
        float m = smax[j][0][lane];
        for (int v = 1; v < NW; ++v) m = fmaxf(m, smax[j][v][lane]);
        m = wave_max_pos(m);
        if (lane == 0) a.out.maxima[(size_t)tile * nsweeps + j] = m;
        if (!((double)m < a.tol)) over |= 1u << j;
    }
    if (lane == 0) red[wave] = over;
    __syncthreads();
    if (wave == 0) {
        over = wave_or(red[min(lane & 15, NW - 1)]);
        if (lane == 0) a.out.bits[tile] = over;
    }
}

}  // namespace
