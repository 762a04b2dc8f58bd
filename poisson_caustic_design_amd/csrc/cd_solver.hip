// Poisson solver for the reference operator (src/solver.cpp:12-61):
//     sum_{valid nbr n} phi_n - cnt * phi_c = D_c
// on the cell-centred grid with Neumann edges (a neighbour outside the grid or
// on a NaN hole of D is not counted).  Replaces poisson_solver
// (src/solver.h:8, src/solver.cpp:70-147).
//
// Method (MI355X-first):
//   * red-black SOR.  Red-black ordering removes the reference's tile data
//     race by construction.  omega defaults to the optimum for this operator
//     (cd_sor_omega); the reference's 2/(1+3.14159265/width) (solver.cpp:71)
//     is kept for the drop-in entry points.
//   * CD_PREC_MIXED: sweeps run in FP32 on a correction e with the right-hand
//     side r = P b - A phi64 (FP64 residual, zero-mean projected); every
//     `check_every` sweeps e is folded into the FP64 base (defect correction)
//     and the FP64 relative residual is evaluated on the device.
//   * CD_PREC_FP64: the same sweeps in FP64 directly on phi.
//   * stop rules are evaluated on the device.  Residual rule: a check sets the
//     `done` flag, and the host, which waits for it, enqueues no more sweeps (a
//     launch that went out early only writes the correction).  Max-update rule:
//     every launch decides from the words of the one before whether the solve
//     stopped in it; then it repeats that launch up to the stop and records its
//     number in `stop_lid`, and the launches after it return at once.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>

#include "cd_internal.h"
#include "cd_sweeps.h"

namespace {

// mask bits: neighbour validity (left, up, right, down) and "cell is a hole"
constexpr uint8_t M_L = 1, M_U = 2, M_R = 4, M_D = 8, M_HOLE = 0x80;

// ---------------------------------------------------------------------------
// right-hand-side statistics, hole mask
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_build_mask(const double* __restrict__ b,
                                                    uint8_t* __restrict__ mask, int w, int h,
                                                    double* __restrict__ partials) {
    __shared__ double smem[16];
    int x = blockIdx.x * blockDim.x + threadIdx.x;
    int y = blockIdx.y * blockDim.y + threadIdx.y;
    double holes = 0.0;
    if (x < w && y < h) {
        size_t i = (size_t)y * w + x;
        uint8_t m = 0;
        if (isnan(b[i])) { m = M_HOLE; holes = 1.0; }
        if (x > 0 && !isnan(b[i - 1])) m |= M_L;
        if (y > 0 && !isnan(b[i - w])) m |= M_U;
        if (x < w - 1 && !isnan(b[i + 1])) m |= M_R;
        if (y < h - 1 && !isnan(b[i + w])) m |= M_D;
        mask[i] = m;
    }
    double s = cd_block_sum(holes, smem);
    if (threadIdx.x == 0 && threadIdx.y == 0)
        partials[blockIdx.y * gridDim.x + blockIdx.x] = s;
}

// pass 1: sum of b over non-hole cells; pass 2 (mean given): sum of (b-mean)^2
__global__ __launch_bounds__(256) void k_rhs_moments(const double* __restrict__ b, int w, int h,
                                                     const SolveDev* __restrict__ st, int pass,
                                                     double* __restrict__ partials) {
    __shared__ double smem[16];
    int x = blockIdx.x * blockDim.x + threadIdx.x;
    int y = blockIdx.y * blockDim.y + threadIdx.y;
    double v = 0.0;
    if (x < w && y < h) {
        double bv = b[(size_t)y * w + x];
        if (!isnan(bv)) {
            if (pass == 0) v = bv;
            else { double d = bv - st->bmean; v = d * d; }
        }
    }
    double s = cd_block_sum(v, smem);
    if (threadIdx.x == 0 && threadIdx.y == 0)
        partials[blockIdx.y * gridDim.x + blockIdx.x] = s;
}

// single block: reduce partials and finish the right-hand-side statistics
__global__ void k_rhs_finish(const double* __restrict__ partials, int nblocks, SolveDev* st,
                             int pass, double count) {
    __shared__ double smem[16];
    double s = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x) s += partials[b];
    s = cd_block_sum(s, smem);
    if (threadIdx.x == 0) {
        if (pass == 0) {
            st->done = 0;
            st->done_check = -1;
            st->sweeps_at_done = -1;
            st->checks = 0;
            st->bsum = s;
            st->bmean = count > 0 ? s / count : 0.0;
            st->rel = INFINITY;
            st->rel0 = INFINITY;
            st->last_max_update = INFINITY;
            st->rmean32 = 0.f;
            st->cur = 0;
            st->stop_lid = INT_MAX;
        } else {
            st->bnorm = sqrt(s);
        }
    }
}

// ---------------------------------------------------------------------------
// defect correction, natural layout: phi64 += the current correction of the
// ping-pong pair; the next batch of sweeps starts from ea = 0
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_flush(double* __restrict__ phi, float* __restrict__ ea,
                                               const float* __restrict__ eb,
                                               const SolveDev* __restrict__ st, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    const bool second = st->cur != 0;
    for (; i < n; i += stride) {
        const float ev = second ? eb[i] : ea[i];
        phi[i] += (double)ev;
        ea[i] = 0.f;
    }
}

__device__ __forceinline__ size_t brick_row(const Brick& b, int c, int Y) {
    return (size_t)c * b.plane + ((size_t)(Y >> 3) * b.nbx) * 512 + (size_t)(Y & 7) * 64;
}
__device__ __forceinline__ unsigned brick_col(int j) { return (unsigned)((j >> 6) * 512 + (j & 63)); }
// bricked index of cell (x, y)
__device__ __forceinline__ size_t brick_at(const Brick& bk, int x, int y) {
    return brick_row(bk, (x + y) & 1, y) + brick_col(x >> 1);
}
// XCD-contiguous workgroup order.  The dispatcher hands consecutive workgroups
// (x fastest, then y, then z) round-robin to the 8 XCDs, each with its own L2;
// this maps the dispatch index to an order in which XCD k takes the k-th
// contiguous eighth of the n workgroups (a bijection on [0, n)), so that
// neighbouring workgroups, whose halos overlap, share an L2.
__device__ __forceinline__ int xcd_order() {
    const int n = gridDim.x * gridDim.y * gridDim.z;
    const int lin = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    const int q = n >> 3, r = n & 7, x = lin & 7;
    return x * q + min(x, r) + (lin >> 3);
}

// Buffer access to a bricked plane pair of at most 2^31 bytes: scalar
// resource + scalar (row) byte offset + the lane's vector byte offset, no
// per-lane 64-bit address arithmetic.  Every access stays in range.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const void* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
template <typename T>
__device__ __forceinline__ T buf_load(__amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned soff);
template <>
__device__ __forceinline__ float buf_load<float>(__amdgpu_buffer_rsrc_t rs, unsigned voff,
                                                 unsigned soff) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, voff, soff, 0));
}
template <>
__device__ __forceinline__ unsigned short buf_load<unsigned short>(__amdgpu_buffer_rsrc_t rs,
                                                                   unsigned voff, unsigned soff) {
    return __builtin_amdgcn_raw_buffer_load_b16(rs, voff, soff, 0);
}

// FP32 -> BF16 (round to nearest even) and back; finite inputs only
__device__ __forceinline__ unsigned short f32_to_bf16(float x) {
    const unsigned u = __float_as_uint(x);
    return (unsigned short)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float bf16_to_f32(unsigned short v) {
    return __uint_as_float((unsigned)v << 16);
}
// right-hand side element of the blocked sweeps: BF16 or FP32 storage
__device__ __forceinline__ float rhs_to_f32(unsigned short v) { return bf16_to_f32(v); }
__device__ __forceinline__ float rhs_to_f32(float v) { return v; }

// blocked path: fold the current ping-pong correction into phi64, zero both
__global__ __launch_bounds__(256) void k_flush_packed(double* __restrict__ phi,
                                                      float* __restrict__ ea,
                                                      float* __restrict__ eb,
                                                      const SolveDev* __restrict__ st, int w,
                                                      int h, Brick bk) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= w || y >= h) return;
    const size_t pi = brick_row(bk, (x + y) & 1, y) + brick_col(x >> 1);
    const float ev = st->cur ? eb[pi] : ea[pi];
    phi[(size_t)y * w + x] += (double)ev;
    ea[pi] = 0.f;
    eb[pi] = 0.f;
}

// ---------------------------------------------------------------------------
// FP64 residual r = (b - bmean) - A phi  (+ FP32 copy for the inner sweeps)
// partials[block] = (sum r, sum r^2)
// ---------------------------------------------------------------------------
// OUT: 0 norms only, 1 FP32 copy of r (natural layout), 2 BF16 copy of r
// (bricked layout, blocked sweeps), 3 FP32 copy of r in the bricked layout
// (blocked sweeps under the max-update rule).  A thread takes ROWS rows (stride
// blockDim.y) of its column before the two block reductions, so a launch
// reduces over few workgroups.  The loads of 4 rows at a time are issued
// before the first is used (clamped, always in-range addresses; cells outside
// the grid contribute nothing): a thread keeps 24 loads in flight instead of
// waiting for each row in turn.
template <int OUT, int ROWS, bool MASK>
__device__ __forceinline__ void residual_rows(const double* __restrict__ phi,
                                              const double* __restrict__ b,
                                              const uint8_t* __restrict__ mask, double bmean,
                                              float* __restrict__ r32,
                                              unsigned short* __restrict__ r16, const Brick& bk,
                                              int w, int h, double& rs, double& rq) {
    constexpr int G = ROWS < 4 ? ROWS : 4;  // rows whose loads are in flight together
    const int ob = xcd_order();
    const int x0 = (ob % gridDim.x) * blockDim.x + threadIdx.x;
    const int y0 = (ob / gridDim.x) * blockDim.y * ROWS + threadIdx.y;
    const int x = min(x0, w - 1);
    const int xl = max(x - 1, 0), xr = min(x + 1, w - 1);
#pragma unroll
    for (int g = 0; g < ROWS; g += G) {
        double c[G], l[G], r[G], u[G], d[G], bb[G];
        uint8_t m[G];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const int y = min(y0 + (g + k) * (int)blockDim.y, h - 1);
            const size_t row = (size_t)y * w;
            c[k] = phi[row + x];
            l[k] = phi[row + xl];
            r[k] = phi[row + xr];
            u[k] = phi[(size_t)max(y - 1, 0) * w + x];
            d[k] = phi[(size_t)min(y + 1, h - 1) * w + x];
            bb[k] = b[row + x];
            if (MASK) m[k] = mask[row + x];
        }
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const int y = y0 + (g + k) * (int)blockDim.y;
            if (x0 >= w || y >= h) break;
            double s = 0.0, cnt = 0.0;
            bool hole = false;
            if (MASK) {
                hole = (m[k] & M_HOLE) != 0;
                if (m[k] & M_L) { cnt += 1.0; s += l[k]; }
                if (m[k] & M_U) { cnt += 1.0; s += u[k]; }
                if (m[k] & M_R) { cnt += 1.0; s += r[k]; }
                if (m[k] & M_D) { cnt += 1.0; s += d[k]; }
            } else {
                if (x > 0) { cnt += 1.0; s += l[k]; }
                if (y > 0) { cnt += 1.0; s += u[k]; }
                if (x < w - 1) { cnt += 1.0; s += r[k]; }
                if (y < h - 1) { cnt += 1.0; s += d[k]; }
            }
            double rv = 0.0;
            if (!hole) {
                rv = (bb[k] - bmean) - (s - cnt * c[k]);
                rs += rv;
                rq += rv * rv;
            }
            const size_t i = (size_t)y * w + x;
            if (OUT == 1) r32[i] = (float)rv;
            if (OUT == 2)
                r16[brick_row(bk, (x + y) & 1, y) + brick_col(x >> 1)] = f32_to_bf16((float)rv);
            if (OUT == 3) r32[brick_row(bk, (x + y) & 1, y) + brick_col(x >> 1)] = (float)rv;
        }
    }
}
template <int OUT, int ROWS>
__global__ __launch_bounds__(256) void k_residual(const double* __restrict__ phi0,
                                                  const double* __restrict__ phi1,
                                                  const double* __restrict__ b,
                                                  const uint8_t* __restrict__ mask,
                                                  const SolveDev* __restrict__ st,
                                                  float* __restrict__ r32,
                                                  unsigned short* __restrict__ r16, Brick bk,
                                                  int w, int h, double* __restrict__ partials) {
    __shared__ double smem[32];
    // FP64 sweeps: the iterate is in either buffer of the pair (phi0, phi1)
    const double* __restrict__ phi = phi1 && st->cur ? phi1 : phi0;
    const double bmean = st->bmean;
    double rs = 0.0, rq = 0.0;
    if (mask)
        residual_rows<OUT, ROWS, true>(phi, b, mask, bmean, r32, r16, bk, w, h, rs, rq);
    else
        residual_rows<OUT, ROWS, false>(phi, b, mask, bmean, r32, r16, bk, w, h, rs, rq);
    double aq[2] = {rs, rq};
    cd_block_sum_n(aq, smem);
    const double a = aq[0], q = aq[1];
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        const size_t bid = (size_t)xcd_order();
        partials[2 * bid] = a;
        partials[2 * bid + 1] = q;
    }
}
// launch of k_residual<OUT, rows> for rows in {1, 2, 4, 8}
template <int OUT>
void launch_residual(int rows, dim3 grid, dim3 blk, hipStream_t s, const double* phi,
                     const double* phi1, const double* b, const uint8_t* mask, const SolveDev* st, float* r32,
                     unsigned short* r16, const Brick& bk, int w, int h, double* partials) {
    switch (rows) {
    case 8: hipLaunchKernelGGL((k_residual<OUT, 8>), grid, blk, 0, s, phi, phi1, b, mask, st, r32, r16, bk, w, h, partials); break;
    case 4: hipLaunchKernelGGL((k_residual<OUT, 4>), grid, blk, 0, s, phi, phi1, b, mask, st, r32, r16, bk, w, h, partials); break;
    case 2: hipLaunchKernelGGL((k_residual<OUT, 2>), grid, blk, 0, s, phi, phi1, b, mask, st, r32, r16, bk, w, h, partials); break;
    default: hipLaunchKernelGGL((k_residual<OUT, 1>), grid, blk, 0, s, phi, phi1, b, mask, st, r32, r16, bk, w, h, partials); break;
    }
}

// single block: finish a convergence check.  The status also goes to the
// host's pinned coherent mirror, its sequence word `seq` last, after every
// other word has been written: the host waits for that word instead of
// synchronising the stream (a round trip of ~30 us per check).
__global__ void k_check(const double* __restrict__ partials, int nblocks, SolveDev* st,
                        SolveDev* host_st, unsigned seq, double count, int check_id,
                        int stop_rule, double tol) {
    constexpr int kWords = (int)(sizeof(SolveDev) / 4);
    constexpr int kSeq = (int)(offsetof(SolveDev, seq) / 4);
    static_assert(sizeof(SolveDev) % 4 == 0 && kWords <= 1024, "status words");
    __shared__ double smem[32];
    __shared__ unsigned words[kWords];
    double a = 0.0, q = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x) {
        a += partials[2 * b];
        q += partials[2 * b + 1];
    }
    double aq[2] = {a, q};
    cd_block_sum_n(aq, smem);
    a = aq[0];
    q = aq[1];
    if (threadIdx.x == 0) {
        double mean = count > 0 ? a / count : 0.0;
        double rn2 = q - count * mean * mean;
        // rounding can make rn2 slightly negative; a NaN must stay NaN (a
        // non-finite iterate never meets the stop rule)
        double rn = rn2 > 0.0 ? sqrt(rn2) : (rn2 == rn2 ? 0.0 : rn2);
        double rel = st->bnorm > 0 ? rn / st->bnorm : (rn > 0 ? INFINITY : 0.0);
        st->rsum = a;
        st->rnorm = rn;
        st->rel = rel;
        if (st->checks == 0) st->rel0 = rel;
        st->checks += 1;
        st->rmean32 = (float)mean;
        if (stop_rule == CD_STOP_RESIDUAL && !st->done && rel <= tol) {
            st->done = 1;
            st->done_check = check_id;
        }
        st->seq = seq;
        const unsigned* src = reinterpret_cast<const unsigned*>(st);
        for (int k = 0; k < kWords; ++k) words[k] = src[k];
    }
    __syncthreads();
    // one word per thread, then the sequence word as a system-scope release
    // (it makes the other threads' words, ordered before it by the barrier,
    // visible to the host first)
    unsigned* dst = reinterpret_cast<unsigned*>(host_st);
    if (threadIdx.x < kWords && threadIdx.x != kSeq) dst[threadIdx.x] = words[threadIdx.x];
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(dst + kSeq, words[kSeq], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// Temporally blocked red-black SOR in the natural row-major layout: FP64 sweeps
// (T = double, e the iterate, r = b) and FP32 sweeps with holes or on grids the
// bricked layout cannot address (T = float, e the correction).  Regions and
// stores as described in cd_sweeps.h.  The update is the reference's
//   delta = omega / cnt * (sum - cnt * val - rhs)   (solver.cpp:47, 56)
// with the operations, and hence the bits, of one half-sweep over the whole
// grid per launch; colour 0 is x+y even.  A neighbour outside the grid or on a
// hole holds zero in the region, so it drops out of the sum; its own update has
// the factor oc = 0 (and with a mask a select: a cell with no neighbour left has
// an infinite update, which 0 would turn into a NaN beside it).  oc = omega / cnt
// and cnt come per cell on tiles at the grid border and with a mask, and are
// constants elsewhere.
//
// A half-sweep per launch was bound by its launches: two of 3.8 us (plus gaps)
// per sweep on a 512 x 512 grid, where 12 sweeps in one launch take 12.9 us, of
// which border tiles set the pace: their omega / cnt are chosen from four values
// (a division per cell before: 13.6 us), and a missing row is read from a row of
// zeros instead of being selected in every half-sweep.
// ---------------------------------------------------------------------------
// Per-cell constants of a wave at the grid border or with a mask.
template <typename T>
struct NatCells {
    T oc[2][NAT_R], cnt[2][NAT_R];
    unsigned live;  // bit c * NAT_R + k: the cell is in the grid and no hole
};

__device__ __forceinline__ float nat_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double nat_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// Rows K0 <= k < K1 of a half-sweep of colour C; mx[p] takes the largest
// |update| of the lane's cells of column parity p.
enum { NAT_INNER = 0, NAT_EDGE = 1, NAT_MASK = 2 };
template <typename T, int C, int KIND, bool TRACK, int K0, int K1>
__device__ __forceinline__ void nat_half(T (&ev)[2][NAT_R], const T (&rv)[2][NAT_R],
                                         const NatCells<T>& cl, T oc4, T up_row, T down_row,
                                         T (&mx)[2]) {
#pragma unroll
    for (int k = K0; k < K1; ++k) {
        const int p = (k + C) & 1;  // column parity of colour-C cells in row k
        const T o = ev[1 - C][k];
        const T up = k > 0 ? ev[1 - C][k - 1] : up_row;
        const T down = k < NAT_R - 1 ? ev[1 - C][k + 1] : down_row;
        const T left = p ? o : lane_prev(o);
        const T right = p ? lane_next(o) : o;
        const T s = left + up + right + down;
        const T v = ev[C][k];
        // (4 v is exact: the fused form has the unfused one's bits)
        const T res = KIND ? s - cl.cnt[C][k] * v : nat_fma((T)-4, v, s);
        const T d = (KIND ? cl.oc[C][k] : oc4) * (res - rv[C][k]);
        const T nv = v + d;
        if (KIND == NAT_MASK) ev[C][k] = (cl.live >> (C * NAT_R + k)) & 1u ? nv : (T)0;
        else ev[C][k] = nv;
        if (TRACK) mx[p] = fmax(mx[p], fabs(d));  // (0, or a NaN that fmax drops, where oc = 0)
    }
}

// omega over 1, 2, 3 and 4 neighbours
template <typename T>
struct NatOmega {
    T o1, o2, o3, o4;
};

// Everything between the loads and the stores of a region: nsweeps sweeps, of
// which the wave takes part in the first `live`.  edge_up / edge_down: the wave's
// first / last row has no row beyond it (it reads the row of zeros in xch[2]).
template <typename T, int KIND, bool TRACK>
__device__ __forceinline__ void nat_run(T (&ev)[2][NAT_R], const T (&rv)[2][NAT_R],
                                        const NatCells<T>& cl, T (*xch)[NAT_NW][2][64], T oc4,
                                        bool edge_up, bool edge_down, int wave, int lane,
                                        int nsweeps, int live, float (*smax)[NAT_NW][64],
                                        bool track0, bool track1) {
    const T* above[2];
    const T* below[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        above[c] = KIND && edge_up ? xch[2][0][0] : xch[c][max(wave - 1, 0)][1];
        below[c] = KIND && edge_down ? xch[2][0][0] : xch[c][min(wave + 1, NAT_NW - 1)][0];
    }
    auto publish = [&](int c) {
        xch[c][wave][0][lane] = ev[c][0];
        xch[c][wave][1][lane] = ev[c][NAT_R - 1];
    };
    const int mine = min(nsweeps, live);
    for (int j = 0; j < mine; ++j) {
        T mx[2] = {(T)0, (T)0};
        T up, down;
        publish(1);
        nat_half<T, 0, KIND, TRACK, 1, NAT_R - 1>(ev, rv, cl, oc4, (T)0, (T)0, mx);
        __syncthreads();
        up = above[1][lane];
        down = below[1][lane];
        nat_half<T, 0, KIND, TRACK, 0, 1>(ev, rv, cl, oc4, up, down, mx);
        nat_half<T, 0, KIND, TRACK, NAT_R - 1, NAT_R>(ev, rv, cl, oc4, up, down, mx);
        publish(0);
        nat_half<T, 1, KIND, TRACK, 1, NAT_R - 1>(ev, rv, cl, oc4, (T)0, (T)0, mx);
        __syncthreads();
        up = above[0][lane];
        down = below[0][lane];
        nat_half<T, 1, KIND, TRACK, 0, 1>(ev, rv, cl, oc4, up, down, mx);
        nat_half<T, 1, KIND, TRACK, NAT_R - 1, NAT_R>(ev, rv, cl, oc4, up, down, mx);
        if (TRACK) {
            smax[j][wave][lane] = fmaxf(track0 ? (float)mx[0] : 0.f, track1 ? (float)mx[1] : 0.f);
        }
    }
    for (int j = mine; j < nsweeps; ++j) {  // (no row of the wave counts for the maxima)
        __syncthreads();
        __syncthreads();
        if (TRACK) smax[j][wave][lane] = 0.f;
    }
}

template <typename T, bool TRACK>
__global__ __launch_bounds__(64 * NAT_NW) void k_rb_natural(
    const T* ein, T* eout, const T* __restrict__ r, const uint8_t* __restrict__ mask,
    SweepTiles tiles, int nsweeps, NatOmega<T> om, const T* __restrict__ rmean, SolveDev* st,
    int out_index, TrackArgs track) {
    __shared__ T xch[3][NAT_NW][2][64];  // the third: one row of zeros
    __shared__ float smax[TRACK ? kTrackSweeps : 1][NAT_NW][64];
    __shared__ unsigned red[TRACK ? NAT_NW : 1];
    // (what the loads' addresses need is read in one go)
    asm volatile("" ::"s"(ein), "s"(r), "s"(mask), "s"(rmean), "s"(tiles.w), "s"(tiles.ntiles));
    const int tile = tile_of_block(tiles.ntiles);
    if (tile >= tiles.ntiles) return;
    const Region g = region_of(tiles, tile);
    const int w = tiles.w, h = tiles.h;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x0 = g.X0 + 2 * lane, Yw = g.Y0 + wave * NAT_R;
    T ev[2][NAT_R], rv[2][NAT_R];
    NatCells<T> cl;
    uint8_t mk[2][NAT_R];
    // branch-free loads from clamped addresses: all in flight together
    const unsigned col[2] = {(unsigned)min(x0, w - 1), (unsigned)min(x0 + 1, w - 1)};
    auto row = [&](int k) { return (size_t)min(Yw + k, h - 1) * w; };
    const unsigned words = TRACK ? track_load<NAT_NW>(track, tiles.ntiles) : 0u;
#pragma unroll
    for (int k = 0; k < NAT_R; ++k)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            ev[c][k] = (ein + row(k))[col[(k + c) & 1]];
            rv[c][k] = (r + row(k))[col[(k + c) & 1]];
            mk[c][k] = 0;
        }
    if (mask) {
#pragma unroll
        for (int k = 0; k < NAT_R; ++k)
#pragma unroll
            for (int c = 0; c < 2; ++c) mk[c][k] = (mask + row(k))[col[(k + c) & 1]];
    }
    const T rm = *rmean;
    if (TRACK) {
        const TrackPlan plan =
            track_decide<NAT_NW>(track, st, tiles.ntiles, nsweeps, words, red);
        if (plan.nsweeps == 0) return;
        nsweeps = __builtin_amdgcn_readfirstlane(plan.nsweeps);
        if (plan.redo) {
            const T* in = eout;
            eout = const_cast<T*>(ein);
            out_index ^= 1;
#pragma unroll
            for (int k = 0; k < NAT_R; ++k)
#pragma unroll
                for (int c = 0; c < 2; ++c) ev[c][k] = (in + row(k))[col[(k + c) & 1]];
        }
    }
    const bool general = mask || g.left || g.right || g.top || g.bottom;
    const T oc4 = om.o4;
    if (general) {
        cl.live = 0u;
        if (wave == 0) xch[2][0][0][lane] = (T)0;  // (the sweeps' first barrier follows)
#pragma unroll
        for (int k = 0; k < NAT_R; ++k)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int x = x0 + ((k + c) & 1), y = Yw + k;
                const uint8_t m = mk[c][k];
                int n = (int)(x > 0) + (int)(y > 0) + (int)(x < w - 1) + (int)(y < h - 1);
                if (mask) n = __popc(m & (M_L | M_U | M_R | M_D));
                const bool live = x < w && y < h && !(m & M_HOLE);
                if (live) cl.live |= 1u << (c * NAT_R + k);
                else ev[c][k] = (T)0;
                cl.cnt[c][k] = (T)n;
                T oc = om.o4;  // (selects, no branches)
                oc = n == 3 ? om.o3 : oc;
                oc = n == 2 ? om.o2 : oc;
                oc = n == 1 ? om.o1 : oc;
                oc = n == 0 ? (T)INFINITY : oc;
                cl.oc[c][k] = live ? oc : (T)0;
                rv[c][k] = live ? rv[c][k] - rm : (T)0;
            }
    } else {
#pragma unroll
        for (int k = 0; k < NAT_R; ++k) {
            rv[0][k] = rv[0][k] - rm;
            rv[1][k] = rv[1][k] - rm;
        }
    }
    // the cells whose updates count for the stop rule: those at distance >= halo
    // from the region's inner borders (all exact; two tiles may count one)
    const int dy0 = wave * NAT_R, hl = tiles.halo;
    const bool rows_ok = (g.top || dy0 >= hl) && (g.bottom || dy0 + NAT_R <= NAT_RY - hl);
    auto col_ok = [&](int dx) { return rows_ok && (g.left || dx >= hl) && (g.right || dx < SW_RX - hl); };
    const bool t0 = TRACK && col_ok(2 * lane), t1 = TRACK && col_ok(2 * lane + 1);
    const int live = live_sweeps<NAT_R, NAT_NW>(g, wave);
    const bool up0 = g.top && wave == 0, down0 = g.bottom && wave == NAT_NW - 1;
    if (mask)
        nat_run<T, NAT_MASK, TRACK>(ev, rv, cl, xch, oc4, up0, down0, wave, lane, nsweeps, live, smax,
                                    t0, t1);
    else if (general)
        nat_run<T, NAT_EDGE, TRACK>(ev, rv, cl, xch, oc4, up0, down0, wave, lane, nsweeps, live, smax,
                                    t0, t1);
    else
        nat_run<T, NAT_INNER, TRACK>(ev, rv, cl, xch, oc4, false, false, wave, lane, nsweeps, live, smax,
                                     t0, t1);
    if (Yw + NAT_R > g.ys0 && Yw < g.ys1) {
        const bool all_rows = Yw >= g.ys0 && Yw + NAT_R <= g.ys1;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (x0 + p < g.xs0 || x0 + p >= g.xs1) continue;
            auto store = [&](int k) {
                (eout + (size_t)(Yw + k) * w)[(unsigned)(x0 + p)] = ev[(k + p) & 1][k];
            };
            if (all_rows) {
#pragma unroll
                for (int k = 0; k < NAT_R; ++k) store(k);
            } else {
#pragma unroll
                for (int k = 0; k < NAT_R; ++k)
                    if (Yw + k >= g.ys0 && Yw + k < g.ys1) store(k);
            }
        }
    }
    if (TRACK) track_store<NAT_NW>(track, smax, red, tile, nsweeps, wave, lane);
    if (threadIdx.x == 0) st->cur = out_index;  // same value from every workgroup
}

// ---------------------------------------------------------------------------
// Temporally blocked red-black SOR (FP32, bricked layout, no holes).
//
// Regions as described in cd_sweeps.h, NW = 16 waves of R rows each, with the
// cells' right-hand side in registers beside them.  Up/down neighbours of a
// cell are the other colour in the rows above/below: registers of the same
// lane, except at a wave's first/last row, which comes through a small LDS
// exchange.  Left/right neighbours are the other colour in the same row: the
// same lane or the adjacent lane, fetched with a DPP wave shift folded into the
// first add.
//
// Residual rule: the right-hand side holds nq = -oc r per cell (oc = omega /
// cnt, cnt = in-grid neighbours; 0 outside the grid), and
//     v' = oc S + ((1 - omega) v + nq),   S = sum of the in-grid neighbours,
// which is v + oc (S - cnt v - r), the reference operator's SOR update
// (solver.cpp:29-47), in five VALU operations per cell (three adds, two FMAs).
// Cells outside the grid have oc = nq = 0 and value 0, and stay 0: they drop
// out of S by themselves.  Max-update rule (TRACK): the right-hand side holds r
// and the update oc (S - cnt v - r) is formed explicitly, as the stop test
// tracks it; a neighbour outside the grid contributes the cell's own value.
//
// What bounds it: dispatch, loads and stores take 4.7 us (R = 4) to 5.6 us
// (R = 8) of a launch whatever its sweeps; a half-sweep of one region per CU
// 0.14 to 0.27 us (0.13 / 0.27 us of it VALU issue of 16 full waves), a further
// region per CU 2.0 us (R = 4, 5 sweeps) to 6 us (R = 8, 8 sweeps), where VALU
// issue and memory phases of two resident workgroups overlap.  Two things cut
// the VALU work: waves whose rows have all become inexact sit out the rest of a
// launch (live_sweeps; a sixth of the work at R = 8, 16 sweeps), and border
// tiles, which every barrier waits for, have a code path per kind of border
// instead of selects per row.  Together 9.4 us for a launch of 14 sweeps at 400 x
// 400 (10.2 before), 18.3 for 15 tracked sweeps at 768 x 768 (21.1 before).  And
// what surrounds the sweeps was more scalar work than it looks: row addresses
// from the two bricks a wave's rows touch, one branch for all cells between inner
// and border tiles, stores grouped by column, no division, arguments read in one
// go (8.6 us, 17.2; 2048 x 2048 16.6 -> 15.3 for 9 sweeps).
//
// Taller regions lose less of their work to the halo, shorter ones
// have the faster half-sweep, more sweeps per launch spread the fixed part over
// a wider halo: blocked_plan weighs these.  Registers: 64 VGPRs (R = 8) keep two
// workgroups per CU; row and column kinds per wave instead of a factor per cell
// made room for that (102 VGPRs before, one workgroup per CU, 21.9 us for 8
// sweeps at 2048 x 2048 against 16.1).  Against those 16.1, when all waves still took
// every sweep and the set-up was longer, and not measured since: 8 waves of 16 rows
// 19.1 us, 12 of 8 18.1, 8 of 8 18.6, 4 of 16 23.6, 16 of 10 24.9.
// ---------------------------------------------------------------------------
// cache policy bits of the blocked kernel's stores
#ifndef CD_BK_STORE_POLICY
#define CD_BK_STORE_POLICY 16  // sc1: written through, not left dirty in L2
#endif

// What a wave's cells meet of the grid border, fixed per wave.  Columns: nothing;
// the left border in lane 0 or the right one in lane 63 (odd cell), or neither;
// a right border anywhere.  Rows: nothing; the wave's first row is the grid's
// first; its last row is the grid's last; its last row lies below the grid's
// last (odd heights); any.  The named rows cost nothing per sweep, a border
// anywhere a select per cell and row.
enum { COLS_IN = 0, COLS_LANES = 1, COLS_ANY = 2 };
enum { ROWS_IN = 0, ROWS_TOP = 1, ROWS_BOTTOM = 2, ROWS_BELOW = 3, ROWS_ANY = 4 };

// Per-lane facts of a region.  Index p: the lane's cell of column parity p.
struct BlockCells {
    float om4, c1;             // omega / 4, 1 - omega
    float oc[2], oc_end[2];    // omega / cnt in a row with both neighbour rows, with one
    bool miss_r[2];            // the cell has no right neighbour
    unsigned end_rows;         // bit k: row k of the wave has one neighbour row
    unsigned out_rows;         // bit k: row k lies outside the grid
    bool first, last;          // the wave's row 0 / R-1 has no row above / below it
};

// Rows K0 <= k < K1 of one half-sweep of colour C.  Only rows 0 and R-1 read
// up_row / down_row (the neighbouring waves' rows).  mx[p]: largest |update|.
//
// Every cell of the region is updated.  A cell at distance d from an inner
// region border takes stale neighbours, but after half-sweep s only cells at
// distance >= s are exact, and those read cells at distance >= s-1 only: the
// stale values never reach the stored cells (distance >= halo) and stay finite
// (each update is a bounded combination of finite values).
template <int C, int COLS, int ROWS, bool TRACK, int R, int K0, int K1>
__device__ __forceinline__ void blocked_half(float (&ev)[2][R], const float (&rv)[2][R],
                                             const BlockCells& g, unsigned end_rows,
                                             unsigned out_rows, float up_row, float down_row,
                                             float (&mx)[2]) {
#pragma unroll
    for (int k = K0; k < K1; ++k) {
        if (ROWS == ROWS_BELOW && k == R - 1) continue;  // below the grid: stays 0
        const int p = (k + C) & 1;  // column parity of colour-C cells in row k (R even)
        const float o = ev[1 - C][k];
        const float v = ev[C][k];
        const bool first = ROWS == ROWS_TOP && k == 0;
        const bool last = (ROWS == ROWS_BOTTOM && k == R - 1) || (ROWS == ROWS_BELOW && k == R - 2);
        // a neighbour row outside the grid
        float up = first ? (TRACK ? v : 0.f) : k > 0 ? ev[1 - C][k - 1] : up_row;
        float down = last ? (TRACK ? v : 0.f) : k < R - 1 ? ev[1 - C][k + 1] : down_row;
        float oc = first || last ? g.oc_end[p] : COLS == COLS_IN ? g.om4 : g.oc[p];
        if (ROWS == ROWS_ANY) {
            oc = (end_rows >> k) & 1u ? g.oc_end[p] : oc;
            oc = (out_rows >> k) & 1u ? 0.f : oc;
        }
        if (TRACK) {
            if (ROWS == ROWS_ANY) {
                if (k == 0) up = g.first ? v : up;
                // (row k is the last in the grid where row k + 1 is not in it)
                const bool below = k < R - 1 ? ((out_rows >> (k + 1)) & 1u) != 0 : g.last;
                down = below ? v : down;
            }
            float s;  // left + up + right
            if (COLS == COLS_IN) {
                s = (p ? o : lane_prev(o)) + up + (p ? lane_next(o) : o);
            } else if (p == 0) {
                s = add_prev(o, up, v) + (COLS == COLS_ANY && g.miss_r[0] ? v : o);
            } else if (COLS == COLS_LANES) {
                s = add_next(o, o + up, v);
            } else {
                const float right = lane_next(o);  // (in every lane, before the select)
                s = o + up + (g.miss_r[1] ? v : right);
            }
            const float t = __builtin_fmaf(-4.f, v, s + down) - rv[C][k];
            const float dl = oc * t;
            ev[C][k] = v + dl;
            mx[p] = fmaxf(mx[p], fabsf(dl));  // (0, or a NaN that fmaxf drops, where oc = 0)
        } else {
            const float sum = (p ? o : lane_prev(o)) + up + (p ? lane_next(o) : o) + down;
            ev[C][k] = __builtin_fmaf(oc, sum, __builtin_fmaf(g.c1, v, rv[C][k]));
        }
    }
}

template <int C, int COLS, int ROWS, bool TRACK, int R>
__device__ __forceinline__ void blocked_step(float (&ev)[2][R], const float (&rv)[2][R],
                                             float (*xch)[BK_NW][2][64], const BlockCells& g,
                                             int wave, int lane, float (&mx)[2]) {
    // publish this wave's first/last row of the colour the update reads
    xch[1 - C][wave][0][lane] = ev[1 - C][0];
    xch[1 - C][wave][1][lane] = ev[1 - C][R - 1];
    // the row kinds are re-read each half-sweep, so that the factors derived
    // from them are not kept in registers per row
    unsigned er = 0, ou = 0;
    if (ROWS == ROWS_ANY) {
        er = __builtin_amdgcn_readfirstlane(g.end_rows);
        ou = __builtin_amdgcn_readfirstlane(g.out_rows);
        asm volatile("" : "+s"(er), "+s"(ou));
    }
    // the inner rows need only this wave's registers: update them while the
    // other waves reach the barrier (the order of the updates of one colour
    // does not matter: they read only the other colour)
    blocked_half<C, COLS, ROWS, TRACK, R, 1, R - 1>(ev, rv, g, er, ou, 0.f, 0.f, mx);
    __syncthreads();
    float up_row = xch[1 - C][wave > 0 ? wave - 1 : 0][1][lane];
    float down_row = xch[1 - C][wave < BK_NW - 1 ? wave + 1 : BK_NW - 1][0][lane];
    if (ROWS == ROWS_ANY && !TRACK) {
        up_row = g.first ? 0.f : up_row;
        down_row = g.last ? 0.f : down_row;
    }
    blocked_half<C, COLS, ROWS, TRACK, R, 0, 1>(ev, rv, g, er, ou, up_row, down_row, mx);
    blocked_half<C, COLS, ROWS, TRACK, R, R - 1, R>(ev, rv, g, er, ou, up_row, down_row, mx);
}

// nsweeps sweeps of a region, of which the wave takes part in the first `live`.
// The waves of a workgroup may take this with different kinds of columns and
// rows: each executes the same number of barriers.
template <int COLS, int ROWS, bool TRACK, int R>
__device__ __forceinline__ void blocked_run(float (&ev)[2][R], const float (&rv)[2][R],
                                            float (*xch)[BK_NW][2][64], const BlockCells& g,
                                            int wave, int lane, int nsweeps, int live,
                                            float (*smax)[BK_NW][64], bool track0, bool track1) {
    const int mine = min(nsweeps, live);
    for (int j = 0; j < mine; ++j) {
        float mx[2] = {0.f, 0.f};
        blocked_step<0, COLS, ROWS, TRACK, R>(ev, rv, xch, g, wave, lane, mx);
        blocked_step<1, COLS, ROWS, TRACK, R>(ev, rv, xch, g, wave, lane, mx);
        if (TRACK) {
            smax[j][wave][lane] = fmaxf(track0 ? mx[0] : 0.f, track1 ? mx[1] : 0.f);
        }
    }
    for (int j = mine; j < nsweeps; ++j) {  // (no row of the wave counts for the maxima)
        __syncthreads();
        __syncthreads();
        if (TRACK) smax[j][wave][lane] = 0.f;
    }
}

// The wave's kinds (uniform) for its R rows from Yw on and the region's columns
// from X0 on.  Without tracking the columns beyond a border hold zeros wherever
// it lies.
template <int R, bool TRACK>
__device__ __forceinline__ int cols_kind(bool left, bool right, int X0, int w) {
    if (!left && !right) return COLS_IN;
    return !TRACK || !right || X0 + SW_RX == w ? COLS_LANES : COLS_ANY;
}
template <int R>
__device__ __forceinline__ int rows_kind(int Yw, int h) {
    if (Yw > 0 && Yw + R < h) return ROWS_IN;
    if (Yw + R < h) return ROWS_TOP;
    if (Yw > 0 && Yw + R == h) return ROWS_BOTTOM;
    return Yw > 0 && Yw + R == h + 1 ? ROWS_BELOW : ROWS_ANY;
}

// The intermediate-grid correction em (bricked, wm x hm, fm x fm fine cells
// per cell), which the learned iteration's first fine smoothing launch
// interpolates bilinearly at the fine cell centres as it loads its region.
struct MidGrid {
    const float* em;
    Brick bkm;
    int wm, hm, fm;
};

// The ends of a batch under the residual rule: its first launch starts from a
// zero correction (zero), its last one adds the correction to the iterate phi
// instead of storing it. A pass of its own that added the correction and
// cleared both buffers took 4.2 us and a launch gap at 400 x 400 (16.7 us at 2048 x
// 2048) before every check; 1.48 -> 1.45 ms for the 16 checks of a solve.
struct BatchEnds {
    double* phi;
    int zero;
};
// (an instantiation of its own: as run-time choices in every launch they cost the
// others 4 to 10 %)
enum { FORM_PLAIN = 0, FORM_PROLONG = 1, FORM_ENDS = 2 };

// Loads of one region: packed column `lane` of the wave's R rows, both colours,
// from the correction (or zero) and the right-hand side.  Columns are clamped
// into the grid; what rows outside it load is not used.
// PROLONG: the correction is the intermediate-grid correction interpolated
// bilinearly at the cell centres (u, v) = ((x, y) + 0.5) / fm - 0.5, not ein;
// the workgroup first stages the intermediate cells its region needs in
// `patch` (each is read by up to 4 fm^2 fine cells), with the intermediate
// grid's border clamping.  All waves of the workgroup must call it.
template <int R>
constexpr int kPatchMax = (SW_RX / 2 + 2) * (BK_NW * R / 2 + 2);  // fm >= 2
template <int R, bool PROLONG, typename RT>
__device__ __forceinline__ void region_load(float (&ev)[2][R], RT (&rr)[2][R], const float* ein,
                                            const RT* rhs, const Brick& bk, const MidGrid& mid,
                                            float* patch, int X0, int Y0, int w, int h, int wave,
                                            int lane, bool zero) {
    const int Yw = Y0 + R * wave;
    const int j = min(X0 / 2 + lane, (w + 1) / 2 - 1);
    const unsigned col = brick_col(j);
    const BrickRows br = brick_rows(bk, Yw, h);
    const __amdgpu_buffer_rsrc_t e_rs[2] = {plane_rsrc(ein, bk.plane * sizeof(float)),
                                            plane_rsrc(ein + bk.plane, bk.plane * sizeof(float))};
    const __amdgpu_buffer_rsrc_t r_rs[2] = {plane_rsrc(rhs, bk.plane * sizeof(RT)),
                                            plane_rsrc(rhs + bk.plane, bk.plane * sizeof(RT))};
    int pi0[2] = {0, 0}, pj0 = 0, pw = 0;
    float ptu[2] = {0.f, 0.f};
    const float inv = PROLONG ? 1.f / mid.fm : 0.f;
    if (PROLONG) {
        // intermediate cells I0..I1 x J0..J1 cover the region's (clamped) cells
        const int xa = min(X0, w - 1), xb = min(X0 + SW_RX - 1, w - 1);
        const int ya = min(Y0, h - 1), yb = min(Y0 + BK_NW * R - 1, h - 1);
        const int I0 = (int)floorf((xa + 0.5f) * inv - 0.5f);
        const int I1 = (int)floorf((xb + 0.5f) * inv - 0.5f) + 1;
        pj0 = (int)floorf((ya + 0.5f) * inv - 0.5f);
        const int J1 = (int)floorf((yb + 0.5f) * inv - 0.5f) + 1;
        pw = I1 - I0 + 1;
        const int n = pw * (J1 - pj0 + 1);
        for (int q = threadIdx.x; q < n; q += BK_THREADS) {
            const int pr = q / pw, pc = q - pr * pw;
            patch[q] = mid.em[brick_at(mid.bkm, min(max(I0 + pc, 0), mid.wm - 1),
                                       min(max(pj0 + pr, 0), mid.hm - 1))];
        }
        // the lane's two cells 2j + t (t = 0, 1): the same columns in every row
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int xx = min(2 * j + t, w - 1);
            const float u = (xx + 0.5f) * inv - 0.5f;
            const int i0 = (int)floorf(u);
            ptu[t] = u - i0;
            pi0[t] = i0 - I0;
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
        int r0 = 0;
        float tv = 0.f;
        const int Yc = min(Yw + k, h - 1);
        if (PROLONG) {
            const float v = (Yc + 0.5f) * inv - 0.5f;
            const int j0 = (int)floorf(v);
            tv = v - j0;
            r0 = (j0 - pj0) * pw;
        }
        const unsigned row = br.at(k) - 64u * k;  // (64 k goes into the instruction)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (PROLONG) {
                const int t = (c + Yc) & 1;
                const float tu = ptu[t];
                const float* pp = patch + r0 + pi0[t];
                const float a = pp[0], b = pp[1], cc = pp[pw], d = pp[pw + 1];
                ev[c][k] = (a * (1.f - tu) + b * tu) * (1.f - tv) + (cc * (1.f - tu) + d * tu) * tv;
            } else {
                ev[c][k] = 0.f;
                if (!zero) ev[c][k] = buf_load<float>(e_rs[c], (col + 64u * k) * 4u, row * 4u);
            }
            rr[c][k] = buf_load<RT>(r_rs[c], (col + 64u * k) * (unsigned)sizeof(RT),
                                    row * (unsigned)sizeof(RT));
        }
    }
}

// The right-hand side is BF16 under the residual rule (every FP64 check
// re-rounds the current residual, so the rounding never reaches the result)
// and FP32 under the max-update rule (TRACK), which cannot see the smooth
// error a rounded right-hand side leaves behind.  FORM_PROLONG: the
// sweeps start from `mid` interpolated at the cells instead of from ein;
// FORM_ENDS: as `ends` says.
// (Registers for two workgroups per CU, but for tracking at 8 rows, which would
// spill; an interpolating launch at 8 rows spills two and still takes a learned
// iteration at 2048 x 2048 from 148 to 145 us.)
template <int R, bool TRACK, int FORM>
__global__ __launch_bounds__(BK_THREADS, TRACK && R > 6 ? 4 : 8) void k_rb_blocked(
    const float* ein, float* eout, const void* __restrict__ rhs, Brick bk, SweepTiles tiles,
    int nsweeps, float om2, float om3, float om4, const float* __restrict__ rmean, SolveDev* st,
    int out_index, MidGrid mid, TrackArgs track, BatchEnds ends) {
    static_assert(R % 2 == 0, "colours alternate by row");
    constexpr bool PROLONG = FORM == FORM_PROLONG, ENDS = FORM == FORM_ENDS;
    __shared__ float xch[2][BK_NW][2][64];
    __shared__ float smax[TRACK ? kTrackSweeps : 1][BK_NW][64];
    __shared__ unsigned red[TRACK ? BK_NW : 1];
    __shared__ float patch[PROLONG ? kPatchMax<R> : 1];
    // What the loads' addresses need is read in one go, and nothing else comes
    // before them (400 x 400: 8.9 -> 8.6 us a launch); not where that spills
    // scalars into the few vector registers left (3 % slower there).
    constexpr bool kLoadsFirst = !TRACK || R > 6;
    if (kLoadsFirst)
        asm volatile("" ::"s"(ein), "s"(rhs), "s"(rmean), "s"(bk.nbx), "s"(bk.plane),
                     "s"(tiles.ntiles), "s"(tiles.inv_x), "s"(tiles.ix));
    const int tile = tile_of_block(tiles.ntiles);
    if (tile >= tiles.ntiles) return;
    const Region rg = region_of(tiles, tile);
    const int w = tiles.w, h = tiles.h;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    using RT = typename std::conditional<TRACK, float, unsigned short>::type;
    const RT* r = static_cast<const RT*>(rhs);
    float ev[2][R], rv[2][R];
    RT rr[2][R];
    const unsigned words = TRACK ? track_load<BK_NW>(track, tiles.ntiles) : 0u;
    region_load<R, PROLONG>(ev, rr, ein, r, bk, mid, patch, rg.X0, rg.Y0, w, h, wave, lane,
                            ENDS && ends.zero);
    if (kLoadsFirst) __builtin_amdgcn_sched_barrier(0);
    // Max-update rule: the solve can have stopped in an earlier launch of the
    // batch, and then leaves the buffers untouched.  Residual rule: only a check
    // stops it, and no sweeps are enqueued after that.
    if (TRACK) {
        const TrackPlan plan =
            track_decide<BK_NW>(track, st, tiles.ntiles, nsweeps, words, red);
        if (plan.nsweeps == 0) return;
        nsweeps = __builtin_amdgcn_readfirstlane(plan.nsweeps);
        if (plan.redo) {
            out_index ^= 1;
            region_load<R, PROLONG>(ev, rr, eout, r, bk, mid, patch, rg.X0, rg.Y0, w, h, wave,
                                    lane, false);
            eout = const_cast<float*>(ein);
        }
    }
    const float rm = *rmean;

    const int Yw = rg.Y0 + R * wave, x0 = rg.X0 + 2 * lane;
    BlockCells g;
    g.om4 = om4;
    g.c1 = 1.f - 4.f * om4;
    g.first = Yw == 0;
    g.last = Yw + R >= h;
    g.end_rows = 0u;
    g.out_rows = 0u;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        if (Yw + k == 0 || Yw + k == h - 1) g.end_rows |= 1u << k;
        if (Yw + k >= h) g.out_rows |= 1u << k;
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const bool in = x0 + p < w;
        const bool side = x0 + p == 0 || x0 + p == w - 1;
        g.miss_r[p] = x0 + p >= w - 1;
        g.oc[p] = in ? (side ? om3 : om4) : 0.f;
        g.oc_end[p] = in ? (side ? om2 : om3) : 0.f;
    }
    const int cols = cols_kind<R, TRACK>(rg.left, rg.right, rg.X0, w), rows = rows_kind<R>(Yw, h);
    // the cells whose updates count for the stop rule: those at distance >= halo
    // from the region's inner borders (all exact; two tiles may count one)
    bool t0 = false, t1 = false;
    if (TRACK) {
        const int hl = tiles.halo, dy0 = R * wave;  // halo is a multiple of R
        const bool rows_ok = (rg.top || dy0 >= hl) && (rg.bottom || dy0 + R <= BK_NW * R - hl);
        auto col_ok = [&](int dx) {
            return rows_ok && (rg.left || dx >= hl) && (rg.right || dx < SW_RX - hl);
        };
        t0 = col_ok(2 * lane);
        t1 = col_ok(2 * lane + 1);
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const float rc = rhs_to_f32(rr[c][k]);
            rv[c][k] = TRACK ? rc - rm : rm - rc;
        }
    int kind = cols == COLS_IN && rows == ROWS_IN ? -1
               : cols == COLS_ANY ? (int)ROWS_ANY : rows;
    // (one branch for all cells, kept apart from the choice of the sweeps' path)
    if (kind >= 0) {
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int p = (k + c) & 1;
                const bool out = (g.out_rows >> k) & 1u;
                const float oc = out ? 0.f : (g.end_rows >> k) & 1u ? g.oc_end[p] : g.oc[p];
                const bool in = !out && x0 + p < w;
                ev[c][k] = in ? ev[c][k] : 0.f;
                rv[c][k] = !TRACK ? rv[c][k] * oc : in ? rv[c][k] : 0.f;
            }
    } else if (!TRACK) {
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int c = 0; c < 2; ++c) rv[c][k] *= g.om4;
    }
    kind = __builtin_amdgcn_readfirstlane(kind);
    asm volatile("" : "+s"(kind));
    const int live = live_sweeps<R, BK_NW>(rg, wave);
#define RUN(COLS, ROWS) blocked_run<COLS, ROWS, TRACK, R>(ev, rv, xch, g, wave, lane, nsweeps, live, smax, t0, t1)
    if (kind < 0) RUN(COLS_IN, ROWS_IN);
    else if (kind == ROWS_IN) RUN(COLS_LANES, ROWS_IN);
    else if (kind == ROWS_TOP) RUN(COLS_LANES, ROWS_TOP);
    else if (kind == ROWS_BOTTOM) RUN(COLS_LANES, ROWS_BOTTOM);
    else if (kind == ROWS_BELOW) RUN(COLS_LANES, ROWS_BELOW);
    else RUN(COLS_ANY, ROWS_ANY);
#undef RUN
    // store: the lane's two columns, each with the wave's rows of the region
    const unsigned col = brick_col(min(rg.X0 / 2 + lane, (w + 1) / 2 - 1));
    const BrickRows br = brick_rows(bk, Yw, h);
    const __amdgpu_buffer_rsrc_t out_rs[2] = {plane_rsrc(eout, bk.plane * sizeof(float)),
                                              plane_rsrc(eout + bk.plane, bk.plane * sizeof(float))};
    const bool all_rows = Yw >= rg.ys0 && Yw + R <= rg.ys1;
    if (ENDS && ends.phi && Yw + R > rg.ys0 && Yw < rg.ys1) {
        // the end of a batch: phi += e (all loads first, from clamped addresses)
        double ph[2][R];
        const unsigned xc[2] = {(unsigned)min(max(x0, rg.xs0), rg.xs1 - 1),
                                (unsigned)min(max(x0 + 1, rg.xs0), rg.xs1 - 1)};
        auto prow = [&](int k) {
            return ends.phi + (size_t)min(max(Yw + k, rg.ys0), rg.ys1 - 1) * w;
        };
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int p = 0; p < 2; ++p) ph[p][k] = prow(k)[xc[p]];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (x0 + p < rg.xs0 || x0 + p >= rg.xs1) continue;
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (Yw + k >= rg.ys0 && Yw + k < rg.ys1)
                    prow(k)[xc[p]] = ph[p][k] + (double)ev[(k + p) & 1][k];
        }
    } else if (Yw + R > rg.ys0 && Yw < rg.ys1) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (x0 + p < rg.xs0 || x0 + p >= rg.xs1) continue;
            auto store = [&](int k) {
                __builtin_amdgcn_raw_buffer_store_b32(
                    __float_as_uint(ev[(k + p) & 1][k]), out_rs[(k + p) & 1], (col + 64u * k) * 4u,
                    (br.at(k) - 64u * k) * 4u, CD_BK_STORE_POLICY);
            };
            if (all_rows) {
#pragma unroll
                for (int k = 0; k < R; ++k) store(k);
            } else {
#pragma unroll
                for (int k = 0; k < R; ++k)
                    if (Yw + k >= rg.ys0 && Yw + k < rg.ys1) store(k);
            }
        }
    }
    if (TRACK) track_store<BK_NW>(track, smax, red, tile, nsweeps, wave, lane);
    if (threadIdx.x == 0) st->cur = out_index;  // same value from every workgroup
}

// ---------------------------------------------------------------------------
// A whole mixed-precision solve of a grid of one region (up to 128 x 128 cells)
// in one launch of one workgroup: the iterate phi, the correction and the
// right-hand side stay in registers; sweeps, checks and the choice of the next
// batch are those of cd_solve_device_internal's loop, with the same operations and
// reductions.  Such a solve was bound by its checks, each three launches and a
// round trip to the host for 10 us of sweeps: 64 x 64 to 1e-6 took 665 us (490
// with launches of a whole batch), 13 checks of about 35 us.  Now 0.36 us a
// sweep, 5.5 us a check (4.8 with sums in an order of its own) and 43 us for the
// launch with its first and last check.
//
// The kernel leaves phi alone and reports `holes` when b holds a NaN, and
// returns at a check after kRegionSweeps sweeps (the host launches it again).
// ---------------------------------------------------------------------------
struct RegionArgs {
    int w, h, max_sweeps, kmax, adaptive, check_holes, resume;
    unsigned seq;
    float om2, om3, om4;
    double tol, margin;
};

// Sums over the grid in the order of the launches that a larger grid's solve
// takes (k_rhs_moments and k_residual with k_rhs_finish and k_check): a tree over
// the 64 cells of a row of a 64 x 4 tile, the tile's rows as (0 + 2) + (1 + 3), a
// tree over the up to 64 tiles.  So the sums, and the solve, have the bits of
// that route.  A lane holds two neighbouring cells of a row, so the tree's steps
// over columns 32, 16, ... 2 apart are steps over lanes 16, 8, ... 1 apart and the
// last one joins the lane's two cells.
//
// fold: M sums at once, M a power of two: at each step a lane passes on the sums
// it will not finish, so that M sums take M - 1 exchanges.  Takes the steps from
// lane distance O on down, log2(M) of them; lane bit O >> j then says which half
// of the sums' index bit j was kept.
template <int O, int M>
__device__ __forceinline__ double fold(const double (&a)[M], int lane) {
    if constexpr (M == 1) {
        return a[0];
    } else {
        double h[M / 2];
        const bool upper = (lane & O) != 0;
#pragma unroll
        for (int i = 0; i < M / 2; ++i) {
            const double keep = upper ? a[2 * i + 1] : a[2 * i];
            const double pass = upper ? a[2 * i] : a[2 * i + 1];
            h[i] = keep + __shfl_xor(pass, O, 64);
        }
        return fold<O / 2, M / 2>(h, lane);
    }
}
constexpr int log2_of(int n) { return n > 1 ? 1 + log2_of(n / 2) : 0; }

// N grid sums of R rows per wave: take(), with each pair of rows, then finish().
// rows: LDS for the row sums of both column halves.
template <int R, int N>
struct GridSum {
    static constexpr int kFirst = log2_of(4 * N);       // steps of take
    static constexpr int kPairs = log2_of(R / 2);       // steps over the pairs
    double g[R / 2];
    // v[r][p][i]: value i of the cell of column parity p in row 2 pair + r
    __device__ __forceinline__ void take(int pair, const double (&v)[2][2][N], int lane) {
        double a[4 * N];
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int i = 0; i < N; ++i) a[r + 2 * i + 2 * N * p] = v[r][p][i];
        g[pair] = fold<16>(a, lane);
    }
    __device__ __forceinline__ void finish(double (&out)[N], double (*rows)[2][R * BK_NW], int w,
                                           int h, int wave, int lane) {
        double t = fold<(16 >> kFirst)>(g, lane);
#pragma unroll
        for (int o = 16 >> (kFirst + kPairs); o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
        t += __shfl_xor(t, 16 >> (kFirst - 1), 64);  // the two cells of a lane
        // this lane's sum: index bits from lane bits 16, 8, ...
        auto bit = [&](int j) { return (lane >> (4 - j)) & 1; };
        int pair = 0;
#pragma unroll
        for (int j = 0; j < kPairs; ++j) pair |= bit(kFirst + j) << j;
        const int i = N > 1 ? bit(1) : 0;
        __syncthreads();  // rows has been read
        rows[i][lane >> 5][R * wave + 2 * pair + bit(0)] = t;
        __syncthreads();
        const int nbx = w > 64 ? 2 : 1, bx = lane & (nbx - 1), y = 4 * (lane / nbx);
#pragma unroll
        for (int n = 0; n < N; ++n) {
            double q = 0.0;
            if (y < h && y < R * BK_NW)
                q = (rows[n][bx][y] + rows[n][bx][y + 2]) + (rows[n][bx][y + 1] + rows[n][bx][y + 3]);
            out[n] = cd_wave_sum(q);
        }
    }
};

template <int R, bool TRACK>
__global__ __launch_bounds__(BK_THREADS) void k_solve_region(const double* __restrict__ b,
                                                             double* __restrict__ phi,
                                                             RegionArgs a, SolveDev* st,
                                                             SolveDev* host_st) {
    __shared__ float xch[2][BK_NW][2][64];
    __shared__ double xphi[BK_NW][2][2][64];
    __shared__ double rowsum[2][2][R * BK_NW];
    __shared__ float smax[TRACK ? kStopGroup : 1][BK_NW][64];
    __shared__ float redm[kStopGroup];
    const int w = a.w, h = a.h;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int Yw = R * wave, x0 = 2 * lane;
    auto in_grid = [&](int c, int k) { return x0 + ((k + c) & 1) < w && Yw + k < h; };
    // clamped cell addresses: a uniform row and one of two lane offsets
    const unsigned col[2] = {(unsigned)min(x0, w - 1), (unsigned)min(x0 + 1, w - 1)};
    auto row = [&](int k) { return (unsigned)(min(Yw + k, h - 1) * w); };
    const double count = (double)w * h;

    // right-hand side statistics (k_rhs_moments)
    double bmean, bnorm, holes;
    {
        double bv[2][R], s[2], q[1];
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int c = 0; c < 2; ++c) bv[c][k] = (b + row(k))[col[(k + c) & 1]];
        GridSum<R, 2> sums;
        GridSum<R, 1> squares;
#pragma unroll
        for (int k = 0; k < R; k += 2) {
            double v[2][2][2];
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const int c = (k + r + p) & 1;
                    const double x = bv[c][k + r];
                    const bool hole = in_grid(c, k + r) && isnan(x);
                    v[r][p][0] = in_grid(c, k + r) && !hole ? x : 0.0;
                    v[r][p][1] = hole ? 1.0 : 0.0;
                }
            sums.take(k / 2, v, lane);
        }
        sums.finish(s, rowsum, w, h, wave, lane);
        bmean = s[0] / count;
        holes = s[1];
#pragma unroll
        for (int k = 0; k < R; k += 2) {
            double v[2][2][1];
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const int c = (k + r + p) & 1;
                    const double d = bv[c][k + r] - bmean;
                    v[r][p][0] = in_grid(c, k + r) && !isnan(bv[c][k + r]) ? d * d : 0.0;
                }
            squares.take(k / 2, v, lane);
        }
        squares.finish(q, rowsum, w, h, wave, lane);
        bnorm = sqrt(q[0]);
    }

    BlockCells g;
    g.om4 = a.om4;
    g.c1 = 1.f - 4.f * a.om4;
    g.first = Yw == 0;
    g.last = Yw + R >= h;
    g.end_rows = 0u;
    g.out_rows = 0u;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        if (Yw + k == 0 || Yw + k == h - 1) g.end_rows |= 1u << k;
        if (Yw + k >= h) g.out_rows |= 1u << k;
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const bool in = x0 + p < w;
        const bool side = x0 + p == 0 || x0 + p == w - 1;
        g.miss_r[p] = x0 + p >= w - 1;
        g.oc[p] = in ? (side ? a.om3 : a.om4) : 0.f;
        g.oc_end[p] = in ? (side ? a.om2 : a.om3) : 0.f;
    }
    const int rows = rows_kind<R>(Yw, h);  // (uniform over the wave)

    double ph[2][R];
    float ev[2][R], rv[2][R];
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const double v = (phi + row(k))[col[(k + c) & 1]];
            ph[c][k] = in_grid(c, k) ? v : 0.0;
            ev[c][k] = 0.f;
        }

    // FP64 check of phi + e (k_flush_packed, k_residual, k_check): folds e, leaves
    // the sweeps' right-hand side in rv; returns the relative residual
    double rnorm = 0.0, rsum = 0.0;
    float rm = 0.f;
    auto check = [&]() -> double {
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                ph[c][k] += (double)ev[c][k];
                ev[c][k] = 0.f;
            }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            xphi[wave][c][0][lane] = ph[c][0];
            xphi[wave][c][1][lane] = ph[c][R - 1];
        }
        __syncthreads();
        double s[2];
        GridSum<R, 2> sums;
#pragma unroll
        for (int kp = 0; kp < R; kp += 2) {
            double vv[2][2][2];
#pragma unroll
            for (int rc = 0; rc < 4; ++rc) {
                const int k = kp + (rc >> 1), c = rc & 1;
                const int p = (k + c) & 1, x = x0 + p, y = Yw + k;
                const double o = ph[1 - c][k];
                double up = k > 0 ? ph[1 - c][k > 0 ? k - 1 : 0]
                                  : xphi[wave > 0 ? wave - 1 : 0][1 - c][1][lane];
                double down = k < R - 1 ? ph[1 - c][k < R - 1 ? k + 1 : 0]
                                        : xphi[wave < BK_NW - 1 ? wave + 1 : 0][1 - c][0][lane];
                if (k == 0 && g.first) up = 0.0;
                if (k == R - 1 && g.last) down = 0.0;
                const double left = p ? o : lane_prev(o), right = p ? lane_next(o) : o;
                const double cnt = (double)((x > 0) + (y > 0) + (x < w - 1) + (y < h - 1));
                double v = ((b + row(k))[col[p]] - bmean) -
                           ((left + up + right + down) - cnt * ph[c][k]);
                if (!in_grid(c, k)) v = 0.0;
                vv[rc >> 1][p][0] = v;
                vv[rc >> 1][p][1] = v * v;
                rv[c][k] = TRACK ? (float)v : bf16_to_f32(f32_to_bf16((float)v));
            }
            sums.take(kp / 2, vv, lane);
        }
        sums.finish(s, rowsum, w, h, wave, lane);
        const double mean = s[0] / count, rn2 = s[1] - count * mean * mean;
        rsum = s[0];
        rnorm = rn2 > 0.0 ? sqrt(rn2) : (rn2 == rn2 ? 0.0 : rn2);
        rm = (float)mean;
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int p = (k + c) & 1;
                const bool out = (g.out_rows >> k) & 1u;
                const float oc = out ? 0.f : (g.end_rows >> k) & 1u ? g.oc_end[p] : g.oc[p];
                if (TRACK) rv[c][k] = in_grid(c, k) ? rv[c][k] - rm : 0.f;
                else rv[c][k] = (rm - rv[c][k]) * oc;
            }
        return bnorm > 0 ? rnorm / bnorm : (rnorm > 0 ? INFINITY : 0.0);
    };
    auto sweep = [&](int n) {
        n = __builtin_amdgcn_readfirstlane(n);  // (the same in every thread)
#define RUN(ROWS) blocked_run<COLS_ANY, ROWS, TRACK, R>(ev, rv, xch, g, wave, lane, n, INT_MAX, smax, true, true)
        if (rows == ROWS_IN) RUN(ROWS_IN);
        else if (rows == ROWS_TOP) RUN(ROWS_TOP);
        else if (rows == ROWS_BOTTOM) RUN(ROWS_BOTTOM);
        else RUN(ROWS_ANY);
#undef RUN
    };
    // the first of n <= kStopGroup sweeps whose largest update is below tol
    double last_max = a.resume ? st->last_max_update : INFINITY;
    auto stopped = [&](int n) -> bool {
        __syncthreads();
        if (wave < n) {  // one wave per sweep
            float m = 0.f;
            for (int v = 0; v < BK_NW; ++v) m = fmaxf(m, smax[wave][v][lane]);
            m = wave_max_pos(m);
            if (lane == 0) redm[wave] = m;
        }
        __syncthreads();  // (also: smax has been read)
        for (int j = 0; j < n; ++j) {
            last_max = (double)redm[j];
            if (last_max < a.tol) return true;
        }
        return false;
    };

    // the solve (cd_solve_device_internal's loop), resumed where it was left
    const bool resume = a.resume != 0;
    int cum = resume ? st->cum : 0, checks = resume ? st->checks : 0;
    int k = resume ? st->batch : a.adaptive ? min(a.kmax, max(8, a.kmax / 4)) : a.kmax;
    int at_done = resume ? st->sweeps_at_done : -1;
    bool confirming = resume && st->confirming, done = false, more = false;
    double rel = INFINITY, rel0 = resume ? st->rel0 : INFINITY, prev = 0.0;
    const bool valid = !(a.check_holes && holes > 0.0);
    if (valid) {
        rel = check();
        if (!resume) {
            rel0 = rel;
            ++checks;
            done = !TRACK && rel <= a.tol;
        }
        prev = rel;
        const int until = cum > INT_MAX - kRegionSweeps ? INT_MAX : cum + kRegionSweeps;
        // (a non-finite first residual still takes one batch, as the launches do)
        while (!done && cum < a.max_sweeps) {
            if (cum >= until) { more = true; break; }
            const int nsw = min(confirming ? kStopGroup : k, a.max_sweeps - cum);
            if (!TRACK) {
                sweep(nsw);
            } else {
                for (int j = 0; j < nsw && !done; j += kStopGroup) {
                    const int n = min(kStopGroup, nsw - j);
                    sweep(n);
                    if (stopped(n)) {
                        done = true;
                        at_done = cum + j + n;
                    }
                }
            }
            cum += nsw;
            rel = check();
            ++checks;
            if (!TRACK) done = rel <= a.tol;
            if (!isfinite(rel)) break;
            if (TRACK) {
                if (done && !confirming && cum < a.max_sweeps) {
                    confirming = true;
                    done = false;
                    at_done = -1;
                    continue;
                }
                confirming = false;
            }
            if (a.adaptive && !done) {
                // geometric rate over the last batch, rho = (rel / prev)^(1 / nsw)
                const double lr = prev > 0 && rel > 0 && rel < prev ? log(rel / prev) / nsw : 0.0;
                int want = a.kmax;
                if (lr < -1.0000005000003333e-6) {  // rho < 0.999999
                    // (out of int's range, as for a tolerance of 0: the fewest)
                    const double need = ceil(log(a.tol / rel) / lr * a.margin) + 2.0;
                    want = fabs(need) < 2147483647.0 ? (int)need : 0;
                }
                k = max(8, min(a.kmax, want));
                prev = rel;
            }
        }
#pragma unroll
        for (int kk = 0; kk < R; ++kk)
#pragma unroll
            for (int c = 0; c < 2; ++c)
                if (in_grid(c, kk)) (phi + row(kk))[col[(kk + c) & 1]] = ph[c][kk];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        SolveDev o{};
        o.holes = valid ? 0 : (int)holes;
        o.done = done;
        o.done_check = done ? checks - 1 : -1;
        o.stop_lid = INT_MAX;
        o.bsum = bmean * count;
        o.sweeps_at_done = at_done;
        o.checks = checks;
        o.bmean = bmean;
        o.bnorm = bnorm;
        o.rsum = rsum;
        o.rnorm = rnorm;
        o.rel = rel;
        o.rel0 = rel0;
        o.last_max_update = last_max;
        o.rmean32 = rm;
        o.cum = cum;
        o.batch = k;
        o.confirming = confirming;
        o.more = more;
        o.seq = a.seq;
        *st = o;
        // the host waits for the sequence word, which goes last
        const unsigned* src = reinterpret_cast<const unsigned*>(&o);
        unsigned* dst = reinterpret_cast<unsigned*>(host_st);
        constexpr int kSeq = (int)(offsetof(SolveDev, seq) / 4);
        for (int i = 0; i < (int)(sizeof(SolveDev) / 4); ++i)
            if (i != kSeq) dst[i] = src[i];
        __hip_atomic_store(dst + kSeq, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Reopen a solve whose max-update stop is to be confirmed on a fresh
// right-hand side (the sweeps that stopped it read r rounded at the last check).
__global__ void k_reopen(SolveDev* st) {
    if (threadIdx.x != 0) return;
    st->done = 0;
    st->stop_lid = INT_MAX;
    st->sweeps_at_done = -1;
}

__global__ void k_set_holes_nan(double* __restrict__ phi, const uint8_t* __restrict__ mask,
                                size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && (mask[i] & M_HOLE)) phi[i] = NAN;
}

template <int R>
void launch_blocked_rows(bool track, const MidGrid* pro, dim3 grid, hipStream_t s,
                         const float* ein, float* eout, const void* rhs, const Brick& bk,
                         const SweepTiles& t, int nsweeps, float om2, float om3, float om4,
                         const float* rmean, SolveDev* st, int out_index, const TrackArgs& tr,
                         const BatchEnds& ends) {
    const dim3 blk(BK_THREADS);
    const MidGrid mid = pro ? *pro : MidGrid{};
    if (track)
        hipLaunchKernelGGL((k_rb_blocked<R, true, FORM_PLAIN>), grid, blk, 0, s, ein, eout, rhs, bk, t,
                           nsweeps, om2, om3, om4, rmean, st, out_index, mid, tr, ends);
    else if (pro)
        hipLaunchKernelGGL((k_rb_blocked<R, false, FORM_PROLONG>), grid, blk, 0, s, ein, eout, rhs, bk, t,
                           nsweeps, om2, om3, om4, rmean, st, out_index, mid, tr, ends);
    else if (ends.phi || ends.zero)
        hipLaunchKernelGGL((k_rb_blocked<R, false, FORM_ENDS>), grid, blk, 0, s, ein, eout, rhs, bk, t,
                           nsweeps, om2, om3, om4, rmean, st, out_index, mid, tr, ends);
    else
        hipLaunchKernelGGL((k_rb_blocked<R, false, FORM_PLAIN>), grid, blk, 0, s, ein, eout, rhs, bk, t,
                           nsweeps, om2, om3, om4, rmean, st, out_index, mid, tr, ends);
}

// one launch of nsweeps sweeps from ein to eout
void launch_blocked(const BlockedPlan& pl, bool track, const MidGrid* pro, hipStream_t s,
                    const float* ein, float* eout, const void* rhs, const Brick& bk, int nsweeps,
                    float om2, float om3, float om4, const float* rmean, SolveDev* st,
                    int out_index, const TrackArgs& tr, const BatchEnds& ends = BatchEnds{}) {
    const dim3 grid(sweep_grid(pl.t.ntiles));
    switch (pl.rows) {
    case 4: launch_blocked_rows<4>(track, pro, grid, s, ein, eout, rhs, bk, pl.t, nsweeps, om2, om3, om4, rmean, st, out_index, tr, ends); break;
    case 6: launch_blocked_rows<6>(track, pro, grid, s, ein, eout, rhs, bk, pl.t, nsweeps, om2, om3, om4, rmean, st, out_index, tr, ends); break;
    default: launch_blocked_rows<8>(track, pro, grid, s, ein, eout, rhs, bk, pl.t, nsweeps, om2, om3, om4, rmean, st, out_index, tr, ends); break;
    }
}

// Over-relaxation factor.  > 0: as given.  < 0: the reference's
// 2/(1+3.14159265/width) (solver.cpp:71).  == 0: the optimum for this
// operator: the Jacobi iteration I + A/4 has spectral radius
// rho_J = 1 - sin^2(pi/(2n)) on the zero-mean subspace (n = larger side), and
// red-black ordering is consistent, so omega = 2/(1 + sqrt(1 - rho_J^2)).
double cd_sor_omega(double requested, int w, int h) {
    if (requested > 0) return requested;
    if (requested < 0) return 2.0 / (1.0 + 3.14159265 / w);
    const int n = std::max(w, h);
    const double s = std::sin(M_PI / (2.0 * n));
    const double rj = 1.0 - s * s;
    return 2.0 / (1.0 + std::sqrt(1.0 - rj * rj));
}

// the next check of an adaptive solve comes after this multiple of the sweeps
// the observed contraction rate predicts (0.9 to 1.5 measured no better on the
// 2048^2 and 1024^2 designs: a check also restarts the FP32 correction, so
// where the checks fall moves the sweep count by a few per cent either way)
#ifndef CD_CHECK_MARGIN
#define CD_CHECK_MARGIN 1.05
#endif

int auto_check_every(int w, int h) {
    // SOR with omega near 2 contracts every mode by ~(1 - 2*pi/n) per sweep.
    // The FP32 correction loses accuracy once it has absorbed a ~10x residual
    // reduction, which takes ~ n*ln(10)/(2*pi) sweeps.
    int n = std::max(w, h);
    int k = (int)std::lround(0.36 * n);
    return std::max(8, std::min(k, 2048));
}


// ---------------------------------------------------------------------------
// Learned correction and training-pair capture (no hole mask, positional
// Neumann counts).  Coarse cell (I,J) averages the f x f fine cells
// [f*I, f*I+f) x [f*J, f*J+f).
// ---------------------------------------------------------------------------
// coarse residual rc = block mean of the projected BF16 residual the blocked
// sweeps see (r16 - rmean32).  f < 8: one thread per coarse cell; larger f:
// one wave per coarse cell (lanes stride over its f^2 fine cells, fixed-order
// shuffle tree).  Statistics of rc follow in k_coarse_stats.
// x8 (may be NULL): rc also written as the input of a linear network, BF16
// channel 0 of 8 (a linear bias-free network commutes with the scaling that
// normalises its input, so that input needs no statistics)
__global__ __launch_bounds__(256) void k_restrict_r16(const unsigned short* __restrict__ r16,
                                                      Brick bk, const SolveDev* __restrict__ st,
                                                      int f, int wc, int hc,
                                                      float* __restrict__ rc,
                                                      unsigned short* __restrict__ x8) {
    const float rm = st->rmean32;
    const int ff = f * f;
    if (f < 8) {
        const int i = blockIdx.x * blockDim.x + threadIdx.x;
        if (i >= wc * hc) return;
        const int J = i / wc, I = i - J * wc;
        float acc = 0.f;
        for (int yy = J * f; yy < J * f + f; ++yy)
            for (int xx = I * f; xx < I * f + f; ++xx)
                acc += bf16_to_f32(r16[brick_at(bk, xx, yy)]) - rm;
        rc[i] = acc / (float)ff;
        if (x8) *reinterpret_cast<uint4*>(x8 + (size_t)i * 8) =
            make_uint4(f32_to_bf16(acc / (float)ff), 0, 0, 0);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (i >= wc * hc) return;  // whole wave
    const int J = i / wc, I = i - J * wc;
    float acc = 0.f;
    for (int k = lane; k < ff; k += 64) {
        const int dy = k / f, dx = k - dy * f;
        acc += bf16_to_f32(r16[brick_at(bk, I * f + dx, J * f + dy)]) - rm;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (lane == 0) {
        rc[i] = acc / (float)ff;
        if (x8) *reinterpret_cast<uint4*>(x8 + (size_t)i * 8) =
            make_uint4(f32_to_bf16(acc / (float)ff), 0, 0, 0);
    }
}

// (mean, rms) of nc coarse values from stats = (sum, sum^2), as every consumer
// of stats computes them
__device__ __forceinline__ void coarse_derived(const double* stats, int nc, double* derived) {
    const double mean = stats[0] / nc;
    const double var = stats[1] / nc - mean * mean;
    derived[0] = mean;
    derived[1] = sqrt(var > 1e-300 ? var : 1e-300);
}

// (sum, sum^2) of the coarse residual in one workgroup (fixed order), for
// coarse grids of up to 64Ki cells; derived (may be NULL) receives (mean, rms);
// x8 (may be NULL) receives the network input: the residual normalised to
// zero mean and unit rms in BF16, channel 0 of 8
__global__ __launch_bounds__(1024) void k_coarse_stats1(const float* __restrict__ rc, int nc,
                                                        double* __restrict__ stats,
                                                        double* __restrict__ derived,
                                                        unsigned short* __restrict__ x8) {
    __shared__ double smem[16];
    __shared__ double ms[2];
    double a = 0.0, q = 0.0;
    for (int i = threadIdx.x; i < nc; i += blockDim.x) {
        const double v = rc[i];
        a += v;
        q += v * v;
    }
    a = cd_block_sum(a, smem);
    q = cd_block_sum(q, smem);
    if (threadIdx.x == 0) {
        stats[0] = a;
        stats[1] = q;
        if (derived) coarse_derived(stats, nc, derived);
        const double mean = a / nc;
        const double var = q / nc - mean * mean;
        ms[0] = mean;
        ms[1] = sqrt(var > 1e-300 ? var : 1e-300);
    }
    if (!x8) return;
    __syncthreads();
    const double mean = ms[0], sig = ms[1];
    for (int i = threadIdx.x; i < nc; i += blockDim.x) {
        uint4 v = make_uint4(0, 0, 0, 0);
        v.x = f32_to_bf16((float)(((double)rc[i] - mean) / sig));
        *reinterpret_cast<uint4*>(x8 + (size_t)i * 8) = v;
    }
}

// (mean, rms) after a multi-workgroup reduction of the coarse statistics
__global__ void k_coarse_derived(const double* __restrict__ stats, int nc,
                                 double* __restrict__ derived) {
    if (threadIdx.x == 0) coarse_derived(stats, nc, derived);
}

// partials (sum, sum^2) of the coarse residual per workgroup of 256 cells
__global__ __launch_bounds__(256) void k_coarse_stats(const float* __restrict__ rc, int nc,
                                                      double* __restrict__ partials) {
    __shared__ double smem[16];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const double v = i < nc ? (double)rc[i] : 0.0;
    const double a = cd_block_sum(v, smem);
    const double q = cd_block_sum(v * v, smem);
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = a;
        partials[2 * blockIdx.x + 1] = q;
    }
}

// stats = (sum, sum^2) over n coarse cells -> x = (rc - mean) / rms
__global__ void k_normalize_coarse(const float* __restrict__ rc, const double* __restrict__ stats,
                                   int n, float* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double mean = stats[0] / n;
    const double var = stats[1] / n - mean * mean;
    const double sig = sqrt(var > 1e-300 ? var : 1e-300);
    x[i] = (float)(((double)rc[i] - mean) / sig);
}

// packed-layout launch: grid (ceil(wpb / 256), rows, 2 colour planes); a
// thread owns packed column j of row Y in plane c, cell x = 2j + ((c+Y)&1)
__device__ __forceinline__ bool packed_thread(const Brick& bk, int w, int Y, int& c, int& j,
                                              int& x) {
    c = blockIdx.z;
    j = blockIdx.x * blockDim.x + threadIdx.x;
    x = 2 * j + ((c + Y) & 1);
    return j < bk.wpb && x < w;
}

// e = rms * (nmax/pi)^2 * bilinear(y) at cell centres (rms = derived[1], one
// value for the whole launch), written in the
// bricked layout of the blocked sweeps (the start of the smoothing); one
// thread per packed element, coalesced writes
__device__ __forceinline__ void prolong_bricked_at(const float* __restrict__ y,
                                                   const double* __restrict__ derived, int w,
                                                   int h, int f, int wc, int hc, double nscale,
                                                   const Brick& bk, float* __restrict__ e) {
    const int yy = blockIdx.y;
    int c, j, xx;
    if (!packed_thread(bk, w, yy, c, j, xx)) return;
    const double sig = derived[1];  // rms of the coarse residual
    const float inv = 1.f / f;  // exact for the power-of-two coarsenings in use
    const float u = (xx + 0.5f) * inv - 0.5f, v = (yy + 0.5f) * inv - 0.5f;
    int i0 = (int)floorf(u), j0 = (int)floorf(v);
    const float tu = u - i0, tv = v - j0;
    const int i1 = min(max(i0 + 1, 0), wc - 1), j1 = min(max(j0 + 1, 0), hc - 1);
    i0 = min(max(i0, 0), wc - 1);
    j0 = min(max(j0, 0), hc - 1);
    const float ev = (y[j0 * wc + i0] * (1.f - tu) + y[j0 * wc + i1] * tu) * (1.f - tv) +
                     (y[j1 * wc + i0] * (1.f - tu) + y[j1 * wc + i1] * tu) * tv;
    e[brick_row(bk, c, yy) + brick_col(j)] = (float)(sig * nscale * (double)ev);
}
__global__ __launch_bounds__(256) void k_prolong_bricked(const float* __restrict__ y,
                                                         const double* __restrict__ derived,
                                                         int w, int h, int f, int wc, int hc,
                                                         double nscale, Brick bk,
                                                         float* __restrict__ e) {
    prolong_bricked_at(y, derived, w, h, f, wc, hc, nscale, bk, e);
}

// Intermediate grid of the learned preconditioner (fm x fm fine cells per
// cell): rm = the block sum of the projected fine residual (r16 - rmean32),
// i.e. fm^2 times its block mean, the right-hand side of the unit-spacing
// operator on that grid; BF16, bricked like the fine right-hand side.  One
// thread per packed element of the intermediate grid.
// With the start of the intermediate-grid correction in the same launch (the
// two share the thread layout): em = the coarse output interpolated there.
__global__ __launch_bounds__(256) void k_restrict_to_mid(const unsigned short* __restrict__ r16,
                                                         Brick bk, const SolveDev* __restrict__ st,
                                                         int fm, int wm, int hm, Brick bkm,
                                                         unsigned short* __restrict__ rm,
                                                         const float* __restrict__ y,
                                                         const double* __restrict__ derived,
                                                         int fc, int wc, int hc, double nscale,
                                                         float* __restrict__ em) {
    prolong_bricked_at(y, derived, wm, hm, fc, wc, hc, nscale, bkm, em);
    const int Ym = blockIdx.y;
    int c, j, xm;
    if (!packed_thread(bkm, wm, Ym, c, j, xm)) return;
    const float rmean = st->rmean32;
    float acc = 0.f;
    for (int dy = 0; dy < fm; ++dy)
        for (int dx = 0; dx < fm; ++dx)
            acc += bf16_to_f32(r16[brick_at(bk, xm * fm + dx, Ym * fm + dy)]) - rmean;
    rm[brick_row(bkm, c, Ym) + brick_col(j)] = f32_to_bf16(acc);
}

// ---------------------------------------------------------------------------
// Flexible conjugate gradients (FCG(1)) preconditioned by the network plus
// smoothing sweeps.  With L the operator (negative semi-definite), r the
// projected residual and z = M(r) the preconditioned residual:
//   beta = -(z . Lp_old) / (p_old . Lp_old)   p = z + beta p_old
//   alpha = (p . r) / (p . Lp)                phi += alpha p
// alpha minimises the energy 1/2 phi'(-L)phi + b'phi along p, so every step
// lowers the energy norm of the error.  Lp = Lz + beta Lp_old needs no second
// stencil pass; p . Lp expands into the dot products taken below.
// ---------------------------------------------------------------------------
struct FcgDev {
    double beta, alpha;
    double pq;     // p . Lp of the current direction
    int have;      // a previous direction exists
    int bad;       // the last step had no descent direction
    const float* pprev;  // the previous direction (one of two ping-pong
                         // buffers; the captured iteration body reads it here)
};

// start of the learned iterations of a solve; p0: the zeroed first direction
// derived (NULL: none): (mean, rms) of an unnormalised input, (0, 1); zero (NULL:
// none): the mean that the intermediate sweeps subtract
__global__ void k_fcg_init(FcgDev* fd, const float* p0, double* derived, float* zero) {
    if (threadIdx.x != 0) return;
    if (derived) {
        derived[0] = 0.0;
        derived[1] = 1.0;
    }
    if (zero) zero[0] = 0.f;
    fd->beta = 0.0;
    fd->alpha = 0.0;
    fd->pq = 0.0;
    fd->have = 0;
    fd->bad = 0;
    fd->pprev = p0;
}

// Lz at packed element (c, Y, j) (cell x): the four neighbours lie in the
// other colour plane, up/down at column j, left/right at (x -+ 1) >> 1
__device__ __forceinline__ float lap_packed(const float* __restrict__ z, const Brick& bk, int c,
                                            int Y, int j, int x, int w, int h, float zc) {
    const int o = 1 - c;
    float s = 0.f, cnt = 0.f;
    if (x > 0) { s += z[brick_row(bk, o, Y) + brick_col((x - 1) >> 1)]; cnt += 1.f; }
    if (x < w - 1) { s += z[brick_row(bk, o, Y) + brick_col((x + 1) >> 1)]; cnt += 1.f; }
    if (Y > 0) { s += z[brick_row(bk, o, Y - 1) + brick_col(j)]; cnt += 1.f; }
    if (Y < h - 1) { s += z[brick_row(bk, o, Y + 1) + brick_col(j)]; cnt += 1.f; }
    return s - cnt * zc;
}

#ifndef CD_DOT_BANDS
#define CD_DOT_BANDS 256
#endif
// partials[4 * block + k]: p_old.Lz (= z.Lp_old: L is symmetric, so Lp_old
// needs neither a stencil pass nor storage), z.r, p_old.r, z.Lz over the
// packed elements of the workgroup's band of consecutive rows of one colour
// plane (fixed order).  Workgroups in XCD-contiguous order: both planes of a
// band, whose stencils read each other, and the neighbouring bands share an
// L2.  Rows go in groups of 4 whose loads are all issued before the first is
// used (clamped, in-range addresses; elements outside the grid contribute
// nothing).
__global__ __launch_bounds__(256) void k_fcg_dots(const float* __restrict__ z,
                                                  const FcgDev* __restrict__ fd,
                                                  const unsigned short* __restrict__ r16,
                                                  const SolveDev* __restrict__ st, Brick bk,
                                                  int w, int h, double* __restrict__ partials) {
    constexpr int G = 4;
    __shared__ double smem[64];
    const float rm = st->rmean32;
    const float* __restrict__ p = fd->pprev;
    // block order (column block fastest, then plane, then band of rows)
    const int ob = xcd_order();
    const int bx = ob % gridDim.x, c = (ob / gridDim.x) & 1, band = ob / (2 * gridDim.x);
    const int o = 1 - c;
    const int rows = (h + gridDim.y - 1) / gridDim.y;  // rows per band
    const int y0 = band * rows, y1 = min(h, y0 + rows);
    const int j0 = bx * blockDim.x + threadIdx.x;
    const int j = min(j0, bk.wpb - 1);
    const unsigned cj = brick_col(j), cjm = brick_col(max(j - 1, 0)),
                   cjp = brick_col(min(j + 1, bk.wpb - 1));
    double d0 = 0.0, d1 = 0.0, d2 = 0.0, d3 = 0.0;
    for (int Yb = y0; Yb < y1; Yb += G) {
        float zc[G], zl[G], zr[G], zu[G], zd[G], pv[G];
        unsigned short rv[G];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const int Y = min(Yb + k, h - 1);
            const int par = (c + Y) & 1;  // x = 2j + par
            const size_t ro = brick_row(bk, o, Y);
            const size_t i = brick_row(bk, c, Y) + cj;
            zc[k] = z[i];
            zl[k] = z[ro + (par ? cj : cjm)];   // (x - 1) >> 1
            zr[k] = z[ro + (par ? cjp : cj)];   // (x + 1) >> 1
            zu[k] = z[brick_row(bk, o, max(Y - 1, 0)) + cj];
            zd[k] = z[brick_row(bk, o, min(Y + 1, h - 1)) + cj];
            pv[k] = p[i];
            rv[k] = r16[i];
        }
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const int Y = Yb + k;
            const int x = 2 * j0 + ((c + Y) & 1);
            if (Y >= y1 || j0 >= bk.wpb || x >= w) continue;
            float sn = 0.f, cnt = 0.f;
            if (x > 0) { sn += zl[k]; cnt += 1.f; }
            if (x < w - 1) { sn += zr[k]; cnt += 1.f; }
            if (Y > 0) { sn += zu[k]; cnt += 1.f; }
            if (Y < h - 1) { sn += zd[k]; cnt += 1.f; }
            const float lz = sn - cnt * zc[k];
            const float rr = bf16_to_f32(rv[k]) - rm;
            d0 += (double)(pv[k] * lz);
            d1 += (double)(zc[k] * rr);
            d2 += (double)(pv[k] * rr);
            d3 += (double)(zc[k] * lz);
        }
    }
    double dd[4] = {d0, d1, d2, d3};
    cd_block_sum_n(dd, smem);
    d0 = dd[0];
    d1 = dd[1];
    d2 = dd[2];
    d3 = dd[3];
    if (threadIdx.x == 0) {
        partials[4 * ob] = d0;
        partials[4 * ob + 1] = d1;
        partials[4 * ob + 2] = d2;
        partials[4 * ob + 3] = d3;
    }
}

// single block: step coefficients from the dot products (fixed summation order)
__global__ void k_fcg_coef(const double* __restrict__ partials, int nblocks, FcgDev* fd) {
    __shared__ double smem[64];
    double d[4] = {0.0, 0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x)
        for (int k = 0; k < 4; ++k) d[k] += partials[4 * b + k];
    cd_block_sum_n(d, smem);
    if (threadIdx.x == 0) {
        const double zq = d[0], zr = d[1], pr = d[2], zlz = d[3];  // zq = z.Lp_old
        double beta = 0.0;
        if (fd->have && fd->pq < 0.0) beta = -zq / fd->pq;
        double pq = zlz + 2.0 * beta * zq + beta * beta * (fd->have ? fd->pq : 0.0);
        double prn = zr + beta * (fd->have ? pr : 0.0);
        double alpha = 0.0;
        fd->bad = 0;
        if (pq < 0.0 && isfinite(pq) && isfinite(prn)) {
            alpha = prn / pq;
        } else {
            // no usable direction: restart from z alone next time
            fd->bad = 1;
            beta = 0.0;
            pq = zlz;
        }
        fd->beta = beta;
        fd->alpha = alpha;
        fd->pq = pq;
        fd->have = fd->bad ? 0 : 1;
    }
}

// The learned iteration's FCG step folded into its convergence check:
// p = z + beta p_old (z: the smoothed correction, packed), phi_out = phi_in +
// alpha p, and the FP64 residual of phi_out with its BF16 copy and partial
// norms (as k_residual<2>).  phi and p are ping-pong pairs.  A wave takes ROWS rows
// of 64 columns one below the other: a row's new values serve as the next row's
// upper and the previous row's lower neighbours, the lanes beside as left and
// right ones; only the rows and columns around the wave's are formed once more
// (with the same FP32 and FP64 operations, so every cell's new value is one
// number).  Bound by memory: reading all five points of three fields per cell took
// 14.9 us at 1024 x 1024 (12.3 now; an iteration at 2048 x 2048 159 -> 147 us).
// fd->pprev is pointed at p_new for the next iteration.
// x8 (may be NULL): the workgroup also writes the next iteration's network
// input, the lf x lf block means of the new residual (BF16, channel 0 of 8 of
// a coarse grid lwc wide).  The host passes x8 only when the workgroups tile
// the grid exactly and cover whole coarse cells: lf divides 64, and the
// 4*ROWS rows of a workgroup are one or two coarse rows.  The FP64 residual is
// mean-free to rounding, so its block means need no projection.
// rows whose loads a thread issues together, and the most rows a thread takes
// (2 / 8 measured as fast at 1024^2, 1 % of an iteration slower at 2048^2)
#ifndef CD_STEP_G
#define CD_STEP_G 4
#endif
#ifndef CD_STEP_ROWS
#define CD_STEP_ROWS 8
#endif
template <int ROWS>
__global__ __launch_bounds__(256) void k_residual_step(const double* __restrict__ phi_in,
                                                       double* __restrict__ phi_out,
                                                       const double* __restrict__ b,
                                                       const SolveDev* __restrict__ st,
                                                       const float* __restrict__ z,
                                                       const float* __restrict__ p_old,
                                                       float* __restrict__ p_new,
                                                       FcgDev* __restrict__ fd,
                                                       unsigned short* __restrict__ r16, Brick bk,
                                                       int w, int h, double* __restrict__ partials,
                                                       unsigned short* __restrict__ x8, int lf,
                                                       int lwc) {
    constexpr int G = ROWS < CD_STEP_G ? ROWS : CD_STEP_G;  // rows whose loads are in flight together
    __shared__ double smem[32];
    __shared__ float csum[2][4][64];  // (coarse row, thread row, column) partial block sums
    __shared__ double rvs[4 * ROWS][64];
    const double bmean = st->bmean;
    const float alpha = (float)fd->alpha, beta = (float)fd->beta;
    const int ob = xcd_order();
    const int bx = ob % gridDim.x, by = ob / gridDim.x;
    const int lane = threadIdx.x;
    const int x0 = bx * 64 + lane;
    const int ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int Y0 = by * 4 * ROWS + ty * ROWS;  // the wave's first row
    const int x = min(x0, w - 1);
    // lanes 0 and 63: the column beyond the wave's
    const bool edge = lane == 0 || lane == 63;
    const int xe = lane == 0 ? max(x - 1, 0) : min(x + 1, w - 1);
    // bricked offsets (a plane pair holds < 2^29 elements in blocked mode)
    const unsigned cj = brick_col(x >> 1), cje = brick_col(xe >> 1);
    // (24-bit multiplies, full rate: row and brick indices are < 2^24)
    const unsigned plane = (unsigned)bk.plane, brow = (unsigned)bk.nbx * 512u;
    auto rowo = [&](int c, int y) -> unsigned {
        return (c ? plane : 0u) + __umul24((unsigned)(y >> 3), brow) + (unsigned)(y & 7) * 64u;
    };
    // buffer resources: 32-bit byte offsets, and reads past either end of a
    // buffer return 0 (the host passes grids of < 2^28 cells)
    const size_t n = (size_t)w * h;
    const __amdgpu_buffer_rsrc_t phi_rs = plane_rsrc(phi_in, n * sizeof(double));
    const __amdgpu_buffer_rsrc_t b_rs = plane_rsrc(b, n * sizeof(double));
    const __amdgpu_buffer_rsrc_t z_rs = plane_rsrc(z, 2 * bk.plane * sizeof(float));
    const __amdgpu_buffer_rsrc_t p_rs = plane_rsrc(p_old, 2 * bk.plane * sizeof(float));
    const __amdgpu_buffer_rsrc_t phio_rs = plane_rsrc(phi_out, n * sizeof(double));
    const __amdgpu_buffer_rsrc_t pn_rs = plane_rsrc(p_new, 2 * bk.plane * sizeof(float));
    const __amdgpu_buffer_rsrc_t r16_rs = plane_rsrc(r16, 2 * bk.plane * sizeof(unsigned short));
    auto ld64 = [](__amdgpu_buffer_rsrc_t rs, unsigned off) {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
    };
    // a cell of phi_in, z and p_old; its new direction and iterate
    struct Cell {
        double ph;
        float z, p;
    };
    auto load = [&](int col, unsigned cjc, int y) {
        Cell c;
        const int yc = min(max(y, 0), h - 1);
        const unsigned bi = (rowo((col + yc) & 1, yc) + cjc) * 4u;
        c.ph = ld64(phi_rs, (__umul24((unsigned)yc, (unsigned)w) + (unsigned)col) * 8u);
        c.z = buf_load<float>(z_rs, bi, 0);
        c.p = buf_load<float>(p_rs, bi, 0);
        return c;
    };
    auto pnew = [&](const Cell& c) { return c.z + beta * c.p; };
    auto phinew = [&](const Cell& c) { return c.ph + (double)(alpha * pnew(c)); };
    Cell mid = load(x, cj, Y0);
    double up = phinew(load(x, cj, Y0 - 1)), cur = phinew(mid);
#pragma unroll
    for (int g = 0; g < ROWS; g += G) {
        Cell next[G], side[G];
        double bb[G];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            next[k] = load(x, cj, Y0 + g + k + 1);
            side[k] = Cell{0.0, 0.f, 0.f};
            if (edge) side[k] = load(xe, cje, Y0 + g + k);
            bb[k] = ld64(b_rs, (__umul24((unsigned)min(Y0 + g + k, h - 1), (unsigned)w) + (unsigned)x) * 8u);
        }
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const int y = Y0 + g + k;
            const double down = phinew(next[k]), beyond = phinew(side[k]);
            double left = lane_prev(cur), right = lane_next(cur);
            left = lane == 0 ? beyond : left;
            right = lane == 63 ? beyond : right;
            // neighbours in the order left, up, right, down
            double s = 0.0, cnt = 0.0;
            if (x > 0) { cnt += 1.0; s += left; }
            if (y > 0) { cnt += 1.0; s += up; }
            if (x < w - 1) { cnt += 1.0; s += right; }
            if (y < h - 1) { cnt += 1.0; s += down; }
            const double rv = (bb[k] - bmean) - (s - cnt * cur);
            const bool in = x0 < w && y < h;
            rvs[ty * ROWS + g + k][lane] = in ? rv : 0.0;
            if (in) {
                const unsigned bi = rowo((x + y) & 1, y) + cj;
                __builtin_amdgcn_raw_buffer_store_b64(
                    __builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned, cur), phio_rs,
                    (__umul24((unsigned)y, (unsigned)w) + (unsigned)x) * 8u, 0, 0);
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(pnew(mid)), pn_rs, bi * 4u, 0, 0);
                __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16((float)rv), r16_rs, bi * 2u, 0, 0);
            }
            up = cur;
            cur = down;
            mid = next[k];
        }
    }
    // the sums take the rows ty, ty + 4, ... (the order of k_residual)
    __syncthreads();
    double rs = 0.0, rq = 0.0;
    float cpart0 = 0.f, cpart1 = 0.f;  // this thread's sums per coarse row
#pragma unroll
    for (int k = 0; k < ROWS; ++k) {
        const double rv = rvs[ty + 4 * k][lane];
        rs += rv;
        rq += rv * rv;
        if (x8) {
            if (ty + 4 * k >= lf) cpart1 += (float)rv;
            else cpart0 += (float)rv;
        }
    }
    double aq[2] = {rs, rq};
    cd_block_sum_n(aq, smem);
    const double a = aq[0], q = aq[1];
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        partials[2 * ob] = a;
        partials[2 * ob + 1] = q;
        if (ob == 0) fd->pprev = p_new;
    }
    if (x8) {  // uniform: every thread of the launch takes this branch or none
        const int ncr = (4 * ROWS) / lf > 1 ? 2 : 1;  // coarse rows of this workgroup
        csum[0][threadIdx.y][threadIdx.x] = cpart0;
        csum[1][threadIdx.y][threadIdx.x] = cpart1;
        __syncthreads();
        if (threadIdx.y < ncr) {
            // thread row cr sums coarse row cr over the four thread rows, then
            // over groups of lf lanes (fixed order: xor tree)
            const int cr = threadIdx.y;
            float v = ((csum[cr][0][threadIdx.x] + csum[cr][1][threadIdx.x]) +
                       csum[cr][2][threadIdx.x]) + csum[cr][3][threadIdx.x];
            for (int o = 1; o < lf; o <<= 1) v += __shfl_xor(v, o, 64);
            if ((threadIdx.x & (lf - 1)) == 0) {
                const int cx = (bx * 64 + threadIdx.x) / lf;
                const int cy = (by * 4 * ROWS) / lf + cr;
                *reinterpret_cast<uint4*>(x8 + ((size_t)cy * lwc + cx) * 8) =
                    make_uint4(f32_to_bf16(v / (float)(lf * lf)), 0, 0, 0);
            }
        }
    }
}

// launch of k_residual_step<rows> for rows in {1, 2, 4, 8}
void launch_residual_step(int rows, dim3 grid, dim3 blk, hipStream_t s, const double* phi_in,
                          double* phi_out, const double* b, const SolveDev* st, const float* z,
                          const float* p_old, float* p_new, FcgDev* fd, unsigned short* r16,
                          const Brick& bk, int w, int h, double* partials, unsigned short* x8,
                          int lf, int lwc) {
    switch (rows) {
    case 8: hipLaunchKernelGGL(k_residual_step<8>, grid, blk, 0, s, phi_in, phi_out, b, st, z, p_old, p_new, fd, r16, bk, w, h, partials, x8, lf, lwc); break;
    case 4: hipLaunchKernelGGL(k_residual_step<4>, grid, blk, 0, s, phi_in, phi_out, b, st, z, p_old, p_new, fd, r16, bk, w, h, partials, x8, lf, lwc); break;
    case 2: hipLaunchKernelGGL(k_residual_step<2>, grid, blk, 0, s, phi_in, phi_out, b, st, z, p_old, p_new, fd, r16, bk, w, h, partials, x8, lf, lwc); break;
    default: hipLaunchKernelGGL(k_residual_step<1>, grid, blk, 0, s, phi_in, phi_out, b, st, z, p_old, p_new, fd, r16, bk, w, h, partials, x8, lf, lwc); break;
    }
}

// coarse FP64 block mean of phi
__global__ void k_restrict_phi(const double* __restrict__ phi, int w, int f, int wc, int hc,
                               double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= wc * hc) return;
    const int J = i / wc, I = i - J * wc;
    double acc = 0.0;
    for (int yy = J * f; yy < J * f + f; ++yy)
        for (int xx = I * f; xx < I * f + f; ++xx) acc += phi[(size_t)yy * w + xx];
    out[i] = acc / (double)(f * f);
}

// target of one captured pair: (phi*_c - phi_k_c) / (rms * (nmax/pi)^2)
__global__ void k_capture_finish(const double* __restrict__ final_c,
                                 const double* __restrict__ phik_c,
                                 const double* __restrict__ stats, int nc, double nscale,
                                 float* __restrict__ t) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nc) return;
    const double mean = stats[0] / nc;
    const double var = stats[1] / nc - mean * mean;
    const double sig = sqrt(var > 1e-300 ? var : 1e-300);
    t[i] = (float)((final_c[i] - phik_c[i]) / (sig * nscale));
}

}  // namespace

// Wait until the check with sequence number seq has written the host's status
// mirror: spin on its sequence word (the status arrives within microseconds of
// the check), then, past a few milliseconds (long sweep batches, or a failed
// launch), synchronise the stream, which also reports errors.
int cd_wait_status(cd_context* ctx, unsigned seq) {
    const volatile unsigned* w = &ctx->host_status->seq;
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0;; ++i) {
        if (*w == seq) {
            std::atomic_thread_fence(std::memory_order_acquire);
            return CD_OK;
        }
        if ((i & 255) == 255 &&
            std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(4))
            break;
    }
    CD_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (ctx->host_status->seq != seq) {
        ctx->set_error("a check finished without writing the host status");
        return CD_ERR_HIP;
    }
    return CD_OK;
}

namespace {

// Whether cd_solve_region takes this solve: mixed precision, at most 128 x 128
// cells, batches a launch can hold, no network and no training-pair capture.
bool region_solve_applies(const cd_context* ctx, int w, int h, const cd_solve_opts* o) {
    if (w < 2 || h < 2 || w > SW_RX || h > 8 * BK_NW) return false;
    if (o->precision != CD_PREC_MIXED) return false;
    if (o->stop != CD_STOP_RESIDUAL && o->stop != CD_STOP_MAX_UPDATE) return false;
    if ((o->learned_init && ctx->net) || ctx->cap_x) return false;
    const int kmax = o->check_every > 0 ? o->check_every : auto_check_every(w, h);
    return std::min(kmax, o->max_sweeps) <= kRegionSweeps;
}

void solve_stats(const SolveDev& hs, const cd_solve_opts* o, int cum, int status,
                 std::chrono::steady_clock::time_point start, cd_solve_stats* out) {
    std::memset(out, 0, sizeof(*out));
    out->status = status;
    // the residual rule stops at the last check, after all enqueued sweeps
    out->sweeps = (hs.done && o->stop == CD_STOP_MAX_UPDATE) ? hs.sweeps_at_done : cum;
    out->checks = hs.checks;
    out->rel_residual = hs.rel;
    out->initial_rel_residual = hs.rel0;
    out->last_max_update = hs.last_max_update;
    out->elapsed_ms = std::chrono::duration<double, std::milli>(
                          std::chrono::steady_clock::now() - start).count();
}

// The whole solve in k_solve_region launches.  holes: NaN cells found in b when
// check_holes (phi is then untouched and nothing is solved).
int cd_solve_region(cd_context* ctx, const double* b, double* phi, int w, int h,
                    const cd_solve_opts* o, SolveDev* sd, bool timers, bool check_holes,
                    int* holes, cd_solve_stats* st_out) {
    const auto t_start = std::chrono::steady_clock::now();
    const bool track = o->stop == CD_STOP_MAX_UPDATE;
    const float om = (float)cd_sor_omega(o->omega, w, h);
    RegionArgs a{};
    a.w = w;
    a.h = h;
    a.max_sweeps = o->max_sweeps;
    a.kmax = o->check_every > 0 ? o->check_every : auto_check_every(w, h);
    a.adaptive = o->check_every <= 0 && !track;
    a.check_holes = check_holes;
    a.om2 = om / 2.f;
    a.om3 = om / 3.f;
    a.om4 = om / 4.f;
    a.tol = o->tol;
    a.margin = CD_CHECK_MARGIN;
    const int rows = h <= 2 * BK_NW ? 2 : h <= 4 * BK_NW ? 4 : 8;
    auto kernel = rows == 2 ? (track ? k_solve_region<2, true> : k_solve_region<2, false>)
                : rows == 4 ? (track ? k_solve_region<4, true> : k_solve_region<4, false>)
                            : (track ? k_solve_region<8, true> : k_solve_region<8, false>);
    for (;;) {
        a.seq = ++ctx->status_seq;
        const int before = a.resume ? ctx->host_status->cum : 0;
        if (timers) CD_TRY(ctx->timer_begin());
        hipLaunchKernelGGL(kernel, dim3(1), dim3(BK_THREADS), 0, ctx->stream, b, phi, a, sd,
                           ctx->host_status);
        CD_CHECK_LAUNCH(ctx);
        CD_TRY(cd_wait_status(ctx, a.seq));
        const SolveDev& hs = *ctx->host_status;
        if (timers)
            CD_TRY(ctx->timer_end(CD_KERNEL_SOR_SWEEP, 1, 12.0 * w * h * (hs.cum - before)));
        if (holes) *holes = hs.holes;
        if (hs.holes) return CD_OK;
        if (!hs.more) break;
        a.resume = 1;
    }
    const SolveDev hs = *ctx->host_status;
    CD_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (timers) CD_TRY(ctx->resolve_timers());
    const int status = !std::isfinite(hs.rel) ? CD_ERR_NAN : hs.done ? CD_OK : CD_ERR_NOT_CONVERGED;
    if (st_out) solve_stats(hs, o, hs.cum, status, t_start, st_out);
    return status;
}

}  // namespace

int cd_solve_device_internal(cd_context* ctx, const double* b, double* phi, const uint8_t* mask,
                             long long valid_cells, int w, int h, const cd_solve_opts* o,
                             cd_solve_stats* st_out, const SolveWork* work) {
    auto t_start = std::chrono::steady_clock::now();
    if (w < 2 || h < 2 || !b || !phi || !o) return CD_ERR_BAD_ARG;
    if (o->stop != CD_STOP_RESIDUAL && o->stop != CD_STOP_MAX_UPDATE) return CD_ERR_BAD_ARG;
    if (o->precision != CD_PREC_MIXED && o->precision != CD_PREC_FP64) return CD_ERR_BAD_ARG;
    const bool mixed = o->precision == CD_PREC_MIXED;
    const size_t n = (size_t)w * h;
    const double count = (double)valid_cells;
    if (!mask && region_solve_applies(ctx, w, h, o)) {
        if (!work) CD_TRY(ctx->ensure(ctx->solve_dev, sizeof(SolveDev)));
        return cd_solve_region(ctx, b, phi, w, h, o,
                               work ? work->sd : ctx->solve_dev.as<SolveDev>(), !work, false,
                               nullptr, st_out);
    }

    // workspace
    const dim3 rblk(RED_BX, RED_BY);
    const dim3 rgrid(div_up(w, RED_BX), div_up(h, RED_BY));
    const int nred = rgrid.x * rgrid.y;
    // FP32 sweeps without holes take k_rb_blocked on the bricked layout; FP64
    // sweeps and hole masks take k_rb_natural, blocked in time as well.
    // (the bricked layout's kernels address a plane pair through 32-bit byte offsets)
    const Brick bk = make_brick(w, h);
    const bool blocked = mixed && mask == nullptr && 2 * bk.plane * sizeof(float) < (1ull << 31);
    const size_t npk = 2 * bk.plane;
    SolveWork ws;
    if (work) {
        ws = *work;
    } else {
        // (sum, sum^2) per block for checks, four dot products per block for FCG
        CD_TRY(ctx->ensure(ctx->partials, cd_partials_bytes(nred)));
        CD_TRY(ctx->ensure(ctx->solve_dev, sizeof(SolveDev)));
        if (!mixed) CD_TRY(ctx->ensure(ctx->e64w, sizeof(double) * n));
        if (mixed) {
            CD_TRY(ctx->ensure(ctx->e32, sizeof(float) * (blocked ? npk : n)));
            // FP32 rhs (natural layout), BF16 rhs (bricked layout) or, under
            // the max-update rule, FP32 rhs (bricked layout)
            const size_t rb = blocked ? (o->stop == CD_STOP_MAX_UPDATE ? sizeof(float) : sizeof(unsigned short)) * npk
                                      : sizeof(float) * n;
            CD_TRY(ctx->ensure(ctx->r32, rb));
            CD_TRY(ctx->ensure(ctx->e32b, sizeof(float) * (blocked ? npk : n)));
        }
        ws.partials = ctx->partials.as<double>();
        ws.sd = ctx->solve_dev.as<SolveDev>();
        ws.e32 = mixed ? ctx->e32.as<float>() : nullptr;
        ws.e32b = mixed ? ctx->e32b.as<float>() : nullptr;
        ws.r = mixed ? ctx->r32.ptr : nullptr;
        ws.phi2 = mixed ? nullptr : ctx->e64w.as<double>();
    }
    double* partials = ws.partials;
    SolveDev* sd = ws.sd;
    float* e32 = mixed ? ws.e32 : nullptr;
    float* e32b = mixed ? ws.e32b : nullptr;
    double* phi2 = mixed ? nullptr : ws.phi2;  // FP64 sweeps: second buffer of the iterate
    float* r32 = mixed ? static_cast<float*>(ws.r) : nullptr;
    unsigned short* r16 = blocked ? static_cast<unsigned short*>(ws.r) : nullptr;
    const int track = o->stop == CD_STOP_MAX_UPDATE;
    // kernel timers record HIP events (created on demand): not with caller buffers
    auto timer_begin = [&]() -> int { return work ? (int)CD_OK : ctx->timer_begin(); };
    auto timer_end = [&](int kernel, long long launches, double bytes) -> int {
        return work ? (int)CD_OK : ctx->timer_end(kernel, launches, bytes);
    };
    // padding stays finite
    if (mixed && blocked) CD_TRY(cd_fill_f32(ctx, r32, track ? npk : npk / 2, 0.f));

    const double omega = cd_sor_omega(o->omega, w, h);
    const int kmax = o->check_every > 0 ? o->check_every : auto_check_every(w, h);
    const bool adaptive = o->check_every <= 0 && o->stop == CD_STOP_RESIDUAL;
    hipStream_t s = ctx->stream;

    // right-hand-side statistics: mean over non-hole cells, ||P b||
    hipLaunchKernelGGL(k_rhs_moments, rgrid, rblk, 0, s, b, w, h, sd, 0, partials);
    hipLaunchKernelGGL(k_rhs_finish, dim3(1), dim3(1024), 0, s, partials, nred, sd, 0, count);
    hipLaunchKernelGGL(k_rhs_moments, rgrid, rblk, 0, s, b, w, h, sd, 1, partials);
    hipLaunchKernelGGL(k_rhs_finish, dim3(1), dim3(1024), 0, s, partials, nred, sd, 1, count);
    CD_CHECK_LAUNCH(ctx);
    // (under the blocked residual rule every batch starts from zero by itself, and
    // learned iterations write their corrections before they read them: what the
    // buffers hold outside the grid is loaded, but not used)
    if (mixed && (track || !blocked)) CD_TRY(cd_fill_f32(ctx, e32, blocked ? npk : n, 0.f));
    if (blocked && track) CD_TRY(cd_fill_f32(ctx, e32b, npk, 0.f));

    const int fblocks = std::min(div_up((long long)n, CD_BLOCK), 65536);
    // residual launch of a check: kResidualRows rows per thread, fewer on
    // smaller grids (more workgroups in flight; the partials stay <= nred)
    const int kResidualRows = nred >= 16384 ? 8 : nred >= 8192 ? 4 : nred >= 4096 ? 2 : 1;
    const dim3 cgrid(div_up(w, RED_BX), div_up(h, RED_BY * kResidualRows));
    const int ncheck = cgrid.x * cgrid.y;  // <= nred
    // the end of every check: k_check on the residual pass's partials, then the
    // host's wait for the status (the residual pass's timer is open)
    // (wait false: the caller enqueues the work that follows and waits itself)
    auto wait_check = [&]() -> int {
        return ctx->profiling ? (int)CD_OK : cd_wait_status(ctx, ctx->status_seq);
    };
    auto finish_check = [&](int check_id, int timer_kernels, double bytes, int nparts,
                            bool wait = true) -> int {
        const unsigned seq = ++ctx->status_seq;
        hipLaunchKernelGGL(k_check, dim3(1), dim3(1024), 0, s, partials, nparts, sd,
                           ctx->host_status, seq, count, check_id, o->stop, o->tol);
        CD_CHECK_LAUNCH(ctx);
        CD_TRY(timer_end(CD_KERNEL_RESIDUAL, timer_kernels, bytes));
        if (ctx->profiling) {
            CD_HIP(ctx, hipStreamSynchronize(s));
            CD_TRY(ctx->resolve_timers());
        } else if (wait) {
            CD_TRY(wait_check());
        }
        return CD_OK;
    };
    // flush: fold the current FP32 correction into phi64 first (the last launch of
    // a batch under the blocked residual rule has done that, and so have learned
    // iterations)
    auto enqueue_check = [&](int check_id, bool flush = true, bool wait = true) -> int {
        CD_TRY(timer_begin());
        if (blocked) {
            if (flush)
                hipLaunchKernelGGL(k_flush_packed, rgrid, rblk, 0, s, phi, e32, e32b, sd, w, h, bk);
            if (track)
                launch_residual<3>(kResidualRows, cgrid, rblk, s, phi, nullptr, b, mask, sd, r32, r16, bk,
                                   w, h, partials);
            else
                launch_residual<2>(kResidualRows, cgrid, rblk, s, phi, nullptr, b, mask, sd, r32, r16, bk,
                                   w, h, partials);
        } else if (mixed) {
            hipLaunchKernelGGL(k_flush, dim3(fblocks), dim3(CD_BLOCK), 0, s, phi, e32, e32b, sd, n);
            launch_residual<1>(kResidualRows, cgrid, rblk, s, phi, nullptr, b, mask, sd, r32, r16, bk, w, h,
                               partials);
        } else {
            launch_residual<0>(kResidualRows, cgrid, rblk, s, phi, phi2, b, mask, sd, r32, r16, bk, w, h,
                               partials);
        }
        return finish_check(check_id, (mixed && flush) ? 3 : 2,
                            (blocked ? (flush ? 48.0 : 18.0) : (mixed ? 44.0 : 16.0)) * (double)n,
                            ncheck, wait);
    };

    const float om = (float)omega;
    const float om2 = om / 2.f, om3 = om / 3.f, om4 = om / 4.f;
    int track_lid = 0;  // tracking launches of this solve
    // count_sweeps sweeps in launches between e32 and e32b, the first reading
    // e32; pro: it starts from this intermediate-grid correction, interpolated
    // at the cells, instead.  ends.zero: it starts from zero instead; ends.phi: the
    // last launch adds the correction to it.  ahead: sweeps of them that one launch
    // has already taken
    auto enqueue_blocked_om = [&](int first, int count_sweeps, float om2, float om3, float om4,
                                  const MidGrid* pro = nullptr, int ahead = 0,
                                  BatchEnds ends = BatchEnds{}) -> int {
        CD_TRY(timer_begin());
        const BlockedPlan pl = blocked_plan(w, h, count_sweeps - ahead, track != 0,
                                            cd_partials_bytes(nred));
        TrackBatch words = track_batch(partials, pl.t.ntiles, pl.sweeps, kStopGroup, o->tol);
        const int skipped = ahead > 0 ? 1 : 0;
        int launches = skipped;
        float* bufs[2] = {e32, e32b};
        const void* rhs = track ? (const void*)r32 : (const void*)r16;
        for (int done_sw = ahead; done_sw < count_sweeps; ++launches) {
            const int nsw = std::min(pl.sweeps, count_sweeps - done_sw);
            float* ein = bufs[launches & 1];
            float* eout = bufs[1 - (launches & 1)];
            launch_blocked(pl, track != 0, launches == 0 ? pro : nullptr, s, ein, eout, rhs, bk,
                           nsw, om2, om3, om4, &sd->rmean32, sd, 1 - (launches & 1),
                           words.launch(++track_lid, nsw, first + done_sw),
                           BatchEnds{done_sw + nsw == count_sweeps ? ends.phi : nullptr,
                                     launches == 0 ? ends.zero : 0});
            done_sw += nsw;
        }
        if (track) {  // the last launch's own decision
            launch_blocked(pl, true, nullptr, s, bufs[launches & 1], bufs[1 - (launches & 1)], rhs,
                           bk, 0, om2, om3, om4, &sd->rmean32, sd, 1 - (launches & 1),
                           words.check(++track_lid));
            ++launches;
        }
        CD_CHECK_LAUNCH(ctx);
        // algorithmic bytes: 12 B per cell per red+black sweep (e read, e write,
        // rhs read), whatever the number of sweeps fused into one launch
        CD_TRY(timer_end(CD_KERNEL_SOR_SWEEP, launches - skipped,
                         12.0 * (double)n * (count_sweeps - ahead)));
        return CD_OK;
    };
    // natural layout: launches of several sweeps between the buffers b0 and b1;
    // FP64 iterates continue in the buffer the last check found current, FP32
    // corrections start in b0 (the check's flush cleared it)
    auto enqueue_natural = [&](auto* b0, auto* b1, const auto* rhs, auto om, const auto* mean,
                               int first, int count_sweeps) -> int {
        using T = std::remove_pointer_t<decltype(b0)>;
        const SweepTiles t = natural_tiles(w, h, sizeof(T) == 8, count_sweeps, track != 0,
                                           cd_partials_bytes(nred));
        const int most = natural_sweeps(t, count_sweeps, track != 0);
        const dim3 grid(sweep_grid(t.ntiles)), blk(64 * NAT_NW);
        const NatOmega<T> oms{om, om / 2, om / 3, om / 4};
        int cur = mixed ? 0 : ctx->host_status->cur;
        TrackBatch words = track_batch(partials, t.ntiles, most, 1, o->tol);
        CD_TRY(timer_begin());
        int launches = 0;
        for (int done_sw = 0; done_sw < count_sweeps; ++launches) {
            const int nsw = std::min(most, count_sweeps - done_sw);
            T* in = cur ? b1 : b0;
            T* out = cur ? b0 : b1;
            const TrackArgs tr = words.launch(++track_lid, nsw, first + done_sw);
            if (track)
                hipLaunchKernelGGL((k_rb_natural<T, true>), grid, blk, 0, s, in, out, rhs, mask, t,
                                   nsw, oms, mean, sd, 1 - cur, tr);
            else
                hipLaunchKernelGGL((k_rb_natural<T, false>), grid, blk, 0, s, in, out, rhs, mask, t,
                                   nsw, oms, mean, sd, 1 - cur, tr);
            cur = 1 - cur;
            done_sw += nsw;
        }
        if (track) {  // the last launch's own decision
            const TrackArgs tr = words.check(++track_lid);
            hipLaunchKernelGGL((k_rb_natural<T, true>), grid, blk, 0, s, cur ? b1 : b0,
                               cur ? b0 : b1, rhs, mask, t, 0, oms, mean, sd, 1 - cur, tr);
            ++launches;
        }
        CD_CHECK_LAUNCH(ctx);
        return timer_end(CD_KERNEL_SOR_SWEEP, launches,
                         (mixed ? 12.0 : 24.0) * (double)n * count_sweeps);
    };
    // a batch of sweeps, of which `ahead` are already enqueued; fold: phi takes the
    // correction (blocked residual rule; else the check's flush does that)
    auto enqueue_sweeps = [&](int first, int count_sweeps, int ahead = 0, bool fold = true) -> int {
        if (blocked)
            return enqueue_blocked_om(first, count_sweeps, om2, om3, om4, nullptr, ahead,
                                      track ? BatchEnds{}
                                            : BatchEnds{fold ? phi : nullptr, 1});
        if (mixed)
            return enqueue_natural(e32, e32b, r32, (float)omega, &sd->rmean32, first, count_sweeps);
        return enqueue_natural(phi, phi2, b, omega, &sd->bmean, first, count_sweeps);
    };

    // ---- learned correction / capture geometry ------------------------------
    const cd_net_arch* arch = ctx->net ? cd_net_arch_of(ctx->net) : nullptr;
    const double nscale = std::pow((double)std::max(w, h) / M_PI, 2.0);
    auto coarse_ok = [&](int f, int lv) {
        const int m = f << (lv - 1);
        return f > 0 && w % f == 0 && h % f == 0 && (w / f) % (1 << (lv - 1)) == 0 &&
               (h / f) % (1 << (lv - 1)) == 0 && m > 0;
    };
    // (the step check addresses the FP64 grids through 32-bit byte offsets)
    bool learned = o->learned_init && arch && blocked && o->stop == CD_STOP_RESIDUAL &&
                   coarse_ok(arch->coarsen, arch->levels) && !work &&
                   (size_t)n * sizeof(double) < (1ull << 31);
    const int lf = arch ? arch->coarsen : 1;
    const int lwc = w / std::max(lf, 1), lhc = h / std::max(lf, 1);
    const bool capture = ctx->cap_x && ctx->cap_coarsen > 0 && w == ctx->cap_coarsen * ctx->cap_w &&
                         h == ctx->cap_coarsen * ctx->cap_h && blocked && !track && !work;
    const int cwc = capture ? ctx->cap_w : 0, chc = capture ? ctx->cap_h : 0;
    constexpr int kMaxPairsPerSolve = 64;
    std::vector<int> cap_slots;
    if (learned) {
        CD_TRY(ctx->ensure(ctx->lc_r, sizeof(float) * (size_t)lwc * lhc));
        CD_TRY(ctx->ensure(ctx->lc_x, sizeof(float) * (size_t)lwc * lhc));
        CD_TRY(ctx->ensure(ctx->lc_y, sizeof(float) * (size_t)lwc * lhc));
        CD_TRY(ctx->ensure(ctx->fcg_p, sizeof(float) * npk));
        CD_TRY(ctx->ensure(ctx->fcg_q, sizeof(float) * npk));
        CD_TRY(ctx->ensure(ctx->fcg_dev, sizeof(FcgDev)));
        CD_TRY(ctx->ensure(ctx->fcg_phi, sizeof(double) * n));
    }
    // intermediate grid of the preconditioner (coarsening a multiple of 4, >= 8)
    const int mid_sweeps = arch ? arch->mid_sweeps : 0;
    const bool mid = learned && mid_sweeps > 0 && lf >= 8 && lf % 4 == 0;
    const int fm = mid ? lf / 4 : 1;
    const int wm = w / fm, hm = h / fm;
    const Brick bkm = make_brick(wm, hm);
    if (mid) {
        const size_t npm = 2 * bkm.plane;
        CD_TRY(ctx->ensure(ctx->fcg_em, sizeof(float) * npm));
        CD_TRY(ctx->ensure(ctx->fcg_emb, sizeof(float) * npm));
        CD_TRY(ctx->ensure(ctx->fcg_rm, sizeof(unsigned short) * npm));
        CD_TRY(ctx->ensure(ctx->fcg_zero, sizeof(float) * 4));
        // the right-hand side's padding stays finite
        CD_TRY(cd_fill_f32(ctx, ctx->fcg_rm.as<float>(), npm / 2, 0.f));
    }
    if (learned || capture)
        CD_TRY(ctx->ensure(ctx->lc_stats, sizeof(double) * 2 * (kMaxPairsPerSolve + 2)));
    if (capture) {
        CD_TRY(ctx->ensure(ctx->cap_phi, sizeof(double) * (size_t)cwc * chc * (kMaxPairsPerSolve + 1)));
        CD_TRY(ctx->ensure(ctx->lc_r, sizeof(float) * (size_t)std::max(cwc * chc, lwc * lhc)));
    }
    // restrict the residual of the last check to (wc x hc) into lc_r; stats
    // slot receives (sum, sum^2) of the coarse residual
    // x8 (may be NULL): also write the network input there (coarse grids of up
    // to 64Ki cells; *x8_done tells whether it was).  direct: x8 receives the
    // coarse residual itself (the input of a linear network) and no statistics
    // are computed
    auto restrict_stats = [&](int f, int wc, int hc, double* stats, double* derived,
                              unsigned short* x8 = nullptr, bool* x8_done = nullptr,
                              bool direct = false) -> int {
        const int nc = wc * hc;
        const int rb = f < 8 ? div_up(nc, 256) : div_up(nc, 4);  // thread / wave per cell
        hipLaunchKernelGGL(k_restrict_r16, dim3(rb), dim3(256), 0, s, r16, bk, sd, f, wc, hc,
                           ctx->lc_r.as<float>(), direct ? x8 : nullptr);
        if (x8_done) *x8_done = direct && x8;
        if (direct && x8) {
            CD_CHECK_LAUNCH(ctx);
            return CD_OK;
        }
        if (nc <= 65536) {
            hipLaunchKernelGGL(k_coarse_stats1, dim3(1), dim3(1024), 0, s, ctx->lc_r.as<float>(),
                               nc, stats, derived, x8);
            if (x8_done) *x8_done = x8 != nullptr;
        } else {
            const int nb = div_up(nc, 256);  // <= nred: the partials buffer is large enough
            hipLaunchKernelGGL(k_coarse_stats, dim3(nb), dim3(256), 0, s, ctx->lc_r.as<float>(),
                               nc, partials);
            CD_TRY(cd_reduce_partials(ctx, partials, nb, 2, stats));
            if (derived)
                hipLaunchKernelGGL(k_coarse_derived, dim3(1), dim3(64), 0, s, stats, nc, derived);
        }
        CD_CHECK_LAUNCH(ctx);
        return CD_OK;
    };
    // restrict the residual of the last check to (wc x hc), normalise into
    // xout; stats slot receives (sum, sum^2) of the coarse residual
    auto restrict_normalize = [&](int f, int wc, int hc, float* xout, double* stats) -> int {
        CD_TRY(restrict_stats(f, wc, hc, stats, nullptr));
        const int nc = wc * hc;
        hipLaunchKernelGGL(k_normalize_coarse, dim3(div_up(nc, 256)), dim3(256), 0, s,
                           ctx->lc_r.as<float>(), stats, nc, xout);
        CD_CHECK_LAUNCH(ctx);
        return CD_OK;
    };
    // the FP64 iterate: phi, or during learned iterations either buffer of the
    // pair (phi, fcg_phi) that the folded FCG steps alternate between
    double* phi_cur = phi;
    auto capture_pair = [&]() -> int {
        if (ctx->cap_count >= ctx->cap_capacity || (int)cap_slots.size() >= kMaxPairsPerSolve)
            return CD_OK;
        const int slot = ctx->cap_count++;
        const int i = (int)cap_slots.size();
        const int nc = cwc * chc;
        double* stats = ctx->lc_stats.as<double>() + 2 * (2 + i);
        CD_TRY(restrict_normalize(ctx->cap_coarsen, cwc, chc, ctx->cap_x + (size_t)slot * nc, stats));
        hipLaunchKernelGGL(k_restrict_phi, dim3(div_up(nc, 256)), dim3(256), 0, s, phi_cur, w,
                           ctx->cap_coarsen, cwc, chc, ctx->cap_phi.as<double>() + (size_t)(i + 1) * nc);
        CD_CHECK_LAUNCH(ctx);
        cap_slots.push_back(slot);
        return CD_OK;
    };
    const float oms = arch ? (float)arch->smooth_omega : om;
    const int nsmooth = arch ? std::max(1, arch->smooth_sweeps) : 4;
    // the smoothing launches start from e32; after `nl` launches the result
    // sits in e32 (nl even) or e32b (nl odd)
    const int smooth_launches = div_up(nsmooth, blocked_plan(w, h, nsmooth, false, 0).sweeps);
    // packed-element kernels: grid (packed width / 256, rows, 2 planes); the
    // dot products stride over rows so that their partials fit nred blocks
    const int pbx = div_up(bk.wpb, 256);
    const dim3 packed_grid(pbx, h, 2);
    // (at most CD_DOT_BANDS bands of rows: each thread accumulates several rows
    // before the block reduction; 1024 measured slower at 1024^2, 128 and 512
    // no faster at 2048^2)
    const int dot_rows = std::max(1, std::min(std::min(h, CD_DOT_BANDS), nred / (2 * pbx)));
    const dim3 dot_grid(pbx, dot_rows, 2);
    const int dot_blocks = 2 * pbx * dot_rows;
    if (dot_blocks > nred) learned = false;  // tiny grids: partials hold nred blocks
    float* zbuf = (smooth_launches & 1) ? e32b : e32;
    int learned_applied = 0, learned_rejected = 0;
    // a linear network maps the unnormalised coarse residual (scaling commutes
    // with it): the restriction writes the network input, no statistics pass
    const bool direct_input = learned && arch->linear;
    // ... and where the check's workgroups cover whole coarse cells, the check
    // that ends an FCG iteration writes the next iteration's network input
    // itself (the iterations after the first start from it)
    // the step check's rows per thread and grid (its partials stay <= nred)
    const int kStepRows = std::min(kResidualRows, CD_STEP_ROWS);
    const dim3 stgrid(div_up(w, RED_BX), div_up(h, RED_BY * kStepRows));
    const int nstep = stgrid.x * stgrid.y;
    const int crows = 4 * kStepRows;  // rows of a step-check workgroup
    const bool fuse_restrict = direct_input && lf >= 2 && lf <= 64 && (lf & (lf - 1)) == 0 &&
                               w % 64 == 0 && h % crows == 0 && crows % lf == 0 &&
                               crows / lf <= 2 && lwc * lf == w && lhc * lf == h;
    unsigned short* net_x8 = nullptr;
    if (fuse_restrict) CD_TRY(cd_net_coarse_input(ctx->net, lhc, lwc, &net_x8));
    bool x8_ready = false;  // the last check wrote the network input

    int check_id = 0;
    int cum = 0;
    CD_TRY(enqueue_check(check_id, !blocked));  // (no correction yet)
    if (capture && !ctx->host_status->done) CD_TRY(capture_pair());
    double prev_rel = ctx->host_status->rel;
    int k = kmax;
    if (adaptive) k = std::min(kmax, std::max(8, kmax / 4));
    bool done = ctx->host_status->done != 0;
    // the warm start, kept while learned iterations run: if they are abandoned
    // with a residual above the starting one (degenerate right-hand sides of
    // folded meshes can do that: a lower energy norm of the error does not
    // bound the residual), plain SOR restarts from it
    const double start_rel = ctx->host_status->rel;
    if (learned && !done) {
        CD_TRY(cd_fill_f32(ctx, ctx->fcg_p.as<float>(), npk, 0.f));
        hipLaunchKernelGGL(k_fcg_init, dim3(1), dim3(64), 0, s, ctx->fcg_dev.as<FcgDev>(),
                           ctx->fcg_p.as<float>(),
                           direct_input ? ctx->lc_stats.as<double>() + 2 : nullptr,
                           mid ? ctx->fcg_zero.as<float>() : nullptr);
        CD_CHECK_LAUNCH(ctx);
        CD_TRY(ctx->ensure(ctx->phi_start, sizeof(double) * n));
        CD_HIP(ctx, hipMemcpyAsync(ctx->phi_start.ptr, phi, sizeof(double) * n,
                                   hipMemcpyDeviceToDevice, s));
    }
    // learned FCG iterations; abandoned for plain SOR when the residual stops
    // falling (the iterate is kept when its residual is below the starting
    // one: every step lowered the error's energy norm)
    double best_rel = ctx->host_status->rel;
    int stall = 0;
    // one FCG iteration up to the next check: restriction, network, prolongation,
    // smoothing sweeps, FCG update.  Launched eagerly the first time in a solve
    // (which also sizes every buffer), then replayed as one captured graph.
    auto fcg_body = [&](int first_sweep) -> int {
        FcgDev* fd = ctx->fcg_dev.as<FcgDev>();
        CD_TRY(timer_begin());
        // slot 0: (sum, sum^2) of the coarse residual; slot 1: (mean, rms)
        double* stats = ctx->lc_stats.as<double>();
        unsigned short* x8 = nullptr;
        bool prepared = false;
        CD_TRY(cd_net_coarse_input(ctx->net, lhc, lwc, &x8));
        if (x8_ready && x8 == net_x8)
            prepared = true;
        else
            CD_TRY(restrict_stats(lf, lwc, lhc, stats, stats + 2, x8, &prepared, direct_input));
        if (prepared)
            CD_TRY(cd_net_forward_prepared(ctx->net, ctx->lc_y.as<float>(), lhc, lwc));
        else
            CD_TRY(cd_net_forward_coarse(ctx->net, ctx->lc_r.as<float>(), stats,
                                         ctx->lc_y.as<float>(), lhc, lwc));
        if (mid) {
            // coarse -> intermediate grid, smoothing there, -> fine grid
            const int pbm = div_up(bkm.wpb, 256);
            unsigned short* rm = ctx->fcg_rm.as<unsigned short>();
            float* em[2] = {ctx->fcg_em.as<float>(), ctx->fcg_emb.as<float>()};
            hipLaunchKernelGGL(k_restrict_to_mid, dim3(pbm, hm, 2), dim3(256), 0, s, r16, bk, sd,
                               fm, wm, hm, bkm, rm, ctx->lc_y.as<float>(), stats + 2, lf / fm,
                               lwc, lhc, nscale, em[0]);
            const BlockedPlan pm = blocked_plan(wm, hm, mid_sweeps, false, 0);
            int cur_m = 0;
            for (int done_sw = 0; done_sw < mid_sweeps;) {
                const int nsw = std::min(pm.sweeps, mid_sweeps - done_sw);
                launch_blocked(pm, false, nullptr, s, em[cur_m], em[1 - cur_m], rm, bkm, nsw,
                               oms / 2.f, oms / 3.f, oms / 4.f, ctx->fcg_zero.as<float>(), sd, 0,
                               TrackArgs{});
                cur_m = 1 - cur_m;
                done_sw += nsw;
            }
            CD_CHECK_LAUNCH(ctx);
            CD_TRY(timer_end(CD_KERNEL_LEARNED, 3, 0.0));
            // the fine smoothing starts from em interpolated at the fine cells
            const MidGrid pro{em[cur_m], bkm, wm, hm, fm};
            CD_TRY(enqueue_blocked_om(first_sweep, nsmooth, oms / 2.f, oms / 3.f, oms / 4.f, &pro));
        } else {
            hipLaunchKernelGGL(k_prolong_bricked, packed_grid, dim3(256), 0, s,
                               ctx->lc_y.as<float>(), stats + 2, w, h, lf, lwc, lhc, nscale, bk,
                               e32);
            CD_CHECK_LAUNCH(ctx);
            CD_TRY(timer_end(CD_KERNEL_LEARNED, 3, 0.0));
            CD_TRY(enqueue_blocked_om(first_sweep, nsmooth, oms / 2.f, oms / 3.f, oms / 4.f));
        }
        CD_TRY(timer_begin());
        hipLaunchKernelGGL(k_fcg_dots, dot_grid, dim3(256), 0, s, zbuf, fd, r16, sd, bk, w, h,
                           partials);
        hipLaunchKernelGGL(k_fcg_coef, dim3(1), dim3(1024), 0, s, partials, dot_blocks, fd);
        CD_CHECK_LAUNCH(ctx);
        CD_TRY(timer_end(CD_KERNEL_LEARNED, 2, 10.0 * (double)n));
        return CD_OK;
    };
    // the check that ends an FCG iteration, with the iteration's step folded
    // in: p = z + beta p_old, phi += alpha p, into the other buffer of each
    // pair (the direction pair is fcg_p / fcg_q)
    double* const phis[2] = {phi, ctx->fcg_phi.as<double>()};
    float* const dirs[2] = {ctx->fcg_p.as<float>(), ctx->fcg_q.as<float>()};
    int fk = 0, pk = 0;  // buffers holding the iterate and the last direction
    auto enqueue_step_check = [&](int check_id) -> int {
        CD_TRY(timer_begin());
        launch_residual_step(kStepRows, stgrid, rblk, s, phis[fk], phis[1 - fk], b, sd, zbuf,
                             dirs[pk], dirs[1 - pk], ctx->fcg_dev.as<FcgDev>(), r16, bk, w, h,
                             partials, fuse_restrict ? net_x8 : nullptr, lf, lwc);
        x8_ready = fuse_restrict;
        fk = 1 - fk;
        pk = 1 - pk;
        phi_cur = phis[fk];
        return finish_check(check_id, 2, 38.0 * (double)n, nstep);
    };
    int fcg_iter = 0;
    while (!done && learned && cum < o->max_sweeps) {
        if (o->max_sweeps - cum < nsmooth) { learned = false; break; }  // a cycle no longer fits
        // profiling keeps the launches separate so that every timer records
        const bool replay = ctx->graphs && !ctx->profiling && fcg_iter > 0;
        if (replay) {
            const cd_context::FcgKey key{w,        h,        nsmooth,
                                         mid ? mid_sweeps : 0,   ctx->net, ctx->gen,
                                         cd_net_gen(ctx->net)};
            if (!(ctx->fcg_exec && ctx->fcg_key == key)) {
                if (ctx->fcg_exec) {
                    CD_HIP(ctx, hipGraphExecDestroy(ctx->fcg_exec));
                    ctx->fcg_exec = nullptr;
                }
                hipGraph_t graph = nullptr;
                CD_HIP(ctx, hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed));
                const int body = fcg_body(cum);
                const hipError_t ce = hipStreamEndCapture(s, &graph);
                if (body != CD_OK) {
                    if (graph) (void)hipGraphDestroy(graph);
                    return body;
                }
                CD_HIP(ctx, ce);
                const hipError_t ie = hipGraphInstantiate(&ctx->fcg_exec, graph, nullptr, nullptr, 0);
                (void)hipGraphDestroy(graph);
                CD_HIP(ctx, ie);
                ctx->fcg_key = key;
            }
            CD_HIP(ctx, hipGraphLaunch(ctx->fcg_exec, s));
        } else {
            CD_TRY(fcg_body(cum));
        }
        ++fcg_iter;
        cum += nsmooth;
        CD_TRY(enqueue_step_check(++check_id));
        ++learned_applied;
        const SolveDev& hs = *ctx->host_status;
        done = hs.done != 0;
        if (!std::isfinite(hs.rel)) stall = 7;  // abandoned below, back to the warm start
        if (capture && !done && std::isfinite(hs.rel) &&
            check_id % std::max(ctx->cap_every, 1) == 0)
            CD_TRY(capture_pair());
#ifdef CD_TRACE_LEARNED
        {
            FcgDev hf;
            CD_HIP(ctx, hipMemcpy(&hf, ctx->fcg_dev.ptr, sizeof(hf), hipMemcpyDeviceToHost));
            fprintf(stderr, "fcg %d: rel %.3e alpha %.3e beta %.3e pq %.3e bad %d\n",
                    learned_applied, hs.rel, hf.alpha, hf.beta, hf.pq, hf.bad);
        }
#endif
        // the residual of CG-type iterations may rise for a few steps before
        // it falls; give up only when 8 iterations bring no halving
        if (hs.rel < 0.5 * best_rel) {
            best_rel = hs.rel;
            stall = 0;
        } else if (++stall >= 8) {
            ++learned_rejected;
            learned = false;
            if (!(hs.rel <= start_rel) && !done) {
                // back to the warm start; the next check recomputes its residual
                CD_HIP(ctx, hipMemcpyAsync(phi, ctx->phi_start.ptr, sizeof(double) * n,
                                           hipMemcpyDeviceToDevice, s));
                fk = 0;
                phi_cur = phi;
                CD_TRY(enqueue_check(++check_id, false));
                done = ctx->host_status->done != 0;
            }
        }
        prev_rel = ctx->host_status->rel;
    }
    if (fk) {  // the iterate ended in the second buffer
        CD_HIP(ctx, hipMemcpyAsync(phi, phis[1], sizeof(double) * n, hipMemcpyDeviceToDevice, s));
        fk = 0;
        phi_cur = phi;
    }
    // Max-update rule in mixed precision: the sweeps see the right-hand side
    // rounded (BF16 / FP32) at the last check, which perturbs every update by
    // up to omega/4 times that rounding of the check's residual.  A stop is
    // therefore confirmed on a fresh FP64 residual: the check after the
    // stopping batch folds the correction and rounds the new residual, and
    // one more launch of sweeps must meet the rule again; if none of its
    // sweeps does, the solve goes on (and a later stop is confirmed the same
    // way).  FP64 sweeps read b itself and stop at once.
    const bool confirm_stop = track && mixed;
    const int confirm_sweeps = blocked ? kStopGroup : 4;
    bool confirming = false;
    // Residual rule on the blocked layout: a full batch (not one sized to end the
    // solve) is expected to be followed by another, whose first launch goes out
    // before the host has the check's status.  It only writes the correction:
    // if the solve stops here, nothing reads it.
    // (A batch has at least 8 sweeps.)  400 x 400: 1.87 -> 1.76 ms to 1e-6.
    constexpr int kAhead = 8;
    const bool look_ahead = blocked && !track && !ctx->profiling && !capture;
    int ahead = 0;  // sweeps of the next batch already enqueued
    while (!done && cum < o->max_sweeps) {
        const int nsw = std::min(confirming ? confirm_sweeps : k, o->max_sweeps - cum);
        CD_TRY(enqueue_sweeps(cum, nsw, ahead));
        cum += nsw;
        ++check_id;
        // (a batch that one early launch took whole has not reached phi yet)
        CD_TRY(enqueue_check(check_id, !blocked || track || ahead == nsw, false));
        ahead = 0;
        if (look_ahead && nsw == kmax && kmax >= kAhead && o->max_sweeps - cum >= kAhead) {
            ahead = std::min(kAhead, blocked_plan(w, h, kAhead, false, 0).sweeps);
            CD_TRY(enqueue_sweeps(cum, ahead, 0, false));
        }
        CD_TRY(wait_check());
        const SolveDev& hs = *ctx->host_status;
        done = hs.done != 0;
        if (!std::isfinite(hs.rel)) break;
        if (confirm_stop) {
            if (done && !confirming && cum < o->max_sweeps) {
                hipLaunchKernelGGL(k_reopen, dim3(1), dim3(64), 0, s, sd);
                CD_CHECK_LAUNCH(ctx);
                confirming = true;
                done = false;
                continue;
            }
            confirming = false;  // confirmed (done) or not: back to full batches
        }
        if (capture && !done && check_id % std::max(ctx->cap_every, 1) == 0)
            CD_TRY(capture_pair());
        if (adaptive && !done) {
            // geometric rate estimate over the last batch -> sweeps still needed
            double rel = hs.rel;
            double rho = (prev_rel > 0 && rel > 0 && rel < prev_rel) ? std::pow(rel / prev_rel, 1.0 / nsw) : 1.0;
            int want = kmax;
            if (rho < 0.999999) {
                double need = std::log(o->tol / rel) / std::log(rho);
                want = (int)std::ceil(need * CD_CHECK_MARGIN) + 2;
            }
            k = std::max(8, std::min(kmax, want));
            prev_rel = rel;
        }
    }
    if (capture && !cap_slots.empty()) {
        const int nc = cwc * chc;
        double* fin = ctx->cap_phi.as<double>();  // slot 0: the final solution
        hipLaunchKernelGGL(k_restrict_phi, dim3(div_up(nc, 256)), dim3(256), 0, s, phi, w,
                           ctx->cap_coarsen, cwc, chc, fin);
        for (size_t i = 0; i < cap_slots.size(); ++i)
            hipLaunchKernelGGL(k_capture_finish, dim3(div_up(nc, 256)), dim3(256), 0, s, fin,
                               fin + (i + 1) * nc, ctx->lc_stats.as<double>() + 2 * (2 + i), nc,
                               nscale, ctx->cap_t + (size_t)cap_slots[i] * nc);
        CD_CHECK_LAUNCH(ctx);
    }
    const SolveDev hs = *ctx->host_status;
    if (!mixed && hs.cur)  // FP64 sweeps: the iterate ended in the second buffer
        CD_HIP(ctx, hipMemcpyAsync(phi, phi2, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    if (mask && o->max_sweeps > 0) {
        hipLaunchKernelGGL(k_set_holes_nan, dim3(div_up((long long)n, CD_BLOCK)), dim3(CD_BLOCK), 0,
                           s, phi, mask, n);
        CD_CHECK_LAUNCH(ctx);
    }
    CD_HIP(ctx, hipStreamSynchronize(s));

    int status = CD_OK;
    if (!std::isfinite(hs.rel)) status = CD_ERR_NAN;
    else if (!hs.done) status = CD_ERR_NOT_CONVERGED;
    if (st_out) {
        solve_stats(hs, o, cum, status, t_start, st_out);
        st_out->learned_applied = learned_applied;
        st_out->learned_rejected = learned_rejected;
    }
    return status;
}

// Sizes of the solve buffers of a w x h grid (see SolveWork).
void cd_solve_work_sizes(int w, int h, size_t* nred, size_t* npk) {
    *nred = (size_t)div_up(w, RED_BX) * div_up(h, RED_BY);
    *npk = 2 * make_brick(w, h).plane;
}

// Hole mask of a right-hand side (NaN cells and their neighbours' validity
// bits) and the number of holes, read back through host_buf (pinned).
int cd_hole_mask(cd_context* ctx, const double* d_rhs, int w, int h, uint8_t* mask,
                 double* partials, double* fill, double* host_buf, long long* holes) {
    const dim3 rblk(RED_BX, RED_BY);
    const dim3 rgrid(div_up(w, RED_BX), div_up(h, RED_BY));
    const int nred = rgrid.x * rgrid.y;
    hipLaunchKernelGGL(k_build_mask, rgrid, rblk, 0, ctx->stream, d_rhs, mask, w, h, partials);
    CD_CHECK_LAUNCH(ctx);
    CD_TRY(cd_reduce_partials(ctx, partials, nred, 1, fill));
    CD_HIP(ctx, hipMemcpyAsync(host_buf, fill, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    CD_HIP(ctx, hipStreamSynchronize(ctx->stream));
    *holes = (long long)host_buf[0];
    return CD_OK;
}

// ---------------------------------------------------------------------------
// Allocation-free solve.  Its buffers (reduction partials, solve state, the
// two ping-pong FP32 corrections, the right-hand side of the sweeps, the hole
// mask and the reduction slots) live in one static device array per GPU,
// sized for grids of up to CD_NOALLOC_MAX_SIDE x CD_NOALLOC_MAX_SIDE cells and
// held until the process ends.  The array's address on each device is taken
// once (hipGetSymbolAddress, with that device current) and kept per device;
// host code passes that address, never the array's name.
// ---------------------------------------------------------------------------
namespace {

constexpr size_t al256(size_t x) { return (x + 255) / 256 * 256; }

struct NoallocLayout {
    size_t partials, sd, e32, e32b, r, mask, fill, total;
};

constexpr NoallocLayout noalloc_layout(int w, int h) {
    // the bricked layout of make_brick and the reduction grid of the checks
    const size_t wp = (size_t)(w + 1) / 2;
    const size_t plane = ((size_t)(h + 7) / 8 * 8) * ((wp + 63) / 64 * 64);
    const size_t npk = 2 * plane;  // >= w*h (natural layout with holes fits)
    const size_t nred = (size_t)((w + RED_BX - 1) / RED_BX) * ((h + RED_BY - 1) / RED_BY);
    NoallocLayout L{};
    size_t o = 0;
    L.partials = o; o += al256(cd_partials_bytes(nred));
    L.sd = o;       o += al256(sizeof(SolveDev));
    L.e32 = o;      o += al256(sizeof(float) * npk);
    L.e32b = o;     o += al256(sizeof(float) * npk);
    L.r = o;        o += al256(sizeof(float) * npk);  // FP32 (max-update rule) or BF16
    L.mask = o;     o += al256((size_t)w * h);
    L.fill = o;     o += al256(sizeof(double) * 4);
    L.total = o;
    return L;
}

constexpr size_t kNoallocScratchBytes =
    noalloc_layout(CD_NOALLOC_MAX_SIDE, CD_NOALLOC_MAX_SIDE).total;
static_assert(kNoallocScratchBytes <= ((size_t)CD_NOALLOC_SCRATCH_MIB << 20) &&
                  kNoallocScratchBytes > ((size_t)(CD_NOALLOC_SCRATCH_MIB - 1) << 20),
              "CD_NOALLOC_SCRATCH_MIB states the scratch size");

static __device__ __align__(256) unsigned char scratch[kNoallocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_ptr[kMaxDevices] = {};

// Device address of this device's scratch (set up on the first call per
// device; the caller has made ctx->device current).
int noalloc_scratch(cd_context* ctx, unsigned char** out) {
    if (ctx->device < 0 || ctx->device >= kMaxDevices) return CD_ERR_BAD_ARG;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[ctx->device]) {
        void* p = nullptr;
        CD_HIP(ctx, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) {
            ctx->set_error("hipGetSymbolAddress returned no address for the solve scratch");
            return CD_ERR_HIP;
        }
        g_scratch_ptr[ctx->device] = static_cast<unsigned char*>(p);
    }
    *out = g_scratch_ptr[ctx->device];
    return CD_OK;
}

}  // namespace

extern "C" {

int cd_poisson_solve_device_noalloc(cd_context* ctx, const double* d_rhs, double* d_phi,
                                    int width, int height, const cd_solve_opts* opts,
                                    cd_solve_stats* stats) {
    if (!ctx || !d_rhs || !d_phi || width < 2 || height < 2) return CD_ERR_BAD_ARG;
    cd_solve_opts def;
    if (!opts) { cd_solve_opts_default(&def); opts = &def; }
    if (opts->learned_init) {
        ctx->set_error("cd_poisson_solve_device_noalloc: learned_init needs the network's "
                       "buffers; use cd_poisson_solve_device");
        return CD_ERR_BAD_ARG;
    }
    const NoallocLayout L = noalloc_layout(width, height);
    if (L.total > kNoallocScratchBytes) {
        ctx->set_error("cd_poisson_solve_device_noalloc: a " + std::to_string(width) + " x " +
                       std::to_string(height) + " grid needs " + std::to_string(L.total) +
                       " bytes of scratch, more than the " +
                       std::to_string(kNoallocScratchBytes) + " held per device (grids up to " +
                       std::to_string(CD_NOALLOC_MAX_SIDE) + " x " +
                       std::to_string(CD_NOALLOC_MAX_SIDE) + ")");
        return CD_ERR_BAD_ARG;
    }
    CD_HIP(ctx, hipSetDevice(ctx->device));
    unsigned char* base = nullptr;
    CD_TRY(noalloc_scratch(ctx, &base));
    SolveWork ws;
    ws.partials = reinterpret_cast<double*>(base + L.partials);
    ws.sd = reinterpret_cast<SolveDev*>(base + L.sd);
    ws.e32 = reinterpret_cast<float*>(base + L.e32);
    ws.e32b = reinterpret_cast<float*>(base + L.e32b);
    ws.r = base + L.r;
    // FP64 sweeps use neither correction: their second buffer lies over both
    ws.phi2 = reinterpret_cast<double*>(base + L.e32);
    uint8_t* mask = base + L.mask;
    double* fill = reinterpret_cast<double*>(base + L.fill);
    if (region_solve_applies(ctx, width, height, opts)) {
        int found = 0;
        const int rc = cd_solve_region(ctx, d_rhs, d_phi, width, height, opts, ws.sd, false, true,
                                       &found, stats);
        if (!found) return rc;
    }
    long long holes = 0;
    CD_TRY(cd_hole_mask(ctx, d_rhs, width, height, mask, ws.partials, fill,
                        reinterpret_cast<double*>(ctx->host_status), &holes));
    const long long n = (long long)width * height;
    return cd_solve_device_internal(ctx, d_rhs, d_phi, holes > 0 ? mask : nullptr, n - holes,
                                    width, height, opts, stats, &ws);
}

int cd_poisson_solve_device(cd_context* ctx, const double* d_rhs, double* d_phi, int width,
                            int height, const cd_solve_opts* opts, cd_solve_stats* stats) {
    if (!ctx || !d_rhs || !d_phi || width < 2 || height < 2) return CD_ERR_BAD_ARG;
    cd_solve_opts def;
    if (!opts) { cd_solve_opts_default(&def); opts = &def; }
    CD_HIP(ctx, hipSetDevice(ctx->device));
    const size_t n = (size_t)width * height;
    size_t nred, npk;
    cd_solve_work_sizes(width, height, &nred, &npk);
    if (region_solve_applies(ctx, width, height, opts)) {
        CD_TRY(ctx->ensure(ctx->solve_dev, sizeof(SolveDev)));
        int found = 0;
        const int rc = cd_solve_region(ctx, d_rhs, d_phi, width, height, opts,
                                       ctx->solve_dev.as<SolveDev>(), true, true, &found, stats);
        if (!found) return rc;
    }
    // hole mask: only used by the solve when the right-hand side contains NaN
    CD_TRY(ctx->ensure(ctx->mask, n));
    CD_TRY(ctx->ensure(ctx->partials, cd_partials_bytes(nred)));  // as the solve
    CD_TRY(ctx->ensure(ctx->fill, sizeof(double) * 4));
    long long holes = 0;
    CD_TRY(cd_hole_mask(ctx, d_rhs, width, height, ctx->mask.as<uint8_t>(),
                        ctx->partials.as<double>(), ctx->fill.as<double>(),
                        reinterpret_cast<double*>(ctx->host_status), &holes));
    const uint8_t* mask = holes > 0 ? ctx->mask.as<uint8_t>() : nullptr;
    return cd_solve_device_internal(ctx, d_rhs, d_phi, mask, (long long)n - holes, width, height,
                                    opts, stats);
}

int cd_context_set_capture(cd_context* ctx, float* d_x, float* d_t, int capacity, int h, int w,
                           int coarsen, int every) {
    if (!ctx) return CD_ERR_BAD_ARG;
    if (d_x && (!d_t || capacity < 1 || h < 1 || w < 1 || coarsen < 1)) return CD_ERR_BAD_ARG;
    ctx->cap_x = d_x;
    ctx->cap_t = d_t;
    ctx->cap_capacity = d_x ? capacity : 0;
    ctx->cap_count = 0;
    ctx->cap_h = h;
    ctx->cap_w = w;
    ctx->cap_coarsen = coarsen;
    ctx->cap_every = every < 1 ? 1 : every;
    return CD_OK;
}

int cd_context_capture_count(const cd_context* ctx, int* count) {
    if (!ctx || !count) return CD_ERR_BAD_ARG;
    *count = ctx->cap_count;
    return CD_OK;
}

int cd_poisson_solve(cd_context* ctx, const double* rhs, double* phi, int width, int height,
                     const cd_solve_opts* opts, cd_solve_stats* stats) {
    if (!ctx || !rhs || !phi || width < 2 || height < 2) return CD_ERR_BAD_ARG;
    CD_HIP(ctx, hipSetDevice(ctx->device));
    const size_t n = (size_t)width * height;
    CD_TRY(ctx->ensure(ctx->b64w, sizeof(double) * n));
    CD_TRY(ctx->ensure(ctx->phi64w, sizeof(double) * n));
    CD_HIP(ctx, hipMemcpyAsync(ctx->b64w.ptr, rhs, sizeof(double) * n, hipMemcpyHostToDevice,
                               ctx->stream));
    CD_HIP(ctx, hipMemcpyAsync(ctx->phi64w.ptr, phi, sizeof(double) * n, hipMemcpyHostToDevice,
                               ctx->stream));
    int st = cd_poisson_solve_device(ctx, ctx->b64w.as<double>(), ctx->phi64w.as<double>(), width,
                                     height, opts, stats);
    if (st != CD_OK && st != CD_ERR_NOT_CONVERGED && st != CD_ERR_NAN) return st;
    CD_HIP(ctx, hipMemcpyAsync(phi, ctx->phi64w.ptr, sizeof(double) * n, hipMemcpyDeviceToHost,
                               ctx->stream));
    CD_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return st;
}

}  // extern "C"
