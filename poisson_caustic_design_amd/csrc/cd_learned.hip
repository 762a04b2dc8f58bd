// Learned initial correction: a bias-free convolutional encoder-decoder with
// hand-written gfx950 kernels (BF16 MFMA, FP32 accumulation) for inference and
// training.  No counterpart in the reference; see cd_api.h for the contract.
//
// Tensors are NHWC.  Activations are BF16 with channel counts that are
// multiples of 8 (16-byte vectors per pixel); gradients are FP32.  A 3x3
// convolution is an implicit GEMM: M = pixels, N = output channels,
// K = 9 * input channels (tap-major: k = tap * Cin + ci, tap = 3*dy + dx),
// computed with v_mfma_f32_16x16x32_bf16.  Lane layouts of that instruction:
//   A (16x32): lane l holds A[l % 16][8*(l/16) + j], j = 0..7
//   B (32x16): lane l holds B[8*(l/16) + j][l % 16]
//   D (16x16): lane l holds D[4*(l/16) + r][l % 16], r = 0..3
#include <hip/hip_runtime.h>

#include <atomic>

#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "cd_internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;

namespace {

inline int div_up(long long a, long long b) { return (int)((a + b - 1) / b); }

__device__ __forceinline__ u16 to_bf16(float x) {
    const unsigned u = __float_as_uint(x);
    return (u16)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float from_bf16(u16 v) { return __uint_as_float((unsigned)v << 16); }

union V8 {
    bf16x8 v;
    uint4 u;
    u16 h[8];
};

// ---------------------------------------------------------------------------
// 3x3 convolution, implicit GEMM on MFMA.
//   IN 0: BF16 input = channel concatenation of x1 (c1 ch) and x2 (c2 ch)
//   IN 1: FP32 input g (c1 ch), multiplied by (mask > 0) when mask != NULL
//   OUT 0: BF16 output (cy ch), optional ReLU
//   OUT 1: FP32 output split by channel into y1 (cy ch) and y2 (cy2 ch)
// wt: BF16 weights [nb*16][kpad], kpad a multiple of 32, zero padded.
// One workgroup = 4 waves = 64 consecutive pixels; a wave computes 16 pixels
// by NB*16 output channels.
// ---------------------------------------------------------------------------
template <int NB, int IN, int OUT>
__global__ __launch_bounds__(256) void k_conv3x3(const u16* __restrict__ x1,
                                                 const u16* __restrict__ x2, int c1, int c2,
                                                 const float* __restrict__ g,
                                                 const u16* __restrict__ mask,
                                                 const u16* __restrict__ wt, int kpad, int B,
                                                 int H, int W, u16* __restrict__ ybf,
                                                 float* __restrict__ y1, float* __restrict__ y2,
                                                 int cy, int cy2, int relu, int mode1) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long npix = (long long)B * H * W;
    const long long p0 = (long long)blockIdx.x * 64 + wave * 16;
    const int cin = IN == 0 ? c1 + c2 : c1;
    const int K = 9 * cin;
    const long long pa = p0 + (lane & 15);
    const bool pvalid = pa < npix;
    int xb = 0, yb = 0, bb = 0;
    if (pvalid) {
        xb = (int)(pa % W);
        const long long t = pa / W;
        yb = (int)(t % H);
        bb = (int)(t / H);
    }
    floatx4 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int kq = 8 * (lane >> 4);
    const u16* wrow = wt + (size_t)(lane & 15) * kpad + kq;
    // A fragment of K chunk kc (8 consecutive k of this lane's pixel)
    auto load_a = [&](int kc) -> V8 {
        V8 a;
        a.u = make_uint4(0, 0, 0, 0);
        const int k = kc + kq;
        if (pvalid && k < K) {
            const int tap = k / cin, ci = k - tap * cin;
            const int yy = yb + tap / 3 - 1, xx = xb + tap % 3 - 1;
            if (yy >= 0 && yy < H && xx >= 0 && xx < W) {
                const long long q = ((long long)bb * H + yy) * W + xx;
                if (IN == 0) {
                    if (ci >= c1) {
                        a.u = *reinterpret_cast<const uint4*>(x2 + q * c2 + (ci - c1));
                    } else if (mode1 == 0) {
                        a.u = *reinterpret_cast<const uint4*>(x1 + q * c1 + ci);
                    } else {
                        // x1 holds [B][H/2][W/2][c1]: nearest 2x upsampling
                        const long long q1 =
                            ((long long)bb * (H >> 1) + (yy >> 1)) * (W >> 1) + (xx >> 1);
                        a.u = *reinterpret_cast<const uint4*>(x1 + q1 * c1 + ci);
                    }
                } else {
                    const float4 g0 = *reinterpret_cast<const float4*>(g + q * c1 + ci);
                    const float4 g1 = *reinterpret_cast<const float4*>(g + q * c1 + ci + 4);
                    float gv[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
                    if (mask) {
                        V8 m;
                        m.u = *reinterpret_cast<const uint4*>(mask + q * c1 + ci);
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            if (!(from_bf16(m.h[j]) > 0.f)) gv[j] = 0.f;
                    }
#pragma unroll
                    for (int j = 0; j < 8; ++j) a.h[j] = to_bf16(gv[j]);
                }
            }
        }
        return a;
    };
    // K is walked in groups of 4 chunks: all loads of a group are issued
    // before its MFMAs (latency overlap); the accumulation order is unchanged
    constexpr int U = 4;
    for (int kc0 = 0; kc0 < kpad; kc0 += 32 * U) {
        V8 a[U], bw[U][NB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kc = kc0 + 32 * u;
            if (kc < kpad) {
                a[u] = load_a(kc);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    bw[u][nb].u = *reinterpret_cast<const uint4*>(wrow + (size_t)nb * 16 * kpad + kc);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (kc0 + 32 * u < kpad) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u].v, bw[u][nb].v, acc[nb],
                                                                      0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const long long p = p0 + 4 * (lane >> 4) + r;
            const int ch = nb * 16 + (lane & 15);
            if (p >= npix) continue;
            float v = acc[nb][r];
            if (OUT == 0) {
                if (ch < cy) {
                    if (relu) v = fmaxf(v, 0.f);
                    ybf[p * cy + ch] = to_bf16(v);
                }
            } else {
                float* dst = nullptr;
                if (ch < cy) dst = y1 + p * cy + ch;
                else if (ch - cy < cy2) dst = y2 + p * cy2 + (ch - cy);
                if (dst) *dst = v;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Forward 3x3 convolution on one 8x8 output tile per workgroup (4 waves, two
// tile rows each).  The tile's input (10x10 pixels with the zero-padded halo,
// x1 read through nearest 2x upsampling when mode1, then x2 concatenated) and
// the weights of this workgroup's NB*16 output channels are staged in LDS by
// one round of coalesced loads; the MFMA loop then reads only LDS.  The A/B
// fragments and the order of the K chunks are those of k_conv3x3<NB, 0, OUT>,
// so every output is bit-identical to it; the tiles cut the latency chain of
// the per-chunk global gathers, which sets the time of these small layers.
//   OUT 0: BF16 output ybf [B][H][W][cy] (ReLU optional);
//   OUT 1: FP32 output yf [B][H][W][cy]; OUT 2: yf (cy ch) and y2 (cy2 ch).
//   IN 1: FP32 gradient g (c1 ch, masked) in place of x1, x2, for the input
//   gradient (transposed weights), as k_conv3x3<NB, 1, 1>.
// grid: (ceil(W/8), ceil(H/8), B * cblocks), output channels
// [16*NB*cblk, 16*NB*(cblk+1)) with cblk = blockIdx.z % cblocks.
// LDS: 100 * (cin + 8) + NB*16 * (kpad + 8) u16 (row paddings spread banks).
// ---------------------------------------------------------------------------
constexpr int CT = 8;  // output tile side

// Stage a P x P patch of the (concatenated) input, image origin (oy, ox), into
// LDS at xs (u16 pixel stride xstride): thread t takes vector t % ng of pixels
// t / ng, t / ng + 256 / ng, ... (one division per thread, none in the loop).
// The loads go in groups of SB without branches (each from a clamped, valid
// pixel; out-of-image pixels are zeroed after the load), so that a group waits
// for one L2 round trip, not one per vector.  mode1 as for k_conv3x3_tile.
template <int P>
__device__ __forceinline__ void stage_patch(u16* __restrict__ xs, int xstride,
                                            const u16* __restrict__ x1,
                                            const u16* __restrict__ x2, int c1, int c2, int H,
                                            int W, int b, int oy, int ox, int mode1) {
    constexpr int SB = 8;
    constexpr int NP = P * P;
    const int ng = (c1 + c2) >> 3;
    const int pstride = 256 / ng;
    const int gi = threadIdx.x % ng;
    const int ci = gi * 8;
    // this thread's source: channels ci.. of x2 (after the c1 of x1) or x1;
    // mode1 applies to x1 only (a pooled input has no x2)
    const bool use2 = ci >= c1;
    const u16* __restrict__ src = use2 ? x2 + (ci - c1) : x1 + ci;
    const int cs = use2 ? c2 : c1;
    const int up = (!use2 && mode1 == 1) ? 1 : 0;  // nearest upsampling: source at half size
    if (threadIdx.x >= pstride * ng) return;
    for (int pb = threadIdx.x / ng; pb < NP; pb += SB * pstride) {
        uint4 v[SB];
        bool ok[SB];
        if (mode1 == 2) {
            // x1 at twice the resolution, 2x2 average pooled as k_avgpool2 does
#pragma unroll
            for (int u = 0; u < SB; ++u) {
                const int px = pb + u * pstride;
                const int yy = oy + px / P, xx = ox + px % P;
                ok[u] = px < NP && yy >= 0 && yy < H && xx >= 0 && xx < W;
                const int yc = min(max(yy, 0), H - 1), xc = min(max(xx, 0), W - 1);
                const long long r0 = ((long long)b * (2 * H) + 2 * yc) * (2 * W) + 2 * xc;
                const long long r1 = r0 + 2 * W;
                V8 p00, p01, p10, p11, o;
                p00.u = *reinterpret_cast<const uint4*>(src + r0 * cs);
                p01.u = *reinterpret_cast<const uint4*>(src + (r0 + 1) * cs);
                p10.u = *reinterpret_cast<const uint4*>(src + r1 * cs);
                p11.u = *reinterpret_cast<const uint4*>(src + (r1 + 1) * cs);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float sm = from_bf16(p00.h[e]) + from_bf16(p01.h[e]) +
                                     from_bf16(p10.h[e]) + from_bf16(p11.h[e]);
                    o.h[e] = to_bf16(0.25f * sm);
                }
                v[u] = o.u;
            }
        } else {
#pragma unroll
            for (int u = 0; u < SB; ++u) {
                const int px = pb + u * pstride;
                const int yy = oy + px / P, xx = ox + px % P;
                ok[u] = px < NP && yy >= 0 && yy < H && xx >= 0 && xx < W;
                const int yc = min(max(yy, 0), H - 1) >> up, xc = min(max(xx, 0), W - 1) >> up;
                const long long q = ((long long)b * (H >> up) + yc) * (W >> up) + xc;
                v[u] = *reinterpret_cast<const uint4*>(src + q * cs);
            }
        }
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            const int px = pb + u * pstride;
            if (px < NP)
                *reinterpret_cast<uint4*>(xs + px * xstride + ci) =
                    ok[u] ? v[u] : make_uint4(0, 0, 0, 0);
        }
    }
}

// The same for an FP32 gradient g of c channels, rounded to BF16 and zeroed where
// mask (NULL: none) is not positive, as k_conv3x3 with IN 1 reads it.
template <int P>
__device__ __forceinline__ void stage_grad(u16* __restrict__ xs, int xstride,
                                           const float* __restrict__ g,
                                           const u16* __restrict__ mask, int c, int H, int W,
                                           int b, int oy, int ox) {
    constexpr int SB = 4;
    constexpr int NP = P * P;
    const int ng = c >> 3;
    const int pstride = 256 / ng;
    const int ci = (threadIdx.x % ng) * 8;
    if (threadIdx.x >= pstride * ng) return;
    for (int pb = threadIdx.x / ng; pb < NP; pb += SB * pstride) {
        float4 v0[SB], v1[SB];
        V8 m[SB];
        bool ok[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            const int px = pb + u * pstride;
            const int yy = oy + px / P, xx = ox + px % P;
            ok[u] = px < NP && yy >= 0 && yy < H && xx >= 0 && xx < W;
            const long long q = (((long long)b * H + min(max(yy, 0), H - 1)) * W +
                                 min(max(xx, 0), W - 1)) * c + ci;
            v0[u] = *reinterpret_cast<const float4*>(g + q);
            v1[u] = *reinterpret_cast<const float4*>(g + q + 4);
            if (mask) m[u].u = *reinterpret_cast<const uint4*>(mask + q);
        }
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            const int px = pb + u * pstride;
            if (px >= NP) continue;
            const float gv[8] = {v0[u].x, v0[u].y, v0[u].z, v0[u].w,
                                 v1[u].x, v1[u].y, v1[u].z, v1[u].w};
            V8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bool on = ok[u] && !(mask && !(from_bf16(m[u].h[e]) > 0.f));
                o.h[e] = on ? to_bf16(gv[e]) : (u16)0;
            }
            *reinterpret_cast<uint4*>(xs + px * xstride + ci) = o.u;
        }
    }
}

// Stage `rows` weight rows of kpad (u16) from wsrc into ws (row stride kpad + 8):
// vector it = row * kv + cv for it = threadIdx.x, +256, ... with (row, cv)
// advanced incrementally, in branch-free groups of 8 loads (a vector past the
// last row is loaded from that row and stored there: the value it has)
__device__ __forceinline__ void stage_weights(u16* __restrict__ ws,
                                              const u16* __restrict__ wsrc, int rows,
                                              int kpad) {
    constexpr int SB = 8;
    const int kv = kpad >> 3, wstride = kpad + 8;
    const int dq = 256 / kv, dr = 256 - dq * kv;
    int row = threadIdx.x / kv, cv = threadIdx.x - row * kv;
    while (row < rows) {
        uint4 v[SB];
        int rr[SB], cc[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            rr[u] = min(row, rows - 1);
            cc[u] = cv;
            v[u] = *reinterpret_cast<const uint4*>(wsrc + (size_t)rr[u] * kpad + cv * 8);
            row += dq;
            cv += dr;
            if (cv >= kv) { cv -= kv; ++row; }
        }
#pragma unroll
        for (int u = 0; u < SB; ++u)
            *reinterpret_cast<uint4*>(ws + rr[u] * wstride + cc[u] * 8) = v[u];
    }
}

// The K loop of a 3x3 convolution read from LDS: an input patch of side P
// (pixel stride xstride, cin channels) and NB*16 weight rows (stride kpad + 8).
// Lane l's A pixel of M-tile m has patch index pbase[m] (its 3x3 neighbourhood
// starts there); acc[m][nb] accumulates output channels nb*16 + (l % 16) in
// the order of the K chunks, the order k_conv3x3 uses.  k = kc + kq = tap *
// cin + cc is tracked incrementally: cin is a multiple of 8, so the lane's 8
// consecutive k lie in one tap.
template <int NB, int MT, int P>
__device__ __forceinline__ void conv_lds(floatx4 (&acc)[MT][NB], const u16* __restrict__ xs,
                                         int xstride, int cin, const u16* __restrict__ ws,
                                         int kpad, const int (&pbase)[MT], int lane) {
    const int K = 9 * cin;
    const int kq = 8 * (lane >> 4);
    const int wstride = kpad + 8;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[m][nb] = floatx4{0.f, 0.f, 0.f, 0.f};
    const u16* wrow = ws + (lane & 15) * wstride + kq;
    int cc = kq, tdy = 0, tdx = 0;
    while (cc >= cin) {
        cc -= cin;
        if (++tdx == 3) { tdx = 0; ++tdy; }
    }
    for (int kc = 0; kc < kpad; kc += 32) {
        V8 a[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            a[m].u = make_uint4(0, 0, 0, 0);
            if (kc + kq < K)
                a[m].u = *reinterpret_cast<const uint4*>(
                    xs + (pbase[m] + tdy * P + tdx) * xstride + cc);
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            V8 bw;
            bw.u = *reinterpret_cast<const uint4*>(wrow + nb * 16 * wstride + kc);
#pragma unroll
            for (int m = 0; m < MT; ++m)
                acc[m][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m].v, bw.v, acc[m][nb],
                                                                     0, 0, 0);
        }
        cc += 32;
        while (cc >= cin) {
            cc -= cin;
            if (++tdx == 3) { tdx = 0; ++tdy; }
        }
    }
}

// A compile-time value, or (0) the runtime one: sizes that are constants in the
// instantiations for the shipped channel counts.
template <int N>
__device__ __forceinline__ int fixed_or(int runtime) { return N > 0 ? N : runtime; }

// The input patch of a workgroup on its way to LDS: vector it = first +
// threadIdx.x + NT*u of the P x P x cin/8 vectors (8 channels of a pixel each),
// u < U, loaded by load() and stored by store(), so that other loads can be
// issued in between.  A vector past the last is that one again, loaded and stored
// where it lies: no branches, so every load is issued before the first store
// waits.  Sources as for stage_patch; POOL: mode1 2.  CIN: channels (0: any).
template <int P, int NT, int U, bool POOL, int CIN>
struct PatchLoad {
    uint4 v[U][POOL ? 4 : 1];
    int px[U], gi[U];  // pixel and 8-channel group
    __device__ __forceinline__ void load(const u16* __restrict__ x1, const u16* __restrict__ x2,
                                         int c1, int c2, int H, int W, int b, int oy, int ox,
                                         int mode1, int first) {
        const int ng = fixed_or<CIN / 8>((c1 + c2) >> 3), last = P * P * ng - 1;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int it = min(first + (int)threadIdx.x + NT * u, last);
            px[u] = it / ng;
            gi[u] = it - px[u] * ng;
            const int ci = gi[u] * 8;
            const bool use2 = !POOL && ci >= c1;  // (a pooled input has no x2)
            const u16* __restrict__ src = use2 ? x2 + (ci - c1) : x1 + ci;
            const int cs = use2 ? c2 : c1;
            const int yc = min(max(oy + px[u] / P, 0), H - 1);
            const int xc = min(max(ox + px[u] % P, 0), W - 1);
            if (POOL) {
                const long long r0 = ((long long)b * (2 * H) + 2 * yc) * (2 * W) + 2 * xc;
                const long long r1 = r0 + 2 * W;
                v[u][0] = *reinterpret_cast<const uint4*>(src + r0 * cs);
                v[u][POOL ? 1 : 0] = *reinterpret_cast<const uint4*>(src + (r0 + 1) * cs);
                v[u][POOL ? 2 : 0] = *reinterpret_cast<const uint4*>(src + r1 * cs);
                v[u][POOL ? 3 : 0] = *reinterpret_cast<const uint4*>(src + (r1 + 1) * cs);
            } else {
                const int up = (!use2 && mode1 == 1) ? 1 : 0;
                const long long q = ((long long)b * (H >> up) + (yc >> up)) * (W >> up) + (xc >> up);
                v[u][0] = *reinterpret_cast<const uint4*>(src + q * cs);
            }
        }
    }
    __device__ __forceinline__ void store(u16* __restrict__ xs, int xstride, int H, int W, int oy,
                                          int ox) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int yy = oy + px[u] / P, xx = ox + px[u] % P;
            const bool in = yy >= 0 && yy < H && xx >= 0 && xx < W;
            V8 o;
            o.u = v[u][0];
            if (POOL) {  // 2x2 average as k_avgpool2 takes it
                V8 p[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) p[e].u = v[u][POOL ? e : 0];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    o.h[e] = to_bf16(0.25f * (from_bf16(p[0].h[e]) + from_bf16(p[1].h[e]) +
                                              from_bf16(p[2].h[e]) + from_bf16(p[3].h[e])));
            }
            o.u = make_uint4(in ? o.u.x : 0, in ? o.u.y : 0, in ? o.u.z : 0, in ? o.u.w : 0);
            *reinterpret_cast<uint4*>(xs + px[u] * xstride + gi[u] * 8) = o.u;
        }
    }
};

// The same for an FP32 gradient g of CIN channels, rounded to BF16 and zeroed where
// mask (NULL: none) is not positive, as stage_grad reads it.
template <int P, int NT, int U, int CIN>
struct GradLoad {
    float4 v0[U], v1[U];
    V8 m[U];
    int px[U], gi[U];
    __device__ __forceinline__ void load(const float* __restrict__ g, const u16* __restrict__ mask,
                                         int H, int W, int b, int oy, int ox) {
        constexpr int ng = CIN / 8;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int it = min((int)threadIdx.x + NT * u, P * P * ng - 1);
            px[u] = it / ng;
            gi[u] = it - px[u] * ng;
            const int yc = min(max(oy + px[u] / P, 0), H - 1);
            const int xc = min(max(ox + px[u] % P, 0), W - 1);
            const long long q = (((long long)b * H + yc) * W + xc) * CIN + gi[u] * 8;
            v0[u] = *reinterpret_cast<const float4*>(g + q);
            v1[u] = *reinterpret_cast<const float4*>(g + q + 4);
            if (mask) m[u].u = *reinterpret_cast<const uint4*>(mask + q);
        }
    }
    __device__ __forceinline__ void store(u16* __restrict__ xs, int H, int W, int oy, int ox,
                                          bool masked) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int yy = oy + px[u] / P, xx = ox + px[u] % P;
            const bool in = yy >= 0 && yy < H && xx >= 0 && xx < W;
            const float gv[8] = {v0[u].x, v0[u].y, v0[u].z, v0[u].w,
                                 v1[u].x, v1[u].y, v1[u].z, v1[u].w};
            V8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bool on = in && !(masked && !(from_bf16(m[u].h[e]) > 0.f));
                o.h[e] = on ? to_bf16(gv[e]) : (u16)0;
            }
            *reinterpret_cast<uint4*>(xs + px[u] * (CIN + 8) + gi[u] * 8) = o.u;
        }
    }
};

// The same for `rows` weight rows of kpad (LDS row stride kpad + 8; KPAD: 0 any).
template <int NT, int U, int KPAD>
struct WeightLoad {
    uint4 v[U];
    __device__ __forceinline__ static int at(int rows, int kv, int first, int u) {
        return min(first + (int)threadIdx.x + NT * u, rows * kv - 1);
    }
    __device__ __forceinline__ void load(const u16* __restrict__ w, int rows, int kpad, int first) {
        const int kv = fixed_or<KPAD / 8>(kpad >> 3);
#pragma unroll
        for (int u = 0; u < U; ++u)  // (rows are contiguous)
            v[u] = reinterpret_cast<const uint4*>(w)[at(rows, kv, first, u)];
    }
    __device__ __forceinline__ void store(u16* __restrict__ ws, int rows, int kpad, int first) {
        const int kv = fixed_or<KPAD / 8>(kpad >> 3);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int it = at(rows, kv, first, u), r = it / kv;
            *reinterpret_cast<uint4*>(ws + r * (kv + 1) * 8 + (it - r * kv) * 8) = v[u];
        }
    }
};

// K of a 3x3 convolution over cin channels, padded to whole chunks
constexpr int conv_kpad(int cin) { return (9 * cin + 31) / 32 * 32; }

// The K loop of conv_lds for NB blocks of 16 output channels (weight rows from
// ws) and MT M-tiles, on a patch of side P.  CIN > 0: unrolled, all offsets
// constants but for the lane's quarter of a chunk, so that the chunks' LDS reads
// and MFMAs have no address chain between them.  CIN 0: conv_lds.  Same chunk
// order, same bits.
template <int CIN, int NB, int MT, int P>
__device__ __forceinline__ void conv_chunks(floatx4 (&acc)[MT][NB], const u16* __restrict__ xs,
                                            int cin, const u16* __restrict__ ws, int kpad,
                                            const int (&pbase)[MT], int lane) {
    if (CIN == 0) {
        conv_lds<NB, MT, P>(acc, xs, cin + 8, cin, ws, kpad, pbase, lane);
        return;
    }
    constexpr int C = CIN > 0 ? CIN : 8, XS = C + 8, KP = conv_kpad(C);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[m][nb] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int qd = lane >> 4;
    const u16* wrow = ws + (lane & 15) * (KP + 8) + 8 * qd;
    const u16* xm[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) xm[m] = xs + pbase[m] * XS;
#pragma unroll
    for (int kc = 0; kc < KP; kc += 32) {
        // patch offset of the lane's 8 consecutive k, one of four constants (past
        // the last tap: anything, the fragment is zeroed)
        auto offset = [&](int k) {
            const int tap = k / C < 9 ? k / C : 0;
            return ((tap / 3) * P + tap % 3) * XS + k % C;
        };
        int off;
        if (C % 32 == 0) {
            off = offset(kc) + 8 * qd;
        } else {
            off = qd == 0 ? offset(kc) : qd == 1 ? offset(kc + 8)
                : qd == 2 ? offset(kc + 16) : offset(kc + 24);
        }
        V8 bw[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
            bw[nb].u = *reinterpret_cast<const uint4*>(wrow + nb * 16 * (KP + 8) + kc);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            V8 a;
            a.u = *reinterpret_cast<const uint4*>(xm[m] + off);
            if (kc + 32 > 9 * C) {
                const bool in = kc + 8 * qd < 9 * C;
                a.u = make_uint4(in ? a.u.x : 0, in ? a.u.y : 0, in ? a.u.z : 0, in ? a.u.w : 0);
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                acc[m][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, bw[nb].v, acc[m][nb],
                                                                     0, 0, 0);
        }
    }
}

// CIN > 0 (mode1 0 or 1): that many input channels; all of the patch's and the
// weights' loads are issued before the first store, the K loop is unrolled.
// At 8 x 128 x 128: 3.1 to 7.1 us a convolution (5.0 to 8.4 staged one after the
// other with a chunk's addresses computed in the K loop).
template <int NB, int OUT, int IN = 0, int CIN = 0>
__global__ __launch_bounds__(256) void k_conv3x3_tile(const u16* __restrict__ x1,
                                                      const u16* __restrict__ x2, int c1, int c2,
                                                      const u16* __restrict__ wt, int kpad, int H,
                                                      int W, int cblocks, u16* __restrict__ ybf,
                                                      float* __restrict__ yf, int cy, int relu,
                                                      int mode1,
                                                      const float* __restrict__ g = nullptr,
                                                      const u16* __restrict__ mask = nullptr,
                                                      float* __restrict__ y2 = nullptr,
                                                      int cy2 = 0) {
    extern __shared__ uint4 tile_lds[];
    u16* xs = reinterpret_cast<u16*>(tile_lds);
    constexpr int KP = CIN > 0 ? conv_kpad(CIN) : 0;
    const int cin = fixed_or<CIN>(c1 + c2);
    const int xstride = cin + 8;                      // u16 per tile pixel
    u16* ws = xs + 100 * xstride;                     // 16-byte aligned: xstride % 8 == 0
    const int cblk = blockIdx.z % cblocks, b = blockIdx.z / cblocks;
    const int tx0 = blockIdx.x * CT, ty0 = blockIdx.y * CT;
    const u16* wb = wt + (size_t)cblk * NB * 16 * kpad;
    if constexpr (CIN > 0) {
        constexpr int UP = (100 * (CIN / 8) + 255) / 256, UW = (NB * 2 * KP + 255) / 256;
        WeightLoad<256, UW, KP> wl;
        if constexpr (IN == 0) {
            PatchLoad<10, 256, UP, false, CIN> pl;
            pl.load(x1, x2, c1, c2, H, W, b, ty0 - 1, tx0 - 1, mode1, 0);
            wl.load(wb, NB * 16, KP, 0);
            pl.store(xs, xstride, H, W, ty0 - 1, tx0 - 1);
        } else {
            GradLoad<10, 256, UP, CIN> gl;
            gl.load(g, mask, H, W, b, ty0 - 1, tx0 - 1);
            wl.load(wb, NB * 16, KP, 0);
            gl.store(xs, H, W, ty0 - 1, tx0 - 1, mask != nullptr);
        }
        wl.store(ws, NB * 16, KP, 0);
    } else {
        if (IN == 0)
            stage_patch<10>(xs, xstride, x1, x2, c1, c2, H, W, b, ty0 - 1, tx0 - 1, mode1);
        else
            stage_grad<10>(xs, xstride, g, mask, c1, H, W, b, ty0 - 1, tx0 - 1);
        stage_weights(ws, wb, NB * 16, kpad);
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // this lane's A pixel: tile row 2*wave + (l%16)/8, column (l%16)%8
    const int ar = 2 * wave + ((lane & 15) >> 3), ac = lane & 7;
    const int pbase[1] = {ar * 10 + ac};
    floatx4 acc2[1][NB];
    conv_chunks<CIN, NB, 1, 10>(acc2, xs, cin, ws, kpad, pbase, lane);
    floatx4(&acc)[NB] = acc2[0];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // D row 4*(l/16) + r is tile pixel (2*wave + row/8, row % 8)
            const int row = 4 * (lane >> 4) + r;
            const int yy = ty0 + 2 * wave + (row >> 3), xx = tx0 + (row & 7);
            const int ch = (cblk * NB + nb) * 16 + (lane & 15);
            if (yy >= H || xx >= W || ch >= cy + (OUT == 2 ? cy2 : 0)) continue;
            const long long p = ((long long)b * H + yy) * W + xx;
            float v = acc[nb][r];
            if (OUT == 0) {
                if (relu) v = fmaxf(v, 0.f);
                ybf[p * cy + ch] = to_bf16(v);
            } else if (OUT == 1 || ch < cy) {
                yf[p * cy + ch] = v;
            } else {
                y2[p * cy2 + ch - cy] = v;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Two consecutive 3x3 convolutions of one resolution level in one launch
// (inference), one 8x8 output tile per workgroup of 8 waves: conv a reads its
// inputs as k_conv3x3_tile does (mode1; POOL: mode 2) on the 12x12 patch around
// the tile and computes the 10x10 region that conv b needs (7 M-tiles of 16
// pixels), which stays in LDS as BF16 (zero outside the image: conv b's padding);
// conv b then computes the tile from it.  Every workgroup computes all output
// channels of both convs (NB*16).  The A/B fragments and the K order of both are
// those of k_conv3x3_tile, and the intermediate is rounded to BF16 as the stored
// tensor is, so the output is bit-identical to the two launches; conv a's output
// is not written.  wb_early: conv b's weights are staged with conv a's at the
// start (separate LDS); else after conv a, over conv a's.
//
// Bound by latency: launch, one memory round trip, two short K loops.  The
// patch's and both convolutions' weight loads are all issued before the first
// LDS store (three round trips one after the other before), 8 waves share the
// M-tiles by output block, and the K loops are unrolled for the chunk counts of
// the shipped networks (CINA, CINB channels; 0: any): with the sizes at run time
// the compiler put every weight load behind its predicate, next to its store, and
// a division per chunk in front of the K loop.  On a 128 x 128 level 0, median of
// a launch (8 -> 16, 16 -> 32 pooled, 32 -> 32 pooled, 64 -> 32, 48 -> 16
// channels): 9.6, 11.7, 11.7, 11.7, 9.6 us before, 4.4, 6.0, 6.4, 7.3, 4.7 now.
// grid: (ceil(W/8), ceil(H/8), B).  LDS (u16): 144 (cin + 8) + 100 (cya + 8) +
// NB*16 (kpada + 8) [+ NB*16 (kpadb + 8)], or max of the two weight blocks.
// ---------------------------------------------------------------------------
constexpr int kPairThreads = 512;
template <int NB, int CINA, int CINB, bool POOL>
__global__ __launch_bounds__(kPairThreads) void k_conv_pair_tile(
    const u16* __restrict__ x1, const u16* __restrict__ x2, int c1, int c2,
    const u16* __restrict__ wa, int kpada, int cya, int relua, const u16* __restrict__ wb,
    int kpadb, int cyb, int relub, u16* __restrict__ ybf, int H, int W, int mode1,
    int wb_early) {
    constexpr int NT = kPairThreads;
    constexpr int KPA = CINA > 0 ? conv_kpad(CINA) : 0, KPB = CINB > 0 ? conv_kpad(CINB) : 0;
    // vectors per thread of a round: all of them where the sizes are constants
    constexpr int UP = CINA > 0 ? (144 * (CINA / 8) + NT - 1) / NT : 2;
    constexpr int UA = CINA > 0 ? (NB * 2 * KPA + NT - 1) / NT : 4;
    constexpr int UB = CINB > 0 ? (NB * 2 * KPB + NT - 1) / NT : 2;
    extern __shared__ uint4 tile_lds[];
    const int cin = fixed_or<CINA>(c1 + c2), cb = fixed_or<CINB>(cya);
    const int ka = fixed_or<KPA>(kpada), kb = fixed_or<KPB>(kpadb);
    const int xstride = cin + 8, istride = cb + 8;
    u16* xs = reinterpret_cast<u16*>(tile_lds);
    u16* ism = xs + 144 * xstride;
    u16* wsa = ism + 100 * istride;
    u16* wsb = wb_early ? wsa + NB * 16 * (ka + 8) : wsa;
    const int b = blockIdx.z;
    const int tx0 = blockIdx.x * CT, ty0 = blockIdx.y * CT;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    {
        PatchLoad<12, NT, UP, POOL, CINA> pl;
        WeightLoad<NT, UA, KPA> la;
        WeightLoad<NT, UB, KPB> lb;
        pl.load(x1, x2, c1, c2, H, W, b, ty0 - 2, tx0 - 2, mode1, 0);
        la.load(wa, NB * 16, ka, 0);
        lb.load(wb, NB * 16, kb, 0);
        pl.store(xs, xstride, H, W, ty0 - 2, tx0 - 2);
        la.store(wsa, NB * 16, ka, 0);
        if (wb_early) lb.store(wsb, NB * 16, kb, 0);
        // what did not fit the first round
        for (int f = UP * NT; CINA == 0 && f < 18 * cin; f += UP * NT) {
            pl.load(x1, x2, c1, c2, H, W, b, ty0 - 2, tx0 - 2, mode1, f);
            pl.store(xs, xstride, H, W, ty0 - 2, tx0 - 2);
        }
        for (int f = UA * NT; CINA == 0 && f < NB * 2 * ka; f += UA * NT) {
            la.load(wa, NB * 16, ka, f);
            la.store(wsa, NB * 16, ka, f);
        }
        for (int f = UB * NT; CINB == 0 && wb_early && f < NB * 2 * kb; f += UB * NT) {
            lb.load(wb, NB * 16, kb, f);
            lb.store(wsb, NB * 16, kb, f);
        }
    }
    __syncthreads();
    // wave -> output block nb and M-tiles: with two blocks each wave takes two
    // M-tiles of conv a and one of conv b, with one block one of each
    const int nb = NB == 2 ? wave & 1 : 0, mg = NB == 2 ? wave >> 1 : wave;
    const int ch = nb * 16 + (lane & 15);
    {
        // (pixels past 100 compute on pixel 0 and are dropped)
        constexpr int MT = NB == 2 ? 2 : 1;
        int pbase[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int q = (mg + 4 * m) * 16 + (lane & 15);
            pbase[m] = q < 100 ? (q / 10) * 12 + q % 10 : 0;
        }
        floatx4 acc[MT][1];
        conv_chunks<CINA, 1, MT, 12>(acc, xs, cin, wsa + nb * 16 * (ka + 8), ka, pbase, lane);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int q = (mg + 4 * m) * 16 + 4 * (lane >> 4) + r;
                if (q >= 100 || ch >= cya) continue;
                const int yy = ty0 - 1 + q / 10, xx = tx0 - 1 + q % 10;
                float v = acc[m][0][r];
                if (relua) v = fmaxf(v, 0.f);
                ism[q * istride + ch] =
                    (yy >= 0 && yy < H && xx >= 0 && xx < W) ? to_bf16(v) : (u16)0;
            }
    }
    __syncthreads();
    if (!wb_early) {
        WeightLoad<NT, UB, KPB> lb;
        for (int f = 0; f < NB * 2 * kb; f += UB * NT) {
            lb.load(wb, NB * 16, kb, f);
            lb.store(wsb, NB * 16, kb, f);
        }
        __syncthreads();
    }
    if (mg >= 4) return;  // conv b has four M-tiles
    // lane's A pixel: tile row 2*mg + (l%16)/8, column (l%16)%8, i.e. region pixel
    // (row + 1, column + 1) whose 3x3 neighbourhood starts at index row*10 + column
    const int ar = 2 * mg + ((lane & 15) >> 3), ac = lane & 7;
    const int pbase[1] = {ar * 10 + ac};
    floatx4 acc[1][1];
    conv_chunks<CINB, 1, 1, 10>(acc, ism, cb, wsb + nb * 16 * (kb + 8), kb, pbase, lane);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 4 * (lane >> 4) + r;
        const int yy = ty0 + 2 * mg + (row >> 3), xx = tx0 + (row & 7);
        if (yy >= H || xx >= W || ch >= cyb) continue;
        const long long p = ((long long)b * H + yy) * W + xx;
        float v = acc[0][0][r];
        if (relub) v = fmaxf(v, 0.f);
        ybf[p * cyb + ch] = to_bf16(v);
    }
}

// ---------------------------------------------------------------------------
// Weight gradient dW[co][tap*cin + ci] += sum_p gm[p][co] * x[p + tap][ci],
// gm = g*(mask>0), x the (concatenated) input, zero outside the image: MFMA with
// M = output channels, N = input channels of one tap, K = pixels.
//
// A workgroup (4 waves) stages an 8 x 32 pixel tile in LDS, channel-major so
// that a fragment's 8 consecutive pixels of a row are 16 contiguous bytes: the
// gradient of NCO*16 output channels rounded to BF16, and the input of NCI*16
// channels with a one-pixel rim, its columns shifted by one so that tap dx = 0
// starts aligned.  One 16-byte and one 4-byte read per input row then give the
// fragments of all three dx (dx = 2 is the same words one dword on, dx = 1 a
// 16-bit funnel shift).  Wave w takes 16 input channels (w % NCI), all 9 taps and
// all NCO blocks, and every (4 / NCI)-th group of 4 x 8 pixels.  The waves'
// sums meet in LDS, each wave sums a share of the entries over them, and go out
// with FP32 atomics, one set per workgroup, after as many tiles as the grid leaves
// it.
//
// Bound by the staging's LDS stores and loads (each input pixel is read once
// per 32 output channels).  Gathering each fragment from global memory, element
// by element with a division per pixel, took 97 us per convolution at 8 x 128 x
// 128 (18 of them, 1.75 of the 2.16 ms of a training gradient); 8 to 18 us
// now (with one wave summing and adding for all, and branches around the loads, 9
// to 21).
// grid: (workgroups over the tiles, ceil(cin / (16 NCI)), ceil(cg / (16 NCO))).
// ---------------------------------------------------------------------------
constexpr int WG_TR = 8, WG_TC = 32;             // tile rows, columns
constexpr int WG_XROW = (WG_TC + 8) / 2;         // dwords per staged input row
// dwords per channel, multiples of 4 with 8 channels' starts on distinct banks
constexpr int WG_XCH = (WG_TR + 2) * WG_XROW + 4;
constexpr int WG_GCH = WG_TR * WG_TC / 2 + 4;

template <int NCI, int NCO>
__global__ __launch_bounds__(256) void k_wgrad(const u16* __restrict__ x1,
                                               const u16* __restrict__ x2, int c1, int c2,
                                               const float* __restrict__ g,
                                               const u16* __restrict__ mask, int cg, int B,
                                               int H, int W, float* __restrict__ dw, int kpad,
                                               int tiles_x, int tiles_y) {
    constexpr int KP = 4 / NCI;    // waves sharing 16 input channels
    constexpr int XG = 2 * NCI;    // groups of 8 input channels
    constexpr int XDW = NCI * 16 * WG_XCH + XG * 4, GDW = NCO * 16 * WG_GCH;
    constexpr int RDW = 4 * 36 * 64;  // the waves' sums of 16 output channels
    __shared__ __align__(16) unsigned lds[XDW + GDW > RDW ? XDW + GDW : RDW];
    unsigned* xs = lds;
    unsigned* gs = lds + XDW;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cb = wave % NCI, kpart = wave / NCI;
    const int cin = c1 + c2;
    const int ci0 = blockIdx.y * NCI * 16, co0 = blockIdx.z * NCO * 16;
    floatx4 acc[9][NCO];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int m = 0; m < NCO; ++m) acc[t][m] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int ntiles = tiles_x * tiles_y * B;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int tx = tile % tiles_x, ty = (tile / tiles_x) % tiles_y, b = tile / (tiles_x * tiles_y);
        const int xo = tx * WG_TC, yo = ty * WG_TR;
        const long long img = (long long)b * H * W;
        __syncthreads();  // the previous tile has been read
        // all of a thread's loads are issued before its first LDS store
        constexpr int XN = (WG_TR + 2) * (WG_TC / 2 + 1) * XG, XIT = (XN + 255) / 256;
        constexpr int GN = WG_TR * (WG_TC / 2) * 4 * NCO, GIT = GN / 256;
        static_assert(GN % 256 == 0, "whole rounds");
        V8 xv[XIT][2];
        float4 gv[GIT][2];
        ushort4 mv[GIT][2];
#pragma unroll
        for (int u = 0; u < XIT; ++u) {
            const int it = threadIdx.x + 256 * u;
            const int gi = it % XG, t = it / XG;
            const int pair = t % (WG_TC / 2 + 1), row = t / (WG_TC / 2 + 1);
            // (clamped addresses, no branches: channels past cin read the last ones)
            const int ci = min(ci0 + gi * 8, cin - 8), yy = yo + row - 1, xx = xo + 2 * pair - 1;
            const bool use2 = ci >= c1;
            const u16* src = use2 ? x2 + (ci - c1) : x1 + ci;
            const int cs = use2 ? c2 : c1;
            const long long r0 = img + (long long)min(max(yy, 0), H - 1) * W;
#pragma unroll
            for (int e = 0; e < 2; ++e)
                xv[u][e].u = *reinterpret_cast<const uint4*>(
                    src + (r0 + min(max(xx + e, 0), W - 1)) * cs);
        }
#pragma unroll
        for (int u = 0; u < GIT; ++u) {
            const int it = threadIdx.x + 256 * u;
            const int q = it % (4 * NCO), t = it / (4 * NCO);
            const int pair = t % (WG_TC / 2), row = t / (WG_TC / 2);
            const int co = min(co0 + 4 * q, cg - 4), yy = min(yo + row, H - 1), xx = xo + 2 * pair;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const long long p = (img + (long long)yy * W + min(xx + e, W - 1)) * cg + co;
                gv[u][e] = *reinterpret_cast<const float4*>(g + p);
                mv[u][e] = make_ushort4(0x3f80, 0x3f80, 0x3f80, 0x3f80);  // 1.0: not masked
                if (mask) mv[u][e] = *reinterpret_cast<const ushort4*>(mask + p);
            }
        }
#pragma unroll
        for (int u = 0; u < XIT; ++u) {
            const int it = threadIdx.x + 256 * u;
            const int gi = it % XG, t = it / XG;
            const int pair = t % (WG_TC / 2 + 1), row = t / (WG_TC / 2 + 1);
            if (it >= XN) continue;
            const int yy = yo + row - 1, xx = xo + 2 * pair - 1;
            const bool rok = ci0 + gi * 8 < cin && yy >= 0 && yy < H;
            const unsigned lo = rok && xx >= 0 && xx < W ? 0xffffu : 0u;
            const unsigned hi = rok && xx + 1 >= 0 && xx + 1 < W ? 0xffff0000u : 0u;
            unsigned* dst = xs + gi * (8 * WG_XCH + 4) + row * WG_XROW + pair;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                dst[e * WG_XCH] = ((unsigned)xv[u][0].h[e] & lo) | (((unsigned)xv[u][1].h[e] << 16) & hi);
        }
#pragma unroll
        for (int u = 0; u < GIT; ++u) {
            const int it = threadIdx.x + 256 * u;
            const int q = it % (4 * NCO), t = it / (4 * NCO);
            const int pair = t % (WG_TC / 2), row = t / (WG_TC / 2);
            unsigned o[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const bool in = co0 + 4 * q < cg && yo + row < H && xo + 2 * pair + e < W;
                const float f[4] = {gv[u][e].x, gv[u][e].y, gv[u][e].z, gv[u][e].w};
                const u16 m[4] = {mv[u][e].x, mv[u][e].y, mv[u][e].z, mv[u][e].w};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    o[k] |= in && from_bf16(m[k]) > 0.f ? (unsigned)to_bf16(f[k]) << (16 * e) : 0u;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) gs[(4 * q + k) * WG_GCH + row * (WG_TC / 2) + pair] = o[k];
        }
        __syncthreads();
        // this lane's channel of the input block
        const int ch = cb * 16 + (lane & 15);
        const unsigned* xc = xs + ch * WG_XCH + (ch >> 3) * 4;
        const unsigned* gc = gs + (lane & 15) * WG_GCH;
        for (int ks = kpart; ks < (WG_TR / 4) * (WG_TC / 8); ks += KP) {
            const int row = (ks / (WG_TC / 8)) * 4 + (lane >> 4), col = (ks % (WG_TC / 8)) * 4;
            V8 a[NCO];
#pragma unroll
            for (int m = 0; m < NCO; ++m)
                a[m].u = *reinterpret_cast<const uint4*>(gc + m * 16 * WG_GCH + row * (WG_TC / 2) + col);
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
                const unsigned* xr = xc + (row + dy) * WG_XROW + col;
                const uint4 d = *reinterpret_cast<const uint4*>(xr);
                const unsigned d4 = xr[4];
                V8 bx[3];
                bx[0].u = d;
                bx[1].u = make_uint4(__builtin_amdgcn_alignbit(d.y, d.x, 16),
                                     __builtin_amdgcn_alignbit(d.z, d.y, 16),
                                     __builtin_amdgcn_alignbit(d.w, d.z, 16),
                                     __builtin_amdgcn_alignbit(d4, d.w, 16));
                bx[2].u = make_uint4(d.y, d.z, d.w, d4);
#pragma unroll
                for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                    for (int m = 0; m < NCO; ++m)
                        acc[3 * dy + dx][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            a[m].v, bx[dx].v, acc[3 * dy + dx][m], 0, 0, 0);
            }
        }
    }
    // sum over the waves of an input block: all waves leave theirs, each then
    // sums and adds its share of the entries
    const int ci = ci0 + cb * 16 + (lane & 15);
    float* red = reinterpret_cast<float*>(lds) + lane;
#pragma unroll
    for (int m = 0; m < NCO; ++m) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 36; ++e) red[(wave * 36 + e) * 64] = acc[e / 4][m][e % 4];
        __syncthreads();
        for (int i = 0; i < 36 / KP; ++i) {
            const int e = kpart * (36 / KP) + i;
            float v = red[(cb * 36 + e) * 64];
#pragma unroll
            for (int k = 1; k < KP; ++k) v += red[((cb + NCI * k) * 36 + e) * 64];
            const int co = co0 + m * 16 + 4 * (lane >> 4) + e % 4;  // output channel row of D
            if (ci < cin && co < cg) atomicAdd(dw + (size_t)co * kpad + (e / 4) * cin + ci, v);
        }
    }
}

// ---- elementwise / pooling ---------------------------------------------------
__global__ void k_prep_input(const float* __restrict__ x, u16* __restrict__ x8, long long npix) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npix) return;
    V8 v;
    v.u = make_uint4(0, 0, 0, 0);
    v.h[0] = to_bf16(x[p]);
    *reinterpret_cast<uint4*>(x8 + p * 8) = v.u;
}

// normalised coarse residual -> 8-channel BF16 network input: x = (rc - mean)
// / rms from stats = (sum, sum^2) over n cells (the solver's coarse residual)
__global__ void k_prep_normalized(const float* __restrict__ rc, const double* __restrict__ stats,
                                  int n, u16* __restrict__ x8) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const double mean = stats[0] / n;
    const double var = stats[1] / n - mean * mean;
    const double sig = sqrt(var > 1e-300 ? var : 1e-300);
    V8 v;
    v.u = make_uint4(0, 0, 0, 0);
    v.h[0] = to_bf16((float)(((double)rc[p] - mean) / sig));
    *reinterpret_cast<uint4*>(x8 + (long long)p * 8) = v.u;
}

// The 2x resampling of channel-last tensors and its adjoints: one thread per 16
// bytes of a pixel's channels (C a multiple of 8), grid x over a row, grid y over
// the rows of all images.  Bound by memory; one element per thread with 64-bit
// divisions took 15.7 us for the largest upsampling at 8 x 128 x 128 (8.7 and 6.4
// the adjoints), 4.6 now (5.5 and 5.2); a training gradient 525 -> 490 us.
dim3 resample_grid(long long rows, long long items) {
    return dim3(div_up(items, 256), (unsigned)std::min<long long>(rows, 65535));
}

__global__ __launch_bounds__(256) void k_avgpool2(const u16* __restrict__ x, u16* __restrict__ y,
                                                  int B, int H, int W, int C) {
    const int Ho = H / 2, Wo = W / 2, ng = C / 8;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= Wo * ng) return;
    const int xo = i / ng, c = (i - xo * ng) * 8;
    for (int row = blockIdx.y; row < B * Ho; row += gridDim.y) {
        const int b = row / Ho, yo = row - b * Ho;
        const u16* p = x + (((long long)b * H + 2 * yo) * W + 2 * xo) * C + c;
        V8 v[4], o;
        v[0].u = *reinterpret_cast<const uint4*>(p);
        v[1].u = *reinterpret_cast<const uint4*>(p + C);
        v[2].u = *reinterpret_cast<const uint4*>(p + (long long)W * C);
        v[3].u = *reinterpret_cast<const uint4*>(p + (long long)W * C + C);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            o.h[e] = to_bf16(0.25f * (from_bf16(v[0].h[e]) + from_bf16(v[1].h[e]) +
                                      from_bf16(v[2].h[e]) + from_bf16(v[3].h[e])));
        *reinterpret_cast<uint4*>(y + ((long long)row * Wo + xo) * C + c) = o.u;
    }
}

// dx[fine] += dy[coarse] / 4
__global__ __launch_bounds__(256) void k_avgpool2_bwd(const float* __restrict__ dy,
                                                      float* __restrict__ dx, int B, int H, int W,
                                                      int C) {
    const int ng = C / 4;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= W * ng) return;
    const int xx = i / ng, c = (i - xx * ng) * 4;
    for (int row = blockIdx.y; row < B * H; row += gridDim.y) {
        const int b = row / H, yy = row - b * H;
        float4* p = reinterpret_cast<float4*>(dx + ((long long)row * W + xx) * C + c);
        const float4 d = *reinterpret_cast<const float4*>(
            dy + (((long long)b * (H / 2) + yy / 2) * (W / 2) + xx / 2) * C + c);
        float4 v = *p;
        v.x += 0.25f * d.x;
        v.y += 0.25f * d.y;
        v.z += 0.25f * d.z;
        v.w += 0.25f * d.w;
        *p = v;
    }
}

// nearest 2x upsampling of x [B][H/2][W/2][C] to y [B][H][W][C]
__global__ __launch_bounds__(256) void k_upsample2(const u16* __restrict__ x, u16* __restrict__ y,
                                                   int B, int H, int W, int C) {
    const int ng = C / 8;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= W * ng) return;
    const int xx = i / ng, c = (i - xx * ng) * 8;
    for (int row = blockIdx.y; row < B * H; row += gridDim.y) {
        const int b = row / H, yy = row - b * H;
        *reinterpret_cast<uint4*>(y + ((long long)row * W + xx) * C + c) =
            *reinterpret_cast<const uint4*>(
                x + (((long long)b * (H / 2) + yy / 2) * (W / 2) + xx / 2) * C + c);
    }
}

// dx[coarse] = sum of the 4 fine gradients
__global__ __launch_bounds__(256) void k_upsample2_bwd(const float* __restrict__ dy,
                                                       float* __restrict__ dx, int B, int H, int W,
                                                       int C) {
    const int Ho = H / 2, Wo = W / 2, ng = C / 4;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= Wo * ng) return;
    const int xo = i / ng, c = (i - xo * ng) * 4;
    for (int row = blockIdx.y; row < B * Ho; row += gridDim.y) {
        const int b = row / Ho, yo = row - b * Ho;
        const float* p = dy + (((long long)b * H + 2 * yo) * W + 2 * xo) * C + c;
        const float4 v0 = *reinterpret_cast<const float4*>(p);
        const float4 v1 = *reinterpret_cast<const float4*>(p + C);
        const float4 v2 = *reinterpret_cast<const float4*>(p + (long long)W * C);
        const float4 v3 = *reinterpret_cast<const float4*>(p + (long long)W * C + C);
        *reinterpret_cast<float4*>(dx + ((long long)row * Wo + xo) * C + c) =
            make_float4(v0.x + v1.x + v2.x + v3.x, v0.y + v1.y + v2.y + v3.y,
                        v0.z + v1.z + v2.z + v3.z, v0.w + v1.w + v2.w + v3.w);
    }
}

// supervised loss on the output y (FP32 [npix]): partial sums of (y - t)^2
// and dL/dy = 2 (y - t) / npix
__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ y, const float* __restrict__ t,
                                              float* __restrict__ gy, long long npix,
                                              double* __restrict__ partials) {
    __shared__ double smem[16];
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double e2 = 0.0;
    if (p < npix) {
        const float d = y[p] - t[p];
        e2 = (double)d * d;
        if (gy) gy[p] = 2.f * d / (float)npix;
    }
    const double s = cd_block_sum(e2, smem);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// Neumann 5-point operator (sum of in-grid neighbours - count * centre) of a
// [B][H][W] field with element stride `stride`
__device__ __forceinline__ float lap_field(const float* __restrict__ v, int stride, long long p,
                                           int x, int y, int H, int W) {
    const float c = v[p * stride];
    float s = 0.f, cnt = 0.f;
    if (x > 0) { s += v[(p - 1) * stride]; cnt += 1.f; }
    if (x < W - 1) { s += v[(p + 1) * stride]; cnt += 1.f; }
    if (y > 0) { s += v[(p - W) * stride]; cnt += 1.f; }
    if (y < H - 1) { s += v[(p + W) * stride]; cnt += 1.f; }
    return s - cnt * c;
}

// out = in + Lc(in) / 8: one symmetric smoothing step (gain 1 - lambda/8 on
// the operator's eigenvalue lambda in [0, 8]); used on the network output and
// to weight the operator loss towards the frequencies the fine smoother
// cannot reach
__global__ __launch_bounds__(256) void k_smooth_step(const float* __restrict__ in,
                                                     float* __restrict__ out, int B, int H, int W) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (long long)B * H * W) return;
    const int xx = (int)(p % W), yy = (int)((p / W) % H);
    out[p] = in[p] + 0.125f * lap_field(in, 1, p, xx, yy, H, W);
}

// k smoothing steps in one launch: an 8x8 output tile with a k-cell halo, the
// (8 + 2k)^2 region, lives in LDS (two buffers), one cell per thread; step st
// updates the cells at distance >= st from the region's border, so the tile
// equals k global steps.  Cells outside the image stay 0, so that adding them
// changes no sum and a cell's count of neighbours is the only condition left.
// Same arithmetic and summation order as k_smooth_step (bit-identical).
// 8x8 tiles: 256 workgroups at 128x128 (16x16 tiles took 1.6 times as long).
constexpr int kSmoothTile = 8;
constexpr int kSmoothMaxK = 12;  // (8 + 2k)^2 <= 1024 threads
// K: the number of steps (0: k).  a holds the region of image origin (X0, Y0), b is
// scratch of the same size; the calls of all threads of the workgroup meet.
// Returns whether this thread's cell (gx, gy) is one of the tile, with its value.
template <int K>
__device__ __forceinline__ bool smooth_region(float* a, float* b, int k, int X0, int Y0, int H,
                                              int W, int& gx, int& gy, float& c) {
    const int steps = K > 0 ? K : k, R = kSmoothTile + 2 * steps, NQ = R * R;
    const int q = min((int)threadIdx.x, NQ - 1), ry = q / R, rx = q - ry * R;
    gy = Y0 + ry;
    gx = X0 + rx;
    const bool inside = gx >= 0 && gx < W && gy >= 0 && gy < H;
    // steps that update this cell: those below its distance to the region's edge
    const int depth = inside ? min(min(rx, R - 1 - rx), min(ry, R - 1 - ry)) : 0;
    const float cnt = (float)((gx > 0) + (gx < W - 1) + (gy > 0) + (gy < H - 1));
    const int ql = max(q - 1, 0), qr = min(q + 1, NQ - 1), qu = max(q - R, 0),
              qd = min(q + R, NQ - 1);
    c = a[q];
#pragma unroll
    for (int st = 1; st <= steps; ++st) {
        const float* src = st & 1 ? a : b;
        float sum = 0.f;
        sum += src[ql];
        sum += src[qr];
        sum += src[qu];
        sum += src[qd];
        c = st <= depth ? c + 0.125f * (sum - cnt * c) : c;
        if (st < steps) {
            (st & 1 ? b : a)[q] = c;  // (threads past the region: the last cell's value)
            __syncthreads();
        }
    }
    return inside && depth >= steps && (int)threadIdx.x < NQ;
}

// k smoothing steps of a field read with element stride istride (8: head
// channel 0), one tile plus its k-cell halo per workgroup of (8 + 2k)^2 threads
// (rounded up to whole waves).  At 8 x 128 x 128, k = 6: 11.3 us with two cells a
// thread and the image's bounds tested in every step, 7.7 us now.
__global__ __launch_bounds__(1024) void k_smooth_tiled(const float* __restrict__ in, int istride,
                                                       float* __restrict__ out, int B, int H,
                                                       int W, int k) {
    extern __shared__ float lds[];
    const int R = kSmoothTile + 2 * k, RR = R * R;
    const int bz = blockIdx.z;
    const int X0 = blockIdx.x * kSmoothTile - k, Y0 = blockIdx.y * kSmoothTile - k;
    const long long base = (long long)bz * H * W;
    const int q = min((int)threadIdx.x, RR - 1);
    const int gx0 = X0 + q % R, gy0 = Y0 + q / R;
    const float v = in[(base + (long long)min(max(gy0, 0), H - 1) * W + min(max(gx0, 0), W - 1)) *
                       istride];
    lds[q] = gx0 >= 0 && gx0 < W && gy0 >= 0 && gy0 < H ? v : 0.f;
    __syncthreads();
    int gx, gy;
    float c;
    if (smooth_region<0>(lds, lds + RR, k, X0, Y0, H, W, gx, gy, c))
        out[base + (long long)gy * W + gx] = c;
}

// Head convolution and output smoothing in one launch (inference, K steps):
// the head (16 output channels of which channel 0 is the output, no ReLU) on
// the (8 + 2K)^2 region around an 8x8 tile, read from a (10 + 2K)^2 input
// patch in LDS with the A/B fragments and K order of k_conv3x3_tile, so its
// values are those k_conv3x3_tile<1, 1> stores; outside the image the region
// holds 0, as k_smooth_tiled loads it; then the K steps as k_smooth_tiled
// takes them.  The output is bit-identical to the two launches.
//
// Bound by latency, as k_conv_pair_tile, and built like it (loads first, CIN > 0
// unrolled for that many channels, 8 waves).  On a 128 x 128 level, 16 channels:
// 11.2 us with 256 threads, a serial staging and bounds tested in every smoothing
// step, 5.5 us now.
// grid (ceil(W/8), ceil(H/8), B); LDS (bytes): 2 P^2 (C + 8) + 2*16 (kpad + 8)
// + 8 R^2, P = R + 2, R = 8 + 2K.
template <int K, int CIN>
__global__ __launch_bounds__(512) void k_head_smooth(const u16* __restrict__ x, int channels,
                                                     const u16* __restrict__ wt, int kpad0, int H,
                                                     int W, float* __restrict__ out) {
    constexpr int NT = 512;
    constexpr int R = kSmoothTile + 2 * K, P = R + 2, NQ = R * R;
    constexpr int MT = (NQ + NT / 4 - 1) / (NT / 4);  // M-tiles of 16 region pixels per wave
    constexpr int KP = CIN > 0 ? conv_kpad(CIN) : 0;
    constexpr int UP = CIN > 0 ? (P * P * (CIN / 8) + NT - 1) / NT : 2;
    constexpr int UW = CIN > 0 ? (2 * KP + NT - 1) / NT : 1;
    static_assert(kSmoothTile == CT, "the head region is centred on the conv tile");
    static_assert(NQ <= NT, "one region cell per thread");
    extern __shared__ uint4 tile_lds[];
    const int C = fixed_or<CIN>(channels), kpad = fixed_or<KP>(kpad0);
    const int xstride = C + 8;
    u16* xs = reinterpret_cast<u16*>(tile_lds);
    u16* ws = xs + P * P * xstride;
    float* a = reinterpret_cast<float*>(ws + 16 * (kpad + 8));
    float* b2 = a + NQ;
    const int b = blockIdx.z;
    const int tx0 = blockIdx.x * CT, ty0 = blockIdx.y * CT;
    const int X0 = tx0 - K, Y0 = ty0 - K;  // region origin
    {
        // (x2 = x with no channels: never read)
        PatchLoad<P, NT, UP, false, CIN> pl;
        WeightLoad<NT, UW, KP> wl;
        pl.load(x, x, C, 0, H, W, b, Y0 - 1, X0 - 1, 0, 0);
        wl.load(wt, 16, kpad, 0);
        pl.store(xs, xstride, H, W, Y0 - 1, X0 - 1);
        wl.store(ws, 16, kpad, 0);
        for (int f = UP * NT; CIN == 0 && f < P * P * (C / 8); f += UP * NT) {
            pl.load(x, x, C, 0, H, W, b, Y0 - 1, X0 - 1, 0, f);
            pl.store(xs, xstride, H, W, Y0 - 1, X0 - 1);
        }
        for (int f = UW * NT; CIN == 0 && f < 2 * kpad; f += UW * NT) {
            wl.load(wt, 16, kpad, f);
            wl.store(ws, 16, kpad, f);
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int pbase[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int q = (wave + 8 * m) * 16 + (lane & 15);
        pbase[m] = q < NQ ? (q / R) * P + q % R : 0;
    }
    floatx4 acc[MT][1];
    conv_chunks<CIN, 1, MT, P>(acc, xs, C, ws, kpad, pbase, lane);
    if ((lane & 15) == 0) {  // output channel 0
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int q = (wave + 8 * m) * 16 + 4 * (lane >> 4) + r;
                if (q >= NQ) continue;
                const int gy = Y0 + q / R, gx = X0 + q % R;
                a[q] = (gy >= 0 && gy < H && gx >= 0 && gx < W) ? acc[m][0][r] : 0.f;
            }
    }
    __syncthreads();
    int gx, gy;
    float c;
    if (smooth_region<K>(a, b2, K, X0, Y0, H, W, gx, gy, c))
        out[((long long)b * H + gy) * W + gx] = c;
}

// operator residual u = cs * Lc y - x
__global__ __launch_bounds__(256) void k_op_residual(const float* __restrict__ y,
                                                     const float* __restrict__ x,
                                                     float* __restrict__ u, int B, int H, int W,
                                                     float cs) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (long long)B * H * W) return;
    const int xx = (int)(p % W), yy = (int)((p / W) % H);
    u[p] = cs * lap_field(y, 1, p, xx, yy, H, W) - x[p];
}

// partial sums of v^2; dv = (2 / npix) v in place when want_grad
__global__ __launch_bounds__(256) void k_sumsq(float* __restrict__ v, long long npix, int want_grad,
                                               double* __restrict__ partials) {
    __shared__ double smem[16];
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double e2 = 0.0;
    if (p < npix) {
        e2 = (double)v[p] * v[p];
        if (want_grad) v[p] = 2.f * v[p] / (float)npix;
    }
    const double s = cd_block_sum(e2, smem);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// energy loss per pixel: with u = cs Lc y - x, J = y'(-cs Lc)y/2 + x'y has
// pixel contributions y (x - u) / 2 and dJ/dy = -u; partial sums of the
// contributions, gy = -u / npix when want_grad
__global__ __launch_bounds__(256) void k_energy(const float* __restrict__ y,
                                                const float* __restrict__ x,
                                                const float* __restrict__ u,
                                                float* __restrict__ gy, long long npix,
                                                int want_grad, double* __restrict__ partials) {
    __shared__ double smem[16];
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double e = 0.0;
    if (p < npix) {
        e = 0.5 * (double)y[p] * ((double)x[p] - (double)u[p]);
        if (want_grad) gy[p] = -u[p] / (float)npix;
    }
    const double s = cd_block_sum(e, smem);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// gy = cs * Lc du (Lc symmetric)
__global__ __launch_bounds__(256) void k_op_grad(const float* __restrict__ du,
                                                 float* __restrict__ gy, int B, int H, int W,
                                                 float cs) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (long long)B * H * W) return;
    const int xx = (int)(p % W), yy = (int)((p / W) % H);
    gy[p] = cs * lap_field(du, 1, p, xx, yy, H, W);
}

// head channel 0 -> y (stride 8 -> 1), and dL/dy -> head gradient
__global__ void k_head_out(const float* __restrict__ head, float* __restrict__ y, long long npix) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < npix) y[p] = head[p * 8];
}
__global__ void k_head_grad(const float* __restrict__ gy, float* __restrict__ ghead,
                            long long npix) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npix) return;
    ghead[p * 8] = gy[p];
#pragma unroll
    for (int c = 1; c < 8; ++c) ghead[p * 8 + c] = 0.f;
}

// FP32 master -> BF16 forward weights [coutpad][kpad] (same layout)
__global__ void k_cast_bf16(const float* __restrict__ w, u16* __restrict__ o, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) o[i] = to_bf16(w[i]);
}

// transposed, tap-flipped BF16 weights for the input gradient:
// wt[ci][tap' * coutA + co] = w[co][(8 - tap') * cin + ci]
__global__ void k_transpose_w(const float* __restrict__ w, u16* __restrict__ wt, int cout, int coutA,
                              int cin, int kpad, int cinpad, int kpadT) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)cinpad * kpadT) return;
    const int ci = (int)(i / kpadT);
    const int kk = (int)(i - (long long)ci * kpadT);
    float v = 0.f;
    if (ci < cin && kk < 9 * coutA) {
        const int tp = kk / coutA, co = kk - tp * coutA;
        if (co < cout) v = w[(size_t)co * kpad + (8 - tp) * cin + ci];
    }
    wt[i] = to_bf16(v);
}

__global__ void k_adam(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                       const float* __restrict__ g, long long n, float lr, float b1, float b2,
                       float c1, float c2, float eps) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

template <typename T>
__global__ void k_zero(T* __restrict__ p, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = T(0);
}

}  // namespace

// ===========================================================================
// host side
// ===========================================================================
struct NetConv {
    int c1, c2, cout, coutA;  // inputs (concatenated), logical and allocated outputs
    int relu;
    int K, kpad, coutpad;     // forward GEMM dims
    int cinpad, kpadT;        // input-gradient GEMM dims
    size_t woff;              // offset in the flat parameter arrays
    size_t nparam;            // coutpad * kpad
    int level;                // resolution level
    // tensors (indices into NetState::acts)
    int in1, in2, out;
};

struct NetTensor {
    int level, C;             // channels (multiple of 8)
    DevBuf act;               // BF16 (or FP32 for the head)
    DevBuf grad;              // FP32
};

struct cd_net {
    cd_context* ctx = nullptr;
    cd_net_arch arch;
    std::vector<NetConv> convs;
    size_t nparam = 0;
    DevBuf w, m, v, gw, wbf, wtbf, partials, head, ghead, x8;
    DevBuf yout, ytmp, gy, ures, utmp;  // FP32 [B][H][W]: output, dL/dy, loss work
    unsigned long long gen = 0;          // bumped when the activation buffers move
    unsigned id = 0;                     // unique per net created in the process
    size_t wtoff_total = 0;
    std::vector<size_t> wtoff;
    long long step = 0;
    // activation tensors for the current (batch, h, w)
    std::vector<NetTensor> t;
    int batch = 0, bh = 0, bw = 0;
    bool weights_dirty = true;
    bool fused_forward = true;  // inference forwards fold the decoder upsampling and the
                                // encoder pooling into the convs
    bool tiled_forward = true;  // forward convolutions on LDS-staged 8x8 tiles (bit-identical)
    bool head_pending = false;  // fused forward left the head to finish_output (k_head_smooth)
};

namespace {

// Dynamic LDS available to k_conv3x3_tile on this context's device (the
// kernels' limit raised to the device's per-workgroup maximum once).
size_t tiled_lds_limit(cd_context* c) {
    static std::atomic<long long> limit{-1};
    long long v = limit.load();
    if (v >= 0) return (size_t)v;
    int bytes = 0;
    if (hipDeviceGetAttribute(&bytes, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device) !=
        hipSuccess)
        bytes = 0;
    const void* fns[] = {reinterpret_cast<const void*>(&k_conv3x3_tile<1, 0>),
                         reinterpret_cast<const void*>(&k_conv3x3_tile<2, 0>),
                         reinterpret_cast<const void*>(&k_conv3x3_tile<1, 1>),
                         reinterpret_cast<const void*>(&k_conv3x3_tile<1, 2, 1>),
                         reinterpret_cast<const void*>(&k_conv3x3_tile<2, 2, 1>),
                         reinterpret_cast<const void*>(&k_conv_pair_tile<1, 8, 16, false>),
                         reinterpret_cast<const void*>(&k_conv_pair_tile<1, 48, 16, false>),
                         reinterpret_cast<const void*>(&k_conv_pair_tile<2, 16, 32, true>),
                         reinterpret_cast<const void*>(&k_conv_pair_tile<2, 32, 32, true>),
                         reinterpret_cast<const void*>(&k_conv_pair_tile<2, 64, 32, false>),
                         reinterpret_cast<const void*>(&k_conv_pair_tile<1, 0, 0, true>),
                         reinterpret_cast<const void*>(&k_conv_pair_tile<1, 0, 0, false>),
                         reinterpret_cast<const void*>(&k_conv_pair_tile<2, 0, 0, true>),
                         reinterpret_cast<const void*>(&k_conv_pair_tile<2, 0, 0, false>),
                         reinterpret_cast<const void*>(&k_head_smooth<6, 0>),
                         reinterpret_cast<const void*>(&k_head_smooth<6, 16>)};
    for (const void* f : fns)
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) !=
            hipSuccess) {
            (void)hipGetLastError();
            bytes = std::min(bytes, 64 * 1024);
        }
    limit.store(bytes);
    return (size_t)bytes;
}

#ifndef CD_CONV_WIDE_MIN_BLOCKS
#define CD_CONV_WIDE_MIN_BLOCKS 512
#endif
constexpr long long kConvWideMinBlocks = CD_CONV_WIDE_MIN_BLOCKS;

// mode1: 0 reads in1 as stored; 1 reads `x1src` (the half-resolution tensor
// in1 is upsampled from) through nearest 2x upsampling instead; 2 reads
// `x1src` (the double-resolution tensor in1 is pooled from) through 2x2
// average pooling (the tiled kernel; otherwise the pooled tensor is written
// first)
int launch_conv(cd_net* n, const NetConv& cv, int B, int H, int W, bool grad_input,
                int mode1 = 0, const u16* x1src = nullptr) {
    cd_context* c = n->ctx;
    hipStream_t s = c->stream;
    const long long npix = (long long)B * H * W;
    const int blocks = div_up(npix, 64);
    // LDS the tiled kernel needs for this convolution (8x8 tile + halo, the
    // weights of up to 32 output channels)
    // 32 output channels per workgroup where the image has enough 8x8 tiles to
    // fill the GPU, else 16 (twice the workgroups, half the weights staged by
    // each: the deep levels' convolutions are bound by that staging)
    const long long tiles_t = (long long)B * div_up(H, CT) * div_up(W, CT);
    const int nbw_t = ((cv.coutpad / 16) % 2 == 0 && tiles_t * (cv.coutpad / 32) >= kConvWideMinBlocks) ? 2 : 1;
    const size_t lds_t = sizeof(u16) * (100 * (size_t)(cv.c1 + cv.c2 + 8) +
                                        (size_t)nbw_t * 16 * (cv.kpad + 8));
    const bool tiled = !grad_input && n->tiled_forward && lds_t <= tiled_lds_limit(c);
    if (mode1 == 2 && cv.c2 > 0) return CD_ERR_BAD_ARG;  // a pooled input has no skip part
    if (mode1 == 2 && !tiled) {
        hipLaunchKernelGGL(k_avgpool2, resample_grid((long long)B * H, W * (cv.c1 / 8)), dim3(256), 0, s, x1src,
                           n->t[cv.in1].act.as<u16>(), B, 2 * H, 2 * W, cv.c1);
        mode1 = 0;
        x1src = nullptr;
    }
    if (tiled) {
        const u16* x1 = mode1 ? x1src
                              : (cv.in1 < 0 ? n->x8.as<u16>() : n->t[cv.in1].act.as<u16>());
        const u16* x2 = cv.in2 < 0 ? nullptr : n->t[cv.in2].act.as<u16>();
        const u16* wt = n->wbf.as<u16>() + cv.woff;
        const int nb = cv.coutpad / 16;
        // up to 32 output channels per workgroup (LDS), the rest in more blocks
        const int nbw = nbw_t;
        const int cblocks = nb / nbw;
        const size_t lds = lds_t;
        const dim3 grid(div_up(W, CT), div_up(H, CT), B * cblocks);
        const bool head = cv.out < 0;  // FP32 output [npix][8]
        if (head && (nbw != 1 || cblocks != 1)) return CD_ERR_BAD_ARG;
        u16* y = head ? nullptr : n->t[cv.out].act.as<u16>();
        float* yf = head ? n->head.as<float>() : nullptr;
        const int cy = head ? 8 : cv.coutA, relu = head ? 0 : cv.relu;
        // input channels of the shipped networks unrolled
        const int cin = mode1 == 2 ? 0 : cv.c1 + cv.c2;
#define TILE(NB, OUT, CIN) hipLaunchKernelGGL((k_conv3x3_tile<NB, OUT, 0, CIN>), grid, dim3(256), lds, s, x1, x2, cv.c1, cv.c2, wt, cv.kpad, H, W, cblocks, y, yf, cy, relu, mode1)
        if (head) {
            if (cin == 16) TILE(1, 1, 16);
            else TILE(1, 1, 0);
        } else if (nbw == 2) {
            if (cin == 16) TILE(2, 0, 16);
            else if (cin == 32) TILE(2, 0, 32);
            else if (cin == 64) TILE(2, 0, 64);
            else TILE(2, 0, 0);
        } else {
            if (cin == 8) TILE(1, 0, 8);
            else if (cin == 16) TILE(1, 0, 16);
            else if (cin == 32) TILE(1, 0, 32);
            else if (cin == 48) TILE(1, 0, 48);
            else if (cin == 64) TILE(1, 0, 64);
            else TILE(1, 0, 0);
        }
#undef TILE
    } else if (!grad_input) {
        const u16* x1 = mode1 ? x1src
                              : (cv.in1 < 0 ? n->x8.as<u16>() : n->t[cv.in1].act.as<u16>());
        const u16* x2 = cv.in2 < 0 ? nullptr : n->t[cv.in2].act.as<u16>();
        const u16* wt = n->wbf.as<u16>() + cv.woff;
        const int nb = cv.coutpad / 16;
        if (cv.out < 0) {  // head: FP32 output [npix][8]
#define CONV_F(NB) hipLaunchKernelGGL((k_conv3x3<NB, 0, 1>), dim3(blocks), dim3(256), 0, s, x1, x2, cv.c1, cv.c2, (const float*)nullptr, (const u16*)nullptr, wt, cv.kpad, B, H, W, (u16*)nullptr, n->head.as<float>(), (float*)nullptr, 8, 0, 0, mode1)
            if (nb == 1) CONV_F(1);
            else return CD_ERR_BAD_ARG;
#undef CONV_F
        } else {
            u16* y = n->t[cv.out].act.as<u16>();
#define CONV_B(NB) hipLaunchKernelGGL((k_conv3x3<NB, 0, 0>), dim3(blocks), dim3(256), 0, s, x1, x2, cv.c1, cv.c2, (const float*)nullptr, (const u16*)nullptr, wt, cv.kpad, B, H, W, y, (float*)nullptr, (float*)nullptr, cv.coutA, 0, cv.relu, mode1)
            switch (nb) {
                case 1: CONV_B(1); break;
                case 2: CONV_B(2); break;
                case 3: CONV_B(3); break;
                case 4: CONV_B(4); break;
                case 6: CONV_B(6); break;
                case 8: CONV_B(8); break;
                default: return CD_ERR_BAD_ARG;
            }
#undef CONV_B
        }
    } else {
        // input gradient: conv of the masked output gradient with transposed weights
        const float* g = cv.out < 0 ? n->ghead.as<float>() : n->t[cv.out].grad.as<float>();
        const u16* mask = (cv.out >= 0 && cv.relu) ? n->t[cv.out].act.as<u16>() : nullptr;
        const u16* wt = n->wtbf.as<u16>() + n->wtoff[&cv - &n->convs[0]];
        float* d1 = n->t[cv.in1].grad.as<float>();
        float* d2 = cv.in2 < 0 ? nullptr : n->t[cv.in2].grad.as<float>();
        const int nb = cv.cinpad / 16;
        // on tiles where their LDS allows, as the forward convolutions: 9 to 25 us
        // by per-chunk global gathers, 5 to 7 on tiles at 8 x 128 x 128
        const int nbg = nb % 2 == 0 && tiles_t * (nb / 2) >= kConvWideMinBlocks ? 2 : 1;
        const size_t lds_g = sizeof(u16) * (100 * (size_t)(cv.coutA + 8) +
                                            (size_t)nbg * 16 * (cv.kpadT + 8));
        if (cv.coutA <= 256 && lds_g <= tiled_lds_limit(c)) {
            const int cblocks = nb / nbg;
            const dim3 grid(div_up(W, CT), div_up(H, CT), B * cblocks);
            auto kernel = nbg == 2 ? k_conv3x3_tile<2, 2, 1> : k_conv3x3_tile<1, 2, 1>;
            if (cv.coutA == 8)  // gradient channels of the shipped networks unrolled
                kernel = nbg == 2 ? k_conv3x3_tile<2, 2, 1, 8> : k_conv3x3_tile<1, 2, 1, 8>;
            else if (cv.coutA == 16)
                kernel = nbg == 2 ? k_conv3x3_tile<2, 2, 1, 16> : k_conv3x3_tile<1, 2, 1, 16>;
            else if (cv.coutA == 32)
                kernel = nbg == 2 ? k_conv3x3_tile<2, 2, 1, 32> : k_conv3x3_tile<1, 2, 1, 32>;
            hipLaunchKernelGGL(kernel, grid, dim3(256), lds_g, s, (const u16*)nullptr,
                               (const u16*)nullptr, cv.coutA, 0, wt, cv.kpadT, H, W, cblocks,
                               (u16*)nullptr, d1, cv.c1, 0, 0, g, mask, d2, cv.c2);
            CD_CHECK_LAUNCH(c);
            return CD_OK;
        }
#define CONV_G(NB) hipLaunchKernelGGL((k_conv3x3<NB, 1, 1>), dim3(blocks), dim3(256), 0, s, (const u16*)nullptr, (const u16*)nullptr, cv.coutA, 0, g, mask, wt, cv.kpadT, B, H, W, (u16*)nullptr, d1, d2, cv.c1, cv.c2, 0, 0)
        switch (nb) {
            case 1: CONV_G(1); break;
            case 2: CONV_G(2); break;
            case 3: CONV_G(3); break;
            case 4: CONV_G(4); break;
            case 6: CONV_G(6); break;
            case 8: CONV_G(8); break;
            default: return CD_ERR_BAD_ARG;
        }
#undef CONV_G
    }
    CD_CHECK_LAUNCH(c);
    return CD_OK;
}

int launch_wgrad(cd_net* n, const NetConv& cv, int B, int H, int W) {
    cd_context* c = n->ctx;
    const u16* x1 = cv.in1 < 0 ? n->x8.as<u16>() : n->t[cv.in1].act.as<u16>();
    const u16* x2 = cv.in2 < 0 ? nullptr : n->t[cv.in2].act.as<u16>();
    const float* g = cv.out < 0 ? n->ghead.as<float>() : n->t[cv.out].grad.as<float>();
    const u16* mask = (cv.out >= 0 && cv.relu) ? n->t[cv.out].act.as<u16>() : nullptr;
    const int cin = cv.c1 + cv.c2;
    const int nci = div_up(cin, 16) % 2 == 0 ? 2 : 1, nco = cv.coutA > 16 ? 2 : 1;
    const int tx = div_up(W, WG_TC), ty = div_up(H, WG_TR);
    const int gy = div_up(cin, 16 * nci), gz = div_up(cv.coutA, 16 * nco);
    // up to 1.5 workgroups per CU, each over the same number of tiles (a training
    // gradient at 8 x 128 x 128 takes 524 us; 528 with up to 256 workgroups, 543
    // with 512, 547 with 768: more atomics)
    const int gmax = std::max(1, 384 / (gy * gz));
    const int gx = div_up(tx * ty * B, div_up(tx * ty * B, gmax));
#define WGRAD(CI, CO) hipLaunchKernelGGL((k_wgrad<CI, CO>), dim3(gx, gy, gz), dim3(256), 0, c->stream, x1, x2, cv.c1, cv.c2, g, mask, cv.coutA, B, H, W, n->gw.as<float>() + cv.woff, cv.kpad, tx, ty)
    if (nci == 1 && nco == 1) WGRAD(1, 1);
    else if (nci == 1) WGRAD(1, 2);
    else if (nco == 1) WGRAD(2, 1);
    else WGRAD(2, 2);
#undef WGRAD
    CD_CHECK_LAUNCH(c);
    return CD_OK;
}

template <typename T>
int zero(cd_context* c, T* p, long long n) {
    if (n <= 0) return CD_OK;
    hipLaunchKernelGGL(k_zero<T>, dim3(div_up(n, 256)), dim3(256), 0, c->stream, p, n);
    CD_CHECK_LAUNCH(c);
    return CD_OK;
}

// Build the layer list (independent of batch size).
void build_layers(cd_net* n) {
    const int L = n->arch.levels;
    const int* C = n->arch.channels;
    n->convs.clear();
    n->t.clear();
    auto tensor = [&](int level, int ch) {
        NetTensor t;
        t.level = level;
        t.C = ch;
        n->t.push_back(std::move(t));
        return (int)n->t.size() - 1;
    };
    auto conv = [&](int in1, int c1, int in2, int c2, int out, int cout, int coutA, int relu,
                    int level) {
        NetConv cv;
        cv.c1 = c1; cv.c2 = c2; cv.cout = cout; cv.coutA = coutA; cv.relu = relu;
        cv.K = 9 * (c1 + c2);
        cv.kpad = (cv.K + 31) / 32 * 32;
        cv.coutpad = (coutA + 15) / 16 * 16;
        cv.cinpad = (c1 + c2 + 15) / 16 * 16;
        cv.kpadT = (9 * coutA + 31) / 32 * 32;
        cv.woff = n->nparam;
        cv.nparam = (size_t)cv.coutpad * cv.kpad;
        n->nparam += cv.nparam;
        cv.level = level;
        cv.in1 = in1; cv.in2 = in2; cv.out = out;
        n->convs.push_back(cv);
    };
    const int act = n->arch.linear ? 0 : 1;  // ReLU on hidden convolutions
    std::vector<int> skip(L);
    int prev = -1, prevC = 8;  // -1: the 8-channel input tensor
    for (int l = 0; l < L; ++l) {
        int in = prev, inC = prevC;
        if (l > 0) {
            const int p = tensor(l, prevC);  // pooled
            n->t[p].level = l;
            in = p;
        }
        const int a = tensor(l, C[l]);
        conv(in, inC, -1, 0, a, C[l], C[l], act, l);
        const int s = tensor(l, C[l]);
        conv(a, C[l], -1, 0, s, C[l], C[l], act, l);
        skip[l] = s;
        prev = s;
        prevC = C[l];
    }
    int d = skip[L - 1], dC = C[L - 1];
    for (int l = L - 2; l >= 0; --l) {
        const int u = tensor(l, dC);  // upsampled
        const int b = tensor(l, C[l]);
        conv(u, dC, skip[l], C[l], b, C[l], C[l], act, l);
        const int e = tensor(l, C[l]);
        conv(b, C[l], -1, 0, e, C[l], C[l], act, l);
        d = e;
        dC = C[l];
    }
    conv(d, dC, -1, 0, -1, 1, 8, 0, 0);  // head: 1 output channel stored with stride 8
    n->wtoff.clear();
    size_t off = 0;
    for (auto& cv : n->convs) {
        n->wtoff.push_back(off);
        off += (size_t)cv.cinpad * cv.kpadT;
    }
    n->wtoff_total = off;
}

int ensure_batch(cd_net* n, int B, int H, int W) {
    cd_context* c = n->ctx;
    const int L = n->arch.levels;
    if (H % (1 << (L - 1)) || W % (1 << (L - 1))) {
        c->set_error("net input size must be divisible by 2^(levels-1)");
        return CD_ERR_BAD_ARG;
    }
    if (n->batch == B && n->bh == H && n->bw == W) return CD_OK;
    ++n->gen;
    for (auto& t : n->t) {
        const long long px = (long long)B * (H >> t.level) * (W >> t.level);
        CD_TRY(c->ensure(t.act, sizeof(u16) * px * t.C));
        CD_TRY(c->ensure(t.grad, sizeof(float) * px * t.C));
    }
    const long long px = (long long)B * H * W;
    CD_TRY(c->ensure(n->x8, sizeof(u16) * px * 8));
    CD_TRY(c->ensure(n->head, sizeof(float) * px * 8));
    CD_TRY(c->ensure(n->ghead, sizeof(float) * px * 8));
    for (DevBuf* b : {&n->yout, &n->ytmp, &n->gy, &n->ures, &n->utmp})
        CD_TRY(c->ensure(*b, sizeof(float) * px));
    CD_TRY(c->ensure(n->partials, sizeof(double) * (size_t)div_up(px, 256)));
    n->batch = B;
    n->bh = H;
    n->bw = W;
    return CD_OK;
}

int refresh_weights(cd_net* n) {
    if (!n->weights_dirty) return CD_OK;
    cd_context* c = n->ctx;
    hipLaunchKernelGGL(k_cast_bf16, dim3(div_up((long long)n->nparam, 256)), dim3(256), 0,
                       c->stream, n->w.as<float>(), n->wbf.as<u16>(), (long long)n->nparam);
    for (size_t i = 0; i < n->convs.size(); ++i) {
        const NetConv& cv = n->convs[i];
        const long long cnt = (long long)cv.cinpad * cv.kpadT;
        hipLaunchKernelGGL(k_transpose_w, dim3(div_up(cnt, 256)), dim3(256), 0, c->stream,
                           n->w.as<float>() + cv.woff, n->wtbf.as<u16>() + n->wtoff[i], cv.cout,
                           cv.coutA, cv.c1 + cv.c2, cv.kpad, cv.cinpad, cv.kpadT);
    }
    CD_CHECK_LAUNCH(c);
    n->weights_dirty = false;
    return CD_OK;
}

// forward pass from the 8-channel input already in n->x8; head output in n->head
// fused (inference): the upsampled decoder inputs are read through the
// convolutions that consume them (a pure index remap) instead of being
// materialised; the output is bit-identical.  Training needs the materialised
// tensors (weight gradients read them).  Pooling stays a separate pass: read
// through the convolution (mode 2) it costs more than it saves.
// Convolutions a and b (b reads only a's output, at a's resolution) in one
// k_conv_pair_tile launch where the LDS allows; returns false (nothing
// launched) where it does not apply.
bool launch_conv_pair(cd_net* n, const NetConv& a, const NetConv& b, int B, int H, int W,
                      int mode1, const u16* x1src, int* err) {
    *err = CD_OK;
    // up to 32 output channels: one workgroup computing all 64 channels of
    // both convs of a 32x32 or 16x16 level (4-16 workgroups) measured 3.6-4.6 us
    // slower than the two launches that split the channels over 4 workgroups
    // per tile
    const int nba = a.coutpad / 16, nbb = b.coutpad / 16;
    if (nba != nbb || !(nba == 1 || nba == 2)) return false;
    if (b.in1 != a.out || b.in2 >= 0 || b.out < 0 || a.out < 0 || b.c1 != a.coutA) return false;
    if (mode1 == 2 && a.c2 > 0) return false;
    const size_t fixed = 144 * (size_t)(a.c1 + a.c2 + 8) + 100 * (size_t)(a.coutA + 8);
    const size_t wa = (size_t)nba * 16 * (a.kpad + 8), wb = (size_t)nbb * 16 * (b.kpad + 8);
    const size_t limit = tiled_lds_limit(n->ctx);
    int early = 1;
    size_t lds = sizeof(u16) * (fixed + wa + wb);
    if (lds > limit) {
        early = 0;
        lds = sizeof(u16) * (fixed + std::max(wa, wb));
        if (lds > limit) return false;
    }
    const u16* x1 = mode1 ? x1src : (a.in1 < 0 ? n->x8.as<u16>() : n->t[a.in1].act.as<u16>());
    const u16* x2 = a.in2 < 0 ? nullptr : n->t[a.in2].act.as<u16>();
    const u16* wta = n->wbf.as<u16>() + a.woff;
    const u16* wtb = n->wbf.as<u16>() + b.woff;
    u16* y = n->t[b.out].act.as<u16>();
    const dim3 grid(div_up(W, CT), div_up(H, CT), B);
    hipStream_t s = n->ctx->stream;
    const int cina = a.c1 + a.c2, cinb = a.coutA;
    const bool pool = mode1 == 2;
#define PAIR(NB, CA, CB, POOL) hipLaunchKernelGGL((k_conv_pair_tile<NB, CA, CB, POOL>), grid, dim3(kPairThreads), lds, s, x1, x2, a.c1, a.c2, wta, a.kpad, a.coutA, a.relu, wtb, b.kpad, b.coutA, b.relu, y, H, W, mode1, early)
    // 16 and 32 channels per level, as in the shipped networks
    if (nba == 1 && !pool && cina == 8 && cinb == 16) PAIR(1, 8, 16, false);
    else if (nba == 1 && !pool && cina == 48 && cinb == 16) PAIR(1, 48, 16, false);
    else if (nba == 2 && pool && cina == 16 && cinb == 32) PAIR(2, 16, 32, true);
    else if (nba == 2 && pool && cina == 32 && cinb == 32) PAIR(2, 32, 32, true);
    else if (nba == 2 && !pool && cina == 64 && cinb == 32) PAIR(2, 64, 32, false);
    else if (nba == 1 && pool) PAIR(1, 0, 0, true);
    else if (nba == 1) PAIR(1, 0, 0, false);
    else if (pool) PAIR(2, 0, 0, true);
    else PAIR(2, 0, 0, false);
#undef PAIR
    return true;
}

// the head + output smoothing kernel applies: 6 smoothing steps (the kernel's
// instantiation), one 16-channel block, no skip input, and the LDS fits
constexpr int kHeadSmoothK = 6;
bool head_smooth_ok(cd_net* n, const NetConv& hd) {
    if (n->arch.out_smooth != kHeadSmoothK || hd.coutpad != 16 || hd.in2 >= 0 || hd.in1 < 0)
        return false;
    constexpr int R = kSmoothTile + 2 * kHeadSmoothK, P = R + 2;
    const size_t lds = sizeof(u16) * ((size_t)P * P * (hd.c1 + 8) + 16 * (size_t)(hd.kpad + 8)) +
                       sizeof(float) * 2 * R * R;
    return lds <= tiled_lds_limit(n->ctx);
}

int forward(cd_net* n, int B, int H, int W, bool fused = false) {
    cd_context* c = n->ctx;
    CD_TRY(refresh_weights(n));
    n->head_pending = false;
    const int L = n->arch.levels;
    const u16* pooled_from = nullptr;  // fused: the next conv pools this tensor as it reads
    for (int idx = 0; idx < (int)n->convs.size(); ++idx) {
        const NetConv& cv0 = n->convs[idx];
        const int Hl = H >> cv0.level, Wl = W >> cv0.level;
        const int mode1 = (fused && cv0.in2 >= 0) ? 1 : pooled_from ? 2 : 0;
        const u16* x1src = mode1 == 1 ? n->t[n->convs[idx - 1].out].act.as<u16>()
                                      : mode1 == 2 ? pooled_from : nullptr;
        // fused: the first conv of a level's pair (encoder, or the decoder's
        // concatenating one) and the next one in one launch where possible
        bool paired = false;
        if (fused && n->tiled_forward && idx + 1 < (int)n->convs.size() &&
            (cv0.in2 >= 0 || (idx < 2 * L && idx % 2 == 0))) {
            int err = CD_OK;
            paired = launch_conv_pair(n, cv0, n->convs[idx + 1], B, Hl, Wl, mode1, x1src, &err);
            CD_TRY(err);
            if (paired) ++idx;  // the pair's second conv is done
        }
        const NetConv& cv = n->convs[idx];
        // fused: the head and the output smoothing run as one launch in
        // finish_output
        if (!paired && fused && n->tiled_forward && cv.out < 0 && head_smooth_ok(n, cv)) {
            n->head_pending = true;
            continue;
        }
        if (!paired) CD_TRY(launch_conv(n, cv, B, Hl, Wl, false, mode1, x1src));
        pooled_from = nullptr;
        // after the second conv of an encoder level below the bottleneck: pool
        if (idx < 2 * L && idx % 2 == 1 && cv.level < L - 1) {
            const NetConv& nx = n->convs[idx + 1];  // next level's first conv reads the pooled tensor
            if (fused) {
                pooled_from = n->t[cv.out].act.as<u16>();
            } else {
                const int C = n->t[nx.in1].C;
                hipLaunchKernelGGL(k_avgpool2,
                                   resample_grid((long long)B * (Hl / 2), (Wl / 2) * (C / 8)),
                                   dim3(256), 0, c->stream, n->t[cv.out].act.as<u16>(), n->t[nx.in1].act.as<u16>(), B, Hl,
                                   Wl, C);
            }
        }
        // before a decoder concat conv: upsample the previous decoder output
        if (!fused && idx + 1 < (int)n->convs.size()) {
            const NetConv& nx = n->convs[idx + 1];
            if (nx.in2 >= 0) {
                const int Hn = H >> nx.level, Wn = W >> nx.level;
                const int C = n->t[nx.in1].C;
                hipLaunchKernelGGL(k_upsample2, resample_grid((long long)B * Hn, Wn * (C / 8)),
                                   dim3(256), 0, c->stream, n->t[cv.out].act.as<u16>(),
                                   n->t[nx.in1].act.as<u16>(), B, Hn, Wn, C);
            }
        }
        CD_CHECK_LAUNCH(c);
    }
    return CD_OK;
}

// backward pass: n->ghead holds dL/dhead; accumulates n->gw.  A tensor's first
// gradient is stored, so that none needs zeroing (21 launches): every tensor has
// one consumer but the skips, whose decoder convolution comes before their
// pooling here, and only the pooling adds.
int backward(cd_net* n, int B, int H, int W) {
    cd_context* c = n->ctx;
    const int L = n->arch.levels;
    for (int idx = (int)n->convs.size() - 1; idx >= 0; --idx) {
        const NetConv& cv = n->convs[idx];
        const int Hl = H >> cv.level, Wl = W >> cv.level;
        // gradient into this conv's output is complete here: its consumers
        // (later convs, pooling, upsampling) were processed before it
        CD_TRY(launch_wgrad(n, cv, B, Hl, Wl));
        if (cv.in1 >= 0) CD_TRY(launch_conv(n, cv, B, Hl, Wl, true));
        // route input gradients through upsampling / pooling
        if (cv.in2 >= 0) {
            // in1 is the upsampled previous decoder output (level+1)
            const NetConv& pv = n->convs[idx - 1];
            const int C = n->t[cv.in1].C;
            hipLaunchKernelGGL(k_upsample2_bwd,
                               resample_grid((long long)B * (Hl / 2), (Wl / 2) * (C / 4)),
                               dim3(256), 0, c->stream, n->t[cv.in1].grad.as<float>(),
                               n->t[pv.out].grad.as<float>(), B, Hl, Wl, C);
        }
        if (idx < 2 * L && idx % 2 == 0 && cv.level > 0) {
            // in1 is the pooled skip of the level above
            const NetConv& pv = n->convs[idx - 1];
            const int C = n->t[cv.in1].C;
            hipLaunchKernelGGL(k_avgpool2_bwd,
                               resample_grid((long long)B * (Hl * 2), (Wl * 2) * (C / 4)),
                               dim3(256), 0, c->stream, n->t[cv.in1].grad.as<float>(),
                               n->t[pv.out].grad.as<float>(), B, Hl * 2, Wl * 2, C);
        }
        CD_CHECK_LAUNCH(c);
    }
    return CD_OK;
}

// k symmetric smoothing steps on a [B][H][W] field held in *a (b is scratch);
// the result ends in *a
int smooth_steps(cd_net* n, DevBuf& a, DevBuf& b, int k, int B, int H, int W) {
    if (k <= 0) return CD_OK;
    const long long px = (long long)B * H * W;
    if (k <= kSmoothMaxK) {
        const int R = kSmoothTile + 2 * k;
        const dim3 grid(div_up(W, kSmoothTile), div_up(H, kSmoothTile), B);
        hipLaunchKernelGGL(k_smooth_tiled, grid, dim3(div_up(R * R, 64) * 64), sizeof(float) * 2 * R * R,
                           n->ctx->stream, a.as<float>(), 1, b.as<float>(), B, H, W, k);
        std::swap(a.ptr, b.ptr);
        std::swap(a.bytes, b.bytes);
    } else {
        for (int i = 0; i < k; ++i) {
            hipLaunchKernelGGL(k_smooth_step, dim3(div_up(px, 256)), dim3(256), 0,
                               n->ctx->stream, a.as<float>(), b.as<float>(), B, H, W);
            std::swap(a.ptr, b.ptr);
            std::swap(a.bytes, b.bytes);
        }
    }
    CD_CHECK_LAUNCH(n->ctx);
    return CD_OK;
}

// network output y = S^out_smooth (head channel 0) into dst (n->yout when null)
int finish_output(cd_net* n, int B, int H, int W, float* dst = nullptr) {
    const long long px = (long long)B * H * W;
    float* y = dst ? dst : n->yout.as<float>();
    const int k = n->arch.out_smooth;
    if (n->head_pending) {  // the fused forward's head with the smoothing
        n->head_pending = false;
        const NetConv& hd = n->convs.back();
        constexpr int R = kSmoothTile + 2 * kHeadSmoothK, P = R + 2;
        const size_t lds = sizeof(u16) * ((size_t)P * P * (hd.c1 + 8) + 16 * (size_t)(hd.kpad + 8)) +
                           sizeof(float) * 2 * R * R;
        const dim3 grid(div_up(W, CT), div_up(H, CT), B);
        const u16* x = n->t[hd.in1].act.as<u16>();
        const u16* wt = n->wbf.as<u16>() + hd.woff;
        if (hd.c1 == 16)  // as in the shipped networks
            hipLaunchKernelGGL((k_head_smooth<kHeadSmoothK, 16>), grid, dim3(512), lds,
                               n->ctx->stream, x, hd.c1, wt, hd.kpad, H, W, y);
        else
            hipLaunchKernelGGL((k_head_smooth<kHeadSmoothK, 0>), grid, dim3(512), lds,
                               n->ctx->stream, x, hd.c1, wt, hd.kpad, H, W, y);
        CD_CHECK_LAUNCH(n->ctx);
        return CD_OK;
    }
    if (k > 0 && k <= kSmoothMaxK) {
        // head channel 0 -> k steps -> y in one launch
        const int R = kSmoothTile + 2 * k;
        const dim3 grid(div_up(W, kSmoothTile), div_up(H, kSmoothTile), B);
        hipLaunchKernelGGL(k_smooth_tiled, grid, dim3(div_up(R * R, 64) * 64), sizeof(float) * 2 * R * R,
                           n->ctx->stream, n->head.as<float>(), 8, y, B, H, W, k);
        CD_CHECK_LAUNCH(n->ctx);
        return CD_OK;
    }
    hipLaunchKernelGGL(k_head_out, dim3(div_up(px, 256)), dim3(256), 0, n->ctx->stream,
                       n->head.as<float>(), n->yout.as<float>(), px);
    CD_CHECK_LAUNCH(n->ctx);
    CD_TRY(smooth_steps(n, n->yout, n->ytmp, k, B, H, W));
    if (dst)
        CD_HIP(n->ctx, hipMemcpyAsync(dst, n->yout.ptr, sizeof(float) * px,
                                      hipMemcpyDeviceToDevice, n->ctx->stream));
    return CD_OK;
}

// dL/dy in n->gy -> dL/dhead (S is symmetric, so its transpose is itself)
int head_grad(cd_net* n, int B, int H, int W) {
    const long long px = (long long)B * H * W;
    CD_TRY(smooth_steps(n, n->gy, n->ytmp, n->arch.out_smooth, B, H, W));
    hipLaunchKernelGGL(k_head_grad, dim3(div_up(px, 256)), dim3(256), 0, n->ctx->stream,
                       n->gy.as<float>(), n->ghead.as<float>(), px);
    CD_CHECK_LAUNCH(n->ctx);
    return CD_OK;
}

int read_loss(cd_net* n, int nb, long long px, double* loss) {
    cd_context* c = n->ctx;
    CD_TRY(c->ensure(c->fill, sizeof(double) * 4));
    CD_TRY(cd_reduce_partials(c, n->partials.as<double>(), nb, 1, c->fill.as<double>()));
    double s = 0.0;
    CD_HIP(c, hipMemcpyAsync(&s, c->fill.ptr, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    CD_HIP(c, hipStreamSynchronize(c->stream));
    if (loss) *loss = s / (double)px;
    return CD_OK;
}

int loss_and_head_grad(cd_net* n, const float* d_t, int B, int H, int W, double* loss,
                       bool want_grad) {
    const long long px = (long long)B * H * W;
    const int nb = div_up(px, 256);
    CD_TRY(finish_output(n, B, H, W));
    hipLaunchKernelGGL(k_loss, dim3(nb), dim3(256), 0, n->ctx->stream, n->yout.as<float>(), d_t,
                       want_grad ? n->gy.as<float>() : nullptr, px, n->partials.as<double>());
    CD_CHECK_LAUNCH(n->ctx);
    if (want_grad) CD_TRY(head_grad(n, B, H, W));
    return read_loss(n, nb, px, loss);
}

// coarse operator scale (n/pi)^2, n the larger side: makes outputs O(1)
inline float op_scale(int H, int W) {
    const double m = (double)std::max(H, W) / M_PI;
    return (float)(m * m);
}

// operator loss: u = cs Lc y - x, v = S^loss_smooth u, loss = mean(v^2);
// dL/dy = cs Lc S^loss_smooth (2 v / npix).  With arch.loss_energy the loss is
// the energy mean(y (x - u) / 2) and dL/dy = -u / npix.
int op_loss_and_head_grad(cd_net* n, const float* d_x, int B, int H, int W, double* loss,
                          bool want_grad) {
    cd_context* c = n->ctx;
    const long long px = (long long)B * H * W;
    const int nb = div_up(px, 256);
    const float cs = op_scale(H, W);
    CD_TRY(finish_output(n, B, H, W));
    hipLaunchKernelGGL(k_op_residual, dim3(nb), dim3(256), 0, c->stream, n->yout.as<float>(), d_x,
                       n->ures.as<float>(), B, H, W, cs);
    CD_CHECK_LAUNCH(c);
    if (n->arch.loss_energy) {
        hipLaunchKernelGGL(k_energy, dim3(nb), dim3(256), 0, c->stream, n->yout.as<float>(), d_x,
                           n->ures.as<float>(), n->gy.as<float>(), px, want_grad ? 1 : 0,
                           n->partials.as<double>());
        CD_CHECK_LAUNCH(c);
        if (want_grad) CD_TRY(head_grad(n, B, H, W));
        return read_loss(n, nb, px, loss);
    }
    CD_TRY(smooth_steps(n, n->ures, n->utmp, n->arch.loss_smooth, B, H, W));
    hipLaunchKernelGGL(k_sumsq, dim3(nb), dim3(256), 0, c->stream, n->ures.as<float>(), px,
                       want_grad ? 1 : 0, n->partials.as<double>());
    CD_CHECK_LAUNCH(c);
    if (want_grad) {
        CD_TRY(smooth_steps(n, n->ures, n->utmp, n->arch.loss_smooth, B, H, W));
        hipLaunchKernelGGL(k_op_grad, dim3(nb), dim3(256), 0, c->stream, n->ures.as<float>(),
                           n->gy.as<float>(), B, H, W, cs);
        CD_CHECK_LAUNCH(c);
        CD_TRY(head_grad(n, B, H, W));
    }
    return read_loss(n, nb, px, loss);
}

int prep(cd_net* n, const float* d_x, int B, int H, int W) {
    CD_TRY(ensure_batch(n, B, H, W));
    const long long px = (long long)B * H * W;
    hipLaunchKernelGGL(k_prep_input, dim3(div_up(px, 256)), dim3(256), 0, n->ctx->stream, d_x,
                       n->x8.as<u16>(), px);
    CD_CHECK_LAUNCH(n->ctx);
    return CD_OK;
}

// one Adam step (beta 0.9/0.999, eps 1e-8) from the accumulated gradient
int adam_step(cd_net* n, float lr) {
    cd_context* c = n->ctx;
    n->step += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)n->step), c2 = 1.f - std::pow(b2, (float)n->step);
    hipLaunchKernelGGL(k_adam, dim3(div_up((long long)n->nparam, 256)), dim3(256), 0, c->stream,
                       n->w.as<float>(), n->m.as<float>(), n->v.as<float>(), n->gw.as<float>(),
                       (long long)n->nparam, lr, b1, b2, c1, c2, 1e-8f);
    CD_CHECK_LAUNCH(c);
    n->weights_dirty = true;
    return CD_OK;
}

}  // namespace

// solver-side entry: forward on the coarse residual rc (batch 1), normalised
// on the fly with stats = (sum, sum^2); output FP32 [h][w]
int cd_net_forward_coarse(cd_net* n, const float* rc, const double* stats, float* d_y, int h,
                          int w) {
    CD_TRY(ensure_batch(n, 1, h, w));
    hipLaunchKernelGGL(k_prep_normalized, dim3(div_up(h * w, 256)), dim3(256), 0, n->ctx->stream,
                       rc, stats, h * w, n->x8.as<u16>());
    CD_CHECK_LAUNCH(n->ctx);
    CD_TRY(forward(n, 1, h, w, n->fused_forward));
    return finish_output(n, 1, h, w, d_y);
}

// The network's BF16 input buffer for one h x w coarse field (sized here),
// for a producer that writes the normalised input itself (channel 0, the
// other 7 zero), and the forward on that input
int cd_net_coarse_input(cd_net* n, int h, int w, unsigned short** x8) {
    CD_TRY(ensure_batch(n, 1, h, w));
    *x8 = n->x8.as<u16>();
    return CD_OK;
}
int cd_net_forward_prepared(cd_net* n, float* d_y, int h, int w) {
    CD_TRY(ensure_batch(n, 1, h, w));
    CD_TRY(forward(n, 1, h, w, n->fused_forward));
    return finish_output(n, 1, h, w, d_y);
}

// solver-side entry: forward on one coarse field (batch 1), output FP32 [h][w]
int cd_net_forward_internal(cd_net* n, const float* d_x, float* d_y, int h, int w) {
    CD_TRY(prep(n, d_x, 1, h, w));
    CD_TRY(forward(n, 1, h, w, n->fused_forward));
    return finish_output(n, 1, h, w, d_y);
}

const cd_net_arch* cd_net_arch_of(const cd_net* n) { return &n->arch; }
unsigned long long cd_net_gen(const cd_net* n) {
    return ((unsigned long long)n->id << 32) | (n->gen & 0xffffffffULL);
}

extern "C" void cd_net_detach(cd_net* n) {
    cd_context* c = n->ctx;
    if (!c) return;
    if (c->net == n) c->net = nullptr;
    for (size_t i = 0; i < c->nets.size(); ++i)
        if (c->nets[i] == n) { c->nets.erase(c->nets.begin() + i); break; }
    n->ctx = nullptr;
}

extern "C" {

void cd_net_arch_default(cd_net_arch* a) {
    if (!a) return;
    std::memset(a, 0, sizeof(*a));
    a->levels = 4;
    a->channels[0] = 16;
    a->channels[1] = 32;
    a->channels[2] = 64;
    a->channels[3] = 64;
    a->coarsen = 4;
    a->smooth_sweeps = 4;
    a->smooth_omega = 1.2;
    a->linear = 1;
    a->out_smooth = 0;
    a->loss_smooth = 0;
    a->loss_energy = 0;
    a->mid_sweeps = 0;
}

int cd_net_create(cd_context* ctx, const cd_net_arch* arch, cd_net** out) {
    if (!ctx || !arch || !out) return CD_ERR_BAD_ARG;
    *out = nullptr;
    if (arch->levels < 2 || arch->levels > 6 || arch->coarsen < 1) return CD_ERR_BAD_ARG;
    if (arch->out_smooth < 0 || arch->out_smooth > 64 || arch->loss_smooth < 0 ||
        arch->loss_smooth > 64 || arch->loss_energy < 0 || arch->loss_energy > 1 ||
        arch->mid_sweeps < 0 || arch->mid_sweeps > 64)
        return CD_ERR_BAD_ARG;
    for (int l = 0; l < arch->levels; ++l)
        if (arch->channels[l] <= 0 || arch->channels[l] % 8 || arch->channels[l] > 128)
            return CD_ERR_BAD_ARG;
    CD_HIP(ctx, hipSetDevice(ctx->device));
    auto* n = new cd_net();
    n->ctx = ctx;
    n->arch = *arch;
    build_layers(n);
    int st = CD_OK;
    if ((st = ctx->ensure(n->w, sizeof(float) * n->nparam)) != CD_OK ||
        (st = ctx->ensure(n->m, sizeof(float) * n->nparam)) != CD_OK ||
        (st = ctx->ensure(n->v, sizeof(float) * n->nparam)) != CD_OK ||
        (st = ctx->ensure(n->gw, sizeof(float) * n->nparam)) != CD_OK ||
        (st = ctx->ensure(n->wbf, sizeof(u16) * n->nparam)) != CD_OK ||
        (st = ctx->ensure(n->wtbf, sizeof(u16) * n->wtoff_total)) != CD_OK ||
        (st = zero(ctx, n->w.as<float>(), (long long)n->nparam)) != CD_OK ||
        (st = zero(ctx, n->m.as<float>(), (long long)n->nparam)) != CD_OK ||
        (st = zero(ctx, n->v.as<float>(), (long long)n->nparam)) != CD_OK) {
        delete n;
        return st;
    }
    static std::atomic<unsigned> next_id{0};
    n->id = ++next_id;
    ctx->nets.push_back(n);
    *out = n;
    return CD_OK;
}

void cd_net_destroy(cd_net* n) {
    if (!n) return;
    if (n->ctx) {
        (void)hipStreamSynchronize(n->ctx->stream);
        cd_net_detach(n);
    }
    delete n;
}

size_t cd_net_num_params(const cd_net* n) { return n ? n->nparam : 0; }

int cd_net_set_params(cd_net* n, const float* host, size_t count) {
    if (!n || !host || count != n->nparam) return CD_ERR_BAD_ARG;
    if (!n->ctx) return CD_ERR_STATE;
    cd_context* c = n->ctx;
    CD_HIP(c, hipMemcpyAsync(n->w.ptr, host, sizeof(float) * count, hipMemcpyHostToDevice,
                             c->stream));
    CD_TRY(zero(c, n->m.as<float>(), (long long)count));
    CD_TRY(zero(c, n->v.as<float>(), (long long)count));
    n->step = 0;
    n->weights_dirty = true;
    CD_HIP(c, hipStreamSynchronize(c->stream));
    return CD_OK;
}

int cd_net_get_params(cd_net* n, float* host, size_t count) {
    if (!n || !host || count != n->nparam) return CD_ERR_BAD_ARG;
    if (!n->ctx) return CD_ERR_STATE;
    cd_context* c = n->ctx;
    CD_HIP(c, hipMemcpyAsync(host, n->w.ptr, sizeof(float) * count, hipMemcpyDeviceToHost,
                             c->stream));
    CD_HIP(c, hipStreamSynchronize(c->stream));
    return CD_OK;
}

int cd_net_init_params(cd_net* n, unsigned long long seed) {
    if (!n) return CD_ERR_BAD_ARG;
    if (!n->ctx) return CD_ERR_STATE;
    std::vector<float> w(n->nparam, 0.f);
    std::mt19937_64 rng(seed);
    for (const NetConv& cv : n->convs) {
        const bool first = cv.in1 < 0 && &cv == &n->convs[0];  // sees input channel 0 only
        const int fan_in = 9 * (first ? 1 : cv.c1 + cv.c2);
        // ReLU: He-normal with a small head.  Linear: variance 1/(3 fan_in)
        // per layer, so the initial operator is close to zero and the first
        // steps of the operator loss are well conditioned.
        const float sd = n->arch.linear ? std::sqrt(1.f / (3.f * fan_in))
                                        : std::sqrt(2.f / (float)fan_in);
        std::normal_distribution<float> nd(0.f, sd);
        // head: small for ReLU nets; zero for linear ones (the zero operator,
        // operator loss exactly 1 at the start: no amplified initial noise)
        const float scale = cv.out < 0 ? (n->arch.linear ? 0.f : 0.1f) : 1.f;
        for (int co = 0; co < cv.cout; ++co)
            for (int k = 0; k < cv.K; ++k) {
                const int ci = k % (cv.c1 + cv.c2);
                if (first && ci != 0) continue;
                w[cv.woff + (size_t)co * cv.kpad + k] = scale * nd(rng);
            }
    }
    return cd_net_set_params(n, w.data(), w.size());
}

int cd_net_forward(cd_net* n, const float* d_x, float* d_y, int batch, int h, int w) {
    if (!n || !d_x || !d_y || batch < 1) return CD_ERR_BAD_ARG;
    if (!n->ctx) return CD_ERR_STATE;
    CD_HIP(n->ctx, hipSetDevice(n->ctx->device));
    CD_TRY(prep(n, d_x, batch, h, w));
    CD_TRY(forward(n, batch, h, w, n->fused_forward));
    CD_TRY(finish_output(n, batch, h, w, d_y));
    CD_HIP(n->ctx, hipStreamSynchronize(n->ctx->stream));
    return CD_OK;
}

int cd_net_set_fused_forward(cd_net* n, int on) {
    if (!n) return CD_ERR_BAD_ARG;
    if (!n->ctx) return CD_ERR_STATE;
    n->fused_forward = on != 0;
    return CD_OK;
}

int cd_net_set_tiled_forward(cd_net* n, int on) {
    if (!n) return CD_ERR_BAD_ARG;
    if (!n->ctx) return CD_ERR_STATE;
    n->tiled_forward = on != 0;
    ++n->gen;  // captured solver graphs hold the previous kernels
    return CD_OK;
}

int cd_net_loss_grad(cd_net* n, const float* d_x, const float* d_t, int batch, int h, int w,
                     double* loss, float* host_grad, size_t count) {
    if (!n || !d_x || !d_t || batch < 1) return CD_ERR_BAD_ARG;
    if (!n->ctx) return CD_ERR_STATE;
    if (host_grad && count != n->nparam) return CD_ERR_BAD_ARG;
    cd_context* c = n->ctx;
    CD_HIP(c, hipSetDevice(c->device));
    CD_TRY(prep(n, d_x, batch, h, w));
    CD_TRY(forward(n, batch, h, w));
    CD_TRY(loss_and_head_grad(n, d_t, batch, h, w, loss, true));
    CD_TRY(zero(c, n->gw.as<float>(), (long long)n->nparam));
    CD_TRY(backward(n, batch, h, w));
    if (host_grad) {
        CD_HIP(c, hipMemcpyAsync(host_grad, n->gw.ptr, sizeof(float) * n->nparam,
                                 hipMemcpyDeviceToHost, c->stream));
    }
    CD_HIP(c, hipStreamSynchronize(c->stream));
    return CD_OK;
}

int cd_net_loss_grad_operator(cd_net* n, const float* d_x, int batch, int h, int w,
                              double* loss, float* host_grad, size_t count) {
    if (!n || !d_x || batch < 1) return CD_ERR_BAD_ARG;
    if (!n->ctx) return CD_ERR_STATE;
    if (host_grad && count != n->nparam) return CD_ERR_BAD_ARG;
    cd_context* c = n->ctx;
    CD_HIP(c, hipSetDevice(c->device));
    CD_TRY(prep(n, d_x, batch, h, w));
    CD_TRY(forward(n, batch, h, w));
    CD_TRY(op_loss_and_head_grad(n, d_x, batch, h, w, loss, true));
    CD_TRY(zero(c, n->gw.as<float>(), (long long)n->nparam));
    CD_TRY(backward(n, batch, h, w));
    if (host_grad) {
        CD_HIP(c, hipMemcpyAsync(host_grad, n->gw.ptr, sizeof(float) * n->nparam,
                                 hipMemcpyDeviceToHost, c->stream));
    }
    CD_HIP(c, hipStreamSynchronize(c->stream));
    return CD_OK;
}

int cd_net_train_step(cd_net* n, const float* d_x, const float* d_t, int batch, int h, int w,
                      float lr, double* loss) {
    CD_TRY(cd_net_loss_grad(n, d_x, d_t, batch, h, w, loss, nullptr, 0));
    return adam_step(n, lr);
}

int cd_net_train_step_operator(cd_net* n, const float* d_x, int batch, int h, int w, float lr,
                               double* loss) {
    CD_TRY(cd_net_loss_grad_operator(n, d_x, batch, h, w, loss, nullptr, 0));
    return adam_step(n, lr);
}

int cd_context_set_net(cd_context* ctx, cd_net* net) {
    if (!ctx) return CD_ERR_BAD_ARG;
    if (net && net->ctx != ctx) return CD_ERR_BAD_ARG;
    ctx->net = net;
    return CD_OK;
}

}  // extern "C"
