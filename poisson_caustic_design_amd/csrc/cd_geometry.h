// Device geometry primitives of the caustic-design path (FP64).  Operation
// order follows the reference expressions so that, compiled without FP
// contraction, results match the FP64 CPU restatement bit for bit.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

namespace cdgeo {

// Structured triangulation of src/mesh.cpp:57-63: cell (i,j) with base vertex
// idx = i*mx + j holds triangle 2k = {idx, idx+1, idx+mx} and
// 2k+1 = {idx+mx, idx+1, idx+mx+1}, k = i*(mx-1) + j.
__device__ __forceinline__ void tri_vertices(int mx, int t, int& a, int& b, int& c) {
    const int cell = t >> 1;
    const int cw = mx - 1;
    const int i = cell / cw, j = cell - i * cw;
    const int idx = i * mx + j;
    if ((t & 1) == 0) { a = idx; b = idx + 1; c = idx + mx; }
    else { a = idx + mx; b = idx + 1; c = idx + mx + 1; }
}

// Triangles adjacent to vertex (x,y), ascending triangle index; returns count.
__device__ __forceinline__ int adjacent_triangles(int mx, int my, int x, int y, int* out) {
    int n = 0;
    const int cw = mx - 1;
    if (y > 0 && x > 0) out[n++] = 2 * ((y - 1) * cw + (x - 1)) + 1;
    if (y > 0 && x < mx - 1) { out[n++] = 2 * ((y - 1) * cw + x); out[n++] = 2 * ((y - 1) * cw + x) + 1; }
    if (y < my - 1 && x > 0) { out[n++] = 2 * (y * cw + (x - 1)); out[n++] = 2 * (y * cw + (x - 1)) + 1; }
    if (y < my - 1 && x < mx - 1) out[n++] = 2 * (y * cw + x);
    return n;
}

// Quad (v_i, mid(ij), centroid(ijk), mid(ik)) of vertex vi in triangle t
// (src/mesh.cpp:174-199); q receives x0,y0,...,x3,y3.
__device__ __forceinline__ void triangle_quad(int mx, const double* __restrict__ xy, int vi, int t,
                                              double* q) {
    int v[3];
    tri_vertices(mx, t, v[0], v[1], v[2]);
    const int p = (v[0] == vi) ? 0 : ((v[1] == vi) ? 1 : 2);
    const int vj = v[(p + 1) % 3], vk = v[(p + 2) % 3];
    const double ax = xy[2 * vi], ay = xy[2 * vi + 1];
    const double bx = xy[2 * vj], by = xy[2 * vj + 1];
    const double cx = xy[2 * vk], cy = xy[2 * vk + 1];
    q[0] = ax; q[1] = ay;
    q[2] = (ax + bx) / 2.0; q[3] = (ay + by) / 2.0;
    q[4] = (ax + bx + cx) / 3.0; q[5] = (ay + by + cy) / 3.0;
    q[6] = (ax + cx) / 2.0; q[7] = (ay + cy) / 2.0;
}

// Signed shoelace area, summation order of polygon_utils.cpp:216-236.
__device__ __forceinline__ double shoelace4(const double* p) {
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int k = (i + 1) & 3;
        s += p[2 * i] * p[2 * k + 1] - p[2 * k] * p[2 * i + 1];
    }
    return 0.5 * s;
}

// Barycentric coordinates (u weights a, v weights b, w = 1-u-v weights c) of
// point p in triangle (a,b,c): the formula of bvh.cpp:162-190 applied with
// (t0,t1,t2) = (c,b,a) as at bvh.cpp:262.
__device__ __forceinline__ void barycentric(double ax, double ay, double bx, double by, double cx,
                                            double cy, double px, double py, double& u, double& v,
                                            double& w) {
    const double v0x = ax - cx, v0y = ay - cy;
    const double v1x = bx - cx, v1y = by - cy;
    const double v2x = px - cx, v2y = py - cy;
    const double d00 = v0x * v0x + v0y * v0y;
    const double d01 = v0x * v1x + v0y * v1y;
    const double d02 = v0x * v2x + v0y * v2y;
    const double d11 = v1x * v1x + v1y * v1y;
    const double d12 = v1x * v2x + v1y * v2y;
    const double den = d00 * d11 - d01 * d01;
    const double inv = 1 / den;
    u = (d11 * d02 - d01 * d12) * inv;
    v = (d00 * d12 - d01 * d02) * inv;
    w = 1.0 - u - v;
}

// inside test of bvh.cpp:264 (eps 1e-12)
__device__ __forceinline__ bool inside(double u, double v) {
    const double eps = 1e-12;
    return u >= -eps && v >= -eps && (u + v) <= 1.0 + eps;
}

// Bilinear lookup with floor/ceil and clamp-to-edge (caustic_design.cpp:156-188).
template <typename F>
__device__ __forceinline__ double bilinear(F at, int w, int h, double x, double y) {
    int x0 = (int)floor(x), y0 = (int)floor(y);
    int x1 = (int)ceil(x), y1 = (int)ceil(y);
    x0 = min(max(x0, 0), w - 1);
    x1 = min(max(x1, 0), w - 1);
    y0 = min(max(y0, 0), h - 1);
    y1 = min(max(y1, 0), h - 1);
    const double fx1 = x - x0, fx0 = 1.0 - fx1;
    const double fy1 = y - y0, fy0 = 1.0 - fy1;
    const double top = fx0 * at(x0, y0) + fx1 * at(x1, y0);
    const double bot = fx0 * at(x0, y1) + fx1 * at(x1, y1);
    return fy0 * top + fy1 * bot;
}

// ---- convex clipping (Sutherland-Hodgman) ---------------------------------
// A subject vertex is kept unless strictly on the outer side of the clip edge;
// a crossing is emitted only for strictly opposite consecutive vertices with
// crossing parameter strictly inside (0,1) (polygon_utils.cpp:43-60, 94-116).
// A side adds at most one vertex to a convex polygon, so three leave 7; 10 has room
// for a further pair, where rounding puts a crossing beyond its segment's end and
// the next side lies between the two.
constexpr int CLIP_MAX = 10;

struct Pt {
    double x, y;
};

// The clip edges are the sides of a pixel square, so the side of a vertex, the
// sign of a cross product with one zero term (polygon_utils.cpp:33-41), is one
// comparison of its coordinate with c, and numerator and denominator of the
// crossing parameter keep one product each, with the square's extent w along the
// edge: bit-equal to the full products.
// Segment s->e of a polygon against one side: AXIS 0: x against c, 1: y; LOW: kept
// at or above c, else at or below.  m vertices were emitted before; returns how many
// were after.
template <int AXIS, bool LOW, typename Emit>
__device__ __forceinline__ int clip_segment(const Pt& s, const Pt& e, double c, double w, int m,
                                            Emit emit) {
    const double su = AXIS ? s.y : s.x, eu = AXIS ? e.y : e.x;
    if (!(LOW ? su < c : su > c) && m < CLIP_MAX) emit(m++, s);
    if (((su < c && eu > c) || (su > c && eu < c)) && m < CLIP_MAX) {
        const double dx = e.x - s.x, dy = e.y - s.y;
        const double den = (AXIS ? dy : dx) * w;
        const double t = ((c - su) * w) / den;
        if (den != 0.0 && t > 0 && t < 1) emit(m++, Pt{s.x + t * dx, s.y + t * dy});
    }
    return m;
}

// the polygon of n vertices that load(i) gives; the next vertex's load is issued
// before the current segment is worked on
template <int AXIS, bool LOW, typename Load, typename Emit>
__device__ __forceinline__ int clip_side(int n, double c, double w, Load load, Emit emit) {
    int m = 0;
    Pt s = load(n - 1), next = load(0);
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
        const Pt e = next;
        next = load(i + 1 < n ? i + 1 : i);
        m = clip_segment<AXIS, LOW>(s, e, c, w, m, emit);
        s = e;
    }
    return m;
}

// Signed area of quad q (4 vertices) intersected with the pixel square of side
// px centred at (cx, cy), its sides taken in the order of
// polygon_utils.cpp:336-346.  Vertex i of the two work polygons is a[i * S] and
// b[i * S] (CLIP_MAX vertices each; S = 64: one column per lane of a wave).  The
// first side takes the quad from registers, and the last side's polygon is not
// stored: its area is summed as its vertices come.
template <int S>
__device__ __forceinline__ double quad_pixel_area(const double* q, double cx, double cy, double px,
                                                  Pt* a, Pt* b) {
    const double l = cx - px / 2.0, r = cx + px / 2.0, lo = cy - px / 2.0, hi = cy + px / 2.0;
    const double w = r - l, h = hi - lo;
    auto to = [](Pt* p) { return [p](int m, Pt v) { p[m * S] = v; }; };
    auto from = [](const Pt* p) { return [p](int i) { return p[i * S]; }; };
    int n = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int k = (i + 3) & 3;
        n = clip_segment<1, true>(Pt{q[2 * k], q[2 * k + 1]}, Pt{q[2 * i], q[2 * i + 1]}, lo, w, n,
                                  to(b));
    }
    if (n == 0) return 0.0;
    n = clip_side<0, true>(n, l, h, from(b), to(a));
    if (n == 0) return 0.0;
    n = clip_side<1, false>(n, hi, w, from(a), to(b));
    if (n == 0) return 0.0;
    Pt first = {0.0, 0.0}, prev = {0.0, 0.0};
    double sum = 0.0;
    n = clip_side<0, false>(n, r, h, from(b), [&](int m, Pt v) {
        if (m == 0) first = v;
        else sum += prev.x * v.y - v.x * prev.y;
        prev = v;
    });
    if (n < 3) return 0.0;
    sum += prev.x * first.y - first.x * prev.y;
    return 0.5 * sum;
}

}  // namespace cdgeo
