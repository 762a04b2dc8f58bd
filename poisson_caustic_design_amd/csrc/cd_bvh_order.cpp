// First-hit order of the reference's triangle BVH, on the host.
//
// The reference locates raster samples and grid vertices in a mesh with a
// bounding-volume hierarchy (bvh.cpp): Bvh::build (bvh.cpp:20-48) partitions
// an array of triangle ids recursively (bvh.cpp:78-155: bounding box of the
// range's vertices, widened by half an epsilon, split at the middle of its
// longer side, leaves of at most 5 triangles or depth 30, mesh.cpp:235,292,349)
// and Bvh::query (bvh.cpp:196-266) walks the tree depth first, first child
// first, and returns the first triangle of a leaf that holds the point.  The
// leaves cover consecutive ranges of the partitioned array in walk order, and
// every box on the way to a triangle's leaf holds the triangle's own box, so
// the triangle returned for a point is the containing triangle with the
// lowest position in the partitioned array.  This file computes that array;
// the rasterization kernels then keep, per sample, the containing triangle of
// lowest position instead of lowest index (the two differ only where
// triangles overlap, i.e. on folded meshes, and on shared edges).
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <exception>
#include <limits>
#include <new>
#include <thread>
#include <utility>
#include <vector>

#include "cd_api.h"

namespace {

constexpr int kLeafSize = 5;   // build_target_bvh(5, 30), mesh.cpp:235
constexpr int kMaxDepth = 30;
// Ranges of at least kParallel triangles at the first kParallelDepth levels take
// a thread for one half (at most 7 more): a thread costs about 20 us, the build
// of 8192 triangles about 500.
constexpr int kParallel = 8192;
constexpr int kParallelDepth = 3;

// A triangle as the build sees it; the array is permuted with the ids, so that
// every pass over a range reads memory in order.
struct Tri {
    double c[2];           // centroid
    double mn[2], mx[2];   // bounding box of the vertices
    int id;
};

// std::fmin / std::fmax against a bound that is never NaN: a NaN v keeps it.
inline double lower(double bound, double v) { return v < bound ? v : bound; }
inline double upper(double bound, double v) { return v > bound ? v : bound; }

struct OrderBuilder {
    const double* xy;
    int mx, T;
    std::vector<Tri> tri;

    void vertices(int t, int v[3]) const {  // mesh.cpp:57-63
        const int cell = t >> 1, cw = mx - 1;
        const int i = cell / cw, j = cell - i * cw, idx = i * mx + j;
        if ((t & 1) == 0) { v[0] = idx; v[1] = idx + 1; v[2] = idx + mx; }
        else { v[0] = idx + mx; v[1] = idx + 1; v[2] = idx + mx + 1; }
    }

    // area-weighted polygon centroid, polygon_utils.cpp:238-263 (a triangle
    // of zero area yields non-finite coordinates there as here), and the box
    Tri triangle(int t) const {
        int v[3];
        vertices(t, v);
        const double inf = std::numeric_limits<double>::infinity();
        Tri r{{0.0, 0.0}, {inf, inf}, {-inf, -inf}, t};
        double sa = 0.0, sx = 0.0, sy = 0.0;
        for (int k = 0; k < 3; ++k) {
            const double x0 = xy[2 * v[k]], y0 = xy[2 * v[k] + 1];
            const double x1 = xy[2 * v[(k + 1) % 3]], y1 = xy[2 * v[(k + 1) % 3] + 1];
            const double a = x0 * y1 - x1 * y0;
            sa += a;
            sx += (x0 + x1) * a;
            sy += (y0 + y1) * a;
            r.mn[0] = lower(r.mn[0], x0);
            r.mn[1] = lower(r.mn[1], y0);
            r.mx[0] = upper(r.mx[0], x0);
            r.mx[1] = upper(r.mx[1], y0);
        }
        sa *= 0.5;
        r.c[0] = sx / (6 * sa);
        r.c[1] = sy / (6 * sa);
        return r;
    }

    // two-sided partition of bvh.cpp:50-76; the split value arrives as float.
    // next: the centroid coordinate after the range's last entry.
    int split(int start, int end, int dim, float split_value, double next) {
        const double s = split_value;
        Tri* t = tri.data();
        int left = start, right = end - 1;
        while (left < right) {
            while (left < end && t[left].c[dim] < s) ++left;
            while (right >= start && t[right].c[dim] >= s) --right;
            if (left >= right) break;
            std::swap(t[left], t[right]);
            ++left;
            --right;
        }
        // the reference reads the centroid at `left` even when left == end
        const double cl = left < end ? t[left].c[dim] : next;
        return cl <= s ? std::min(end, left + 1) : left;
    }

    // next: the centroid of the entry after the range.  The walk takes the
    // first half before the second, so while a range is being partitioned that
    // entry is the one its ancestors' splits put there: a value of the call,
    // which lets the halves go in parallel.  Past the array's end (undefined in
    // the reference) it is NaN, not below any split value.
    // (Nothing in here throws: a thread that cannot be had, for whatever reason, only
    // leaves its half to this one.)
    void node(int start, int end, int level, const double next[2]) noexcept {
        const double inf = std::numeric_limits<double>::infinity();
        double mn[2] = {inf, inf}, mx_[2] = {-inf, -inf};
        if (end - start <= kLeafSize || level >= kMaxDepth) return;
        for (int i = start; i < end; ++i)
            for (int d = 0; d < 2; ++d) {
                mn[d] = lower(mn[d], tri[i].mn[d]);
                mx_[d] = upper(mx_[d], tri[i].mx[d]);
            }
        for (int d = 0; d < 2; ++d) {
            mn[d] -= 0.5 * DBL_EPSILON;
            mx_[d] += 0.5 * DBL_EPSILON;
        }
        const int dim = (mx_[0] - mn[0]) < (mx_[1] - mn[1]) ? 1 : 0;
        const int m = split(start, end, dim, (float)(0.5 * (mx_[dim] + mn[dim])), next[dim]);
        if (m == start || m == end) return;
        const double mid[2] = {tri[m].c[0], tri[m].c[1]};
        if (end - start >= kParallel && level < kParallelDepth) {
            std::thread first;
            try {
                first = std::thread([&] { node(start, m, level + 1, mid); });
            } catch (const std::exception&) {  // no thread or memory: one after the other
            }
            if (first.joinable()) {
                node(m, end, level + 1, next);
                first.join();
                return;
            }
        }
        node(start, m, level + 1, mid);
        node(m, end, level + 1, next);
    }
};

}  // namespace

extern "C" int cd_bvh_first_hit_order(const double* xy, int mx, int my, int* order) {
    if (!xy || !order || mx < 2 || my < 2) return CD_ERR_BAD_ARG;
    const long long T = 2LL * (mx - 1) * (my - 1);
    if (T > (long long)std::numeric_limits<int>::max() / 2) return CD_ERR_BAD_ARG;
    try {
        OrderBuilder b{xy, mx, (int)T, {}};
        b.tri.reserve((size_t)T);
        for (int t = 0; t < (int)T; ++t) b.tri.push_back(b.triangle(t));
        const double nan = std::numeric_limits<double>::quiet_NaN(), past[2] = {nan, nan};
        b.node(0, (int)T, 0, past);
        for (int t = 0; t < (int)T; ++t) order[t] = b.tri[t].id;
    } catch (const std::bad_alloc&) {
        return CD_ERR_OOM;
    }
    return CD_OK;
}
