// Host part of scene compilation: the welded edge candidates of a mesh and the
// convex hulls of its coplanar groups (what the public call does before any
// kernel runs). Plain C++ on host arrays; no device work, no HIP.
#include "wc_error.h"
#include "../../include/wcmi.h"

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <numeric>
#include <vector>

namespace wc {
namespace {

struct EdgeKey {
    int64_t v[6];  // the two welded end points, the lexicographically lower first
    bool operator==(const EdgeKey& o) const { return std::memcmp(v, o.v, sizeof(v)) == 0; }
};

uint64_t hash_key(const EdgeKey& k) {
    uint64_t h = 0x9E3779B97F4A7C15ull;
    for (int64_t x : k.v) {
        h ^= (uint64_t)x;
        h *= 0xFF51AFD7ED558CCDull;
        h ^= h >> 32;
    }
    return h;
}

struct EdgeEntry {
    EdgeKey key;
    int uses;      // face edges on this key
    int first[2];  // the first two of them, 3 f + k
};

struct P2 {
    double x, y;
};

// A host array's index, from its end where negative; -1 outside the array.
int64_t array_index(int64_t i, int64_t count) {
    if (i < 0) i += count;
    return i >= 0 && i < count ? i : -1;
}

// hull of points sorted by (x, y), as the monotone chain builds one side
void half_hull(const std::vector<P2>& seq, std::vector<P2>& out) {
    out.clear();
    for (const P2& p : seq) {
        while (out.size() >= 2) {
            const P2 &a = out[out.size() - 2], &b = out.back();
            if (!((b.x - a.x) * (p.y - a.y) - (b.y - a.y) * (p.x - a.x) <= 0.0)) break;
            out.pop_back();
        }
        out.push_back(p);
    }
}

}  // namespace
}  // namespace wc

using namespace wc;

extern "C" int wc_edge_candidates(const long long* welded, int vertex_count, const int* faces, int face_count,
                                  const long long* face_structure, const long long* structure_vertex_base,
                                  int structure_count, const int* face_group, const int* face_material,
                                  long long* vertex_ids, long long* face_ids, long long* public_ids, int* count) {
    if (vertex_count < 0 || face_count < 0 || structure_count < 0)
        return wc_fail("wc_edge_candidates: sizes must be non-negative");
    if (!count) return wc_fail("wc_edge_candidates: count is null");
    *count = 0;
    if (face_count == 0) return 0;
    if (!welded || !faces || !face_structure || !structure_vertex_base || !face_group || !face_material ||
        !vertex_ids || !face_ids || !public_ids)
        return wc_fail("wc_edge_candidates: null argument");
    if (face_count > 0x7fffffff / 6) return wc_fail("wc_edge_candidates: too many faces (%d)", face_count);
    try {
        const int n = 3 * face_count;
        for (int f = 0; f < face_count; ++f)
            if (face_structure[f] < 0 || face_structure[f] >= structure_count)
                return wc_fail("wc_edge_candidates: face %d belongs to structure %lld of %d", f, face_structure[f],
                               structure_count);
        for (int i = 0; i < n; ++i)
            if (array_index(faces[i], vertex_count) < 0)
                return wc_fail("wc_edge_candidates: face %d names vertex %d of %d", i / 3, faces[i], vertex_count);
        auto corner = [&](int e, int k) { return faces[3 * (e / 3) + (e % 3 + k) % 3]; };
        // public id of a face edge: the rank of its (structure, lower, higher local vertex) among the distinct ones
        struct Record {
            int64_t s, a, b;
            int e;
        };
        std::vector<Record> records((size_t)n);
        for (int e = 0; e < n; ++e) {
            const int64_t s = face_structure[e / 3], base = structure_vertex_base[s];
            const int64_t a = corner(e, 0) - base, b = corner(e, 1) - base;
            records[e] = {s, std::min(a, b), std::max(a, b), e};
        }
        std::sort(records.begin(), records.end(), [](const Record& x, const Record& y) {
            return x.s != y.s ? x.s < y.s : (x.a != y.a ? x.a < y.a : x.b < y.b);
        });
        std::vector<int64_t> id((size_t)n);
        int64_t rank = -1;
        for (int i = 0; i < n; ++i) {
            const Record& r = records[i];
            if (i == 0 || r.s != records[i - 1].s || r.a != records[i - 1].a || r.b != records[i - 1].b) ++rank;
            id[r.e] = rank;
        }
        // face edges by welded end points, in order of first appearance
        size_t slots = 16;
        while (slots < 2 * (size_t)n) slots <<= 1;
        std::vector<int> table(slots, -1);
        std::vector<EdgeEntry> entries;
        entries.reserve((size_t)n);
        for (int e = 0; e < n; ++e) {
            const long long *a = welded + 3 * array_index(corner(e, 0), vertex_count),
                            *b = welded + 3 * array_index(corner(e, 1), vertex_count);
            if (std::lexicographical_compare(b, b + 3, a, a + 3)) std::swap(a, b);
            EdgeKey key;
            for (int k = 0; k < 3; ++k) {
                key.v[k] = a[k];
                key.v[3 + k] = b[k];
            }
            size_t slot = hash_key(key) & (slots - 1);
            while (table[slot] >= 0 && !(entries[table[slot]].key == key)) slot = (slot + 1) & (slots - 1);
            if (table[slot] < 0) {
                table[slot] = (int)entries.size();
                entries.push_back({key, 1, {e, -1}});
            } else {
                EdgeEntry& t = entries[table[slot]];
                if (t.uses == 1) t.first[1] = e;
                ++t.uses;
            }
        }
        int out = 0;
        for (const EdgeEntry& t : entries) {
            if (t.uses > 2) continue;
            const int e0 = t.first[0], e1 = t.first[1], f0 = e0 / 3, f1 = e1 >= 0 ? e1 / 3 : -1;
            if (f1 >= 0 && face_group[f1] == face_group[f0]) continue;
            long long* v = vertex_ids + 4 * (size_t)out;
            v[0] = corner(e0, 0);
            v[1] = corner(e0, 1);
            v[2] = corner(e0, 2);
            v[3] = f1 >= 0 ? corner(e1, 2) : -1;
            long long* i = face_ids + 6 * (size_t)out;
            i[0] = f0;
            i[1] = f1;
            i[2] = face_group[f0];
            i[3] = f1 >= 0 ? face_group[f1] : -1;
            i[4] = face_material[f0];
            i[5] = f1 >= 0 ? face_material[f1] : -1;
            public_ids[out] = f1 >= 0 ? std::min(id[e0], id[e1]) : id[e0];
            ++out;
        }
        *count = out;
    } catch (const std::exception& e) {
        return wc_fail("wc_edge_candidates: %s", e.what());
    }
    return 0;
}

extern "C" int wc_group_hulls(const double* vertices, int vertex_count, const int* faces, int face_count,
                              const int* group_face_offset, const int* group_faces, int listed_count,
                              const double* group_plane, int group_count, int* hull_offset, double* hull_points) {
    if (vertex_count < 0 || face_count < 0 || listed_count < 0 || group_count < 0 || !hull_offset)
        return wc_fail("wc_group_hulls: invalid arguments");
    hull_offset[0] = 0;
    if (group_count == 0) return 0;
    if (!vertices || !faces || !group_face_offset || !group_faces || !group_plane || !hull_points)
        return wc_fail("wc_group_hulls: null argument");
    for (int g = 0; g < group_count; ++g)
        if (group_face_offset[g] < 0 || group_face_offset[g] > group_face_offset[g + 1] ||
            group_face_offset[g + 1] > listed_count)
            return wc_fail("wc_group_hulls: group %d lists faces %d to %d of %d", g, group_face_offset[g],
                           group_face_offset[g + 1], listed_count);
    for (int i = group_face_offset[0]; i < group_face_offset[group_count]; ++i) {
        const int64_t f = array_index(group_faces[i], face_count);
        if (f < 0) return wc_fail("wc_group_hulls: face %d of %d is listed", group_faces[i], face_count);
        for (int k = 0; k < 3; ++k)
            if (array_index(faces[3 * f + k], vertex_count) < 0)
                return wc_fail("wc_group_hulls: face %lld names vertex %d of %d", (long long)f, faces[3 * f + k],
                               vertex_count);
    }
    try {
        std::vector<P2> pts, rev, lower, upper;
        size_t total = 0;
        for (int g = 0; g < group_count; ++g) {
            const double* n = group_plane + 4 * (size_t)g;
            // in-plane basis: u orthogonal to n, w = n x u
            const bool x_axis = std::fabs(n[0]) < 0.9;
            double u[3] = {0.0, x_axis ? n[2] : 0.0, x_axis ? -n[1] : 0.0};
            if (!x_axis) {
                u[0] = -n[2];
                u[2] = n[0];
            }
            const double len = std::sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
            for (double& c : u) c /= len;
            const double w[3] = {n[1] * u[2] - n[2] * u[1], n[2] * u[0] - n[0] * u[2], n[0] * u[1] - n[1] * u[0]};
            const double o[3] = {n[0] * n[3], n[1] * n[3], n[2] * n[3]};
            const int begin = group_face_offset[g], end = group_face_offset[g + 1];
            pts.clear();
            bool finite = true;
            for (int i = begin; i < end; ++i) {
                const int* face = faces + 3 * array_index(group_faces[i], face_count);
                for (int k = 0; k < 3; ++k) {
                    const double* p = vertices + 3 * array_index(face[k], vertex_count);
                    const double d[3] = {p[0] - o[0], p[1] - o[1], p[2] - o[2]};
                    const P2 q{d[0] * u[0] + d[1] * u[1] + d[2] * u[2], d[0] * w[0] + d[1] * w[1] + d[2] * w[2]};
                    finite = finite && std::isfinite(q.x) && std::isfinite(q.y);
                    pts.push_back(q);
                }
            }
            if (end - begin == 1) {
                const double area = (pts[1].x - pts[0].x) * (pts[2].y - pts[0].y) -
                                    (pts[1].y - pts[0].y) * (pts[2].x - pts[0].x);
                if (area < 0.0) std::reverse(pts.begin(), pts.end());
            } else if (!pts.empty()) {
                if (finite) {
                    std::sort(pts.begin(), pts.end(),
                              [](const P2& a, const P2& b) { return a.x != b.x ? a.x < b.x : a.y < b.y; });
                    pts.erase(std::unique(pts.begin(), pts.end(),
                                          [](const P2& a, const P2& b) { return a.x == b.x && a.y == b.y; }),
                              pts.end());
                }
                if (pts.size() >= 3) {
                    rev.assign(pts.rbegin(), pts.rend());
                    half_hull(pts, lower);
                    half_hull(rev, upper);
                    pts.assign(lower.begin(), lower.end() - 1);
                    pts.insert(pts.end(), upper.begin(), upper.end() - 1);
                }
            }
            for (const P2& q : pts) {
                double* out = hull_points + 3 * total++;
                for (int k = 0; k < 3; ++k) out[k] = o[k] + q.x * u[k] + q.y * w[k];
            }
            hull_offset[g + 1] = (int)total;
        }
    } catch (const std::exception& e) {
        return wc_fail("wc_group_hulls: %s", e.what());
    }
    return 0;
}
