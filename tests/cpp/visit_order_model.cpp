// Host model of the closest-hit loops that do not keep the reference's order of
// visits: leaf tests deferred and flushed at random, and groups of lanes that take
// up to G nodes off a stack of (node, bound) pairs a round.  Same arithmetic as the
// kernels (built without contraction); compared with a walk in the reference's
// order by tests/test_visit_order_model.py.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <random>
#include <utility>
#include <vector>

namespace {

struct V3 {
    float x, y, z;
};
V3 sub(V3 a, V3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
V3 cross(V3 a, V3 b) { return {a.y * b.z - b.y * a.z, a.z * b.x - b.z * a.x, a.x * b.y - b.x * a.y}; }
float dot(V3 a, V3 b) {
    const float x = a.x * b.x, y = a.y * b.y, z = a.z * b.z;
    return (x + y) + z;
}
float lo(float a, float b) { return a < b ? a : b; }
float hi(float a, float b) { return a > b ? a : b; }

constexpr float kEps = 1.192092896e-07f, kInit = 3.4028232635611926e+38f, kInf = HUGE_VALF, kMax = 3.402823466e+38f;
constexpr uint32_t kNone = ~0u;

struct Tri {
    V3 p, e1, e2;
    uint32_t id;
    float box[6];
};
struct Ray {
    V3 o, d, inv;
};
struct Tree {
    std::vector<Tri> tris;
    std::vector<uint32_t> words;
    std::vector<float> boxes;
    const float* box(uint32_t child, bool internal) const { return internal ? &boxes[6 * child] : tris[child].box; }
};

float tri_t(const Ray& r, const Tri& c) {
    const V3 q = cross(r.d, c.e2);
    const float det = dot(c.e1, q);
    if (det > -kEps && det < kEps) return kInf;
    const float inv = 1.0f / det;
    const V3 s = sub(r.o, c.p);
    const float u = inv * dot(s, q);
    if (u < 0.0f) return kInf;
    const V3 k = cross(s, c.e1);
    const float v = inv * dot(r.d, k);
    if (v < 0.0f || (u + v) > 1.0f) return kInf;
    const float t = inv * dot(c.e2, k);
    return t >= 0.0f ? t : kInf;
}

float box_h(const Ray& r, const float* b, bool* nan) {
    const float x0 = (b[0] - r.o.x) * r.inv.x, x1 = (b[3] - r.o.x) * r.inv.x;
    const float y0 = (b[1] - r.o.y) * r.inv.y, y1 = (b[4] - r.o.y) * r.inv.y;
    const float z0 = (b[2] - r.o.z) * r.inv.z, z1 = (b[5] - r.o.z) * r.inv.z;
    if (nan && (x0 != x0 || x1 != x1 || y0 != y0 || y1 != y1 || z0 != z0 || z1 != z1)) *nan = true;
    const float n = hi(hi(lo(x0, x1), lo(y0, y1)), lo(z0, z1)), f = lo(lo(hi(x0, x1), hi(y0, y1)), hi(z0, z1));
    return n <= f && f > 0.0f ? n : kInf;
}

struct Hit {
    float t = kInit;
    uint32_t id = kNone;
    float bound = kInit;
    bool tie = false;
};

// One tested triangle, h the distance of its own box (0: reference's order).
float take(Hit& b, float t, uint32_t id, float h) {
    const float c = hi(hi(t, h), 0.0f), other = hi(t, b.t);
    const bool better = t < b.t || (t == b.t && id < b.id);
    if (better) {
        b.bound = c;
        b.t = t;
        b.id = id;
    }
    if (other < b.bound) b.tie = true;
    return c;
}

// The reference's walk.
Hit in_order(const Tree& T, const Ray& r) {
    Hit b;
    std::vector<uint32_t> stack;
    uint32_t node = 0;
    for (;;) {
        const uint32_t w = T.words[node], l = w >> 2;
        const bool in0 = w & 1u, in1 = w & 2u;
        for (uint32_t k = 0; k < 2; ++k)
            if (!(w >> k & 1u)) take(b, tri_t(r, T.tris[l + k]), T.tris[l + k].id, 0.0f);
        const float h0 = box_h(r, T.box(l, in0), nullptr), h1 = box_h(r, T.box(l + 1, in1), nullptr);
        const bool g0 = in0 && h0 <= b.t, g1 = in1 && h1 <= b.t;
        if (g0 || g1) {
            const bool sw = g1 && (!g0 || h1 < h0);
            if (g0 && g1) stack.push_back(sw ? l : l + 1);
            node = sw ? l + 1 : l;
        } else {
            if (stack.empty()) return b;
            node = stack.back();
            stack.pop_back();
        }
    }
}

// Leaf tests deferred; bare: culled by the best distance so far instead.
Hit deferred(const Tree& T, const Ray& r, std::mt19937& rng, bool bare) {
    Hit b;
    float best = kInit;
    std::vector<uint32_t> stack;
    std::vector<std::pair<uint32_t, float>> noted;
    const uint32_t eager = rng() % 8u;
    uint32_t node = 0;
    bool nan = false, more = true;
    while (more) {
        const uint32_t w = T.words[node], l = w >> 2;
        const bool in0 = w & 1u, in1 = w & 2u;
        const float h0 = box_h(r, T.box(l, in0), &nan), h1 = box_h(r, T.box(l + 1, in1), &nan);
        if (!in0) noted.push_back({l, h0});
        if (!in1) noted.push_back({l + 1, h1});
        const float bound = bare ? best : b.bound;
        const bool g0 = in0 && h0 <= bound, g1 = in1 && h1 <= bound;
        if (g0 || g1) {
            const bool sw = g1 && (!g0 || h1 < h0);
            if (g0 && g1) stack.push_back(sw ? l : l + 1);
            node = sw ? l + 1 : l;
        } else if (stack.empty()) {
            more = false;
        } else {
            node = stack.back();
            stack.pop_back();
        }
        if (!more || noted.size() > 2 || rng() % 8u < eager) {
            for (const auto& p : noted) {
                const float t = tri_t(r, T.tris[p.first]);
                take(b, t, T.tris[p.first].id, p.second);
                best = lo(best, t);
            }
            noted.clear();
        }
    }
    b.tie |= nan;
    return b;
}

// A group of `lanes`, taking up to that many nodes a round (a random number of
// them); bare: all culled by the best distance of any lane.
Hit grouped(const Tree& T, const Ray& r, uint32_t lanes, std::mt19937& rng, bool bare) {
    struct Entry {
        uint32_t node;
        float bound;
    };
    std::vector<Hit> own(lanes);
    std::vector<Entry> stack{{0u, kInit}};
    float best = kInit;
    bool nan = false;
    while (!stack.empty()) {
        uint32_t k = std::min<uint32_t>(lanes, static_cast<uint32_t>(stack.size()));
        if (!bare && (rng() & 1u)) k = 1u + rng() % k;
        const size_t base = stack.size() - k;
        const std::vector<Entry> top(stack.begin() + base, stack.end());
        stack.resize(base);
        std::vector<float> h0(k), h1(k), bound(k);
        for (uint32_t j = 0; j < k; ++j) {
            const uint32_t w = T.words[top[j].node], l = w >> 2;
            h0[j] = box_h(r, T.box(l, w & 1u), &nan);
            h1[j] = box_h(r, T.box(l + 1, w & 2u), &nan);
            bound[j] = top[j].bound;
            for (uint32_t q = 0; q < 2; ++q) {
                if (w >> q & 1u) continue;
                const float t = tri_t(r, T.tris[l + q]);
                bound[j] = lo(bound[j], take(own[j], t, T.tris[l + q].id, q ? h1[j] : h0[j]));
                best = lo(best, t);
            }
        }
        for (uint32_t j = k - 1; j-- > 0;) bound[j] = lo(bound[j], bound[j + 1]);
        if (base > 0) stack[base - 1].bound = lo(stack[base - 1].bound, bound[0]);
        for (uint32_t j = 0; j < k; ++j) {
            const uint32_t w = T.words[top[j].node], l = w >> 2;
            const float p = bare ? best : bound[j];
            const bool g0 = (w & 1u) && h0[j] <= p, g1 = (w & 2u) && h1[j] <= p;
            if (!g0 && !g1) continue;
            const bool sw = g1 && (!g0 || h1[j] < h0[j]);
            if (g0 && g1) stack.push_back({sw ? l : l + 1, p});
            stack.push_back({sw ? l + 1 : l, p});
        }
    }
    Hit b = *std::min_element(own.begin(), own.end(),
                              [](const Hit& x, const Hit& y) { return x.t < y.t || (x.t == y.t && x.id < y.id); });
    for (const Hit& o : own) b.tie |= o.tie || (o.id != b.id && o.id != kNone && o.t < b.bound);
    b.tie |= nan;
    return b;
}

}  // namespace

// counts: rays that hit; deferred: other hits than the reference's with bare
// culling, other hits that are no ties, ties; the same three of groups.
extern "C" void visit_orders(uint32_t n, const float* corners, const uint32_t* ids, const uint32_t* words,
                             const float* boxes, uint32_t nrays, const float* rays, uint32_t seed, uint64_t* counts) {
    Tree T;
    T.tris.resize(n);
    for (uint32_t i = 0; i < n; ++i) {
        const float* v = corners + 9 * static_cast<size_t>(i);
        Tri& c = T.tris[i];
        c.p = {v[0], v[1], v[2]};
        c.e1 = sub({v[3], v[4], v[5]}, c.p);
        c.e2 = sub({v[6], v[7], v[8]}, c.p);
        c.id = ids[i];
        for (int a = 0; a < 3; ++a) {
            c.box[a] = lo(lo(lo(kMax, v[a]), v[3 + a]), v[6 + a]);
            c.box[3 + a] = hi(hi(hi(-kMax, v[a]), v[3 + a]), v[6 + a]);
        }
    }
    T.words.assign(words, words + n - 1);
    T.boxes.assign(boxes, boxes + 6 * static_cast<size_t>(n - 1));
    std::mt19937 rng(seed);
    for (uint32_t i = 0; i < nrays; ++i) {
        const float* v = rays + 6 * static_cast<size_t>(i);
        const Ray r{{v[0], v[1], v[2]}, {v[3], v[4], v[5]}, {1.0f / v[3], 1.0f / v[4], 1.0f / v[5]}};
        const Hit want = in_order(T, r);
        auto other = [&](const Hit& b) { return b.id != want.id || b.t != want.t; };
        auto count = [&](uint64_t* c, const Hit& bare, const Hit& b) {
            c[0] += other(bare);
            c[1] += !b.tie && other(b);
            c[2] += b.tie;
        };
        counts[0] += want.id != kNone;
        count(counts + 1, deferred(T, r, rng, true), deferred(T, r, rng, false));
        const uint32_t lanes = 2u << rng() % 5u;
        count(counts + 4, grouped(T, r, lanes, rng, true), grouped(T, r, lanes, rng, false));
    }
}
