// cone_slab_clear never clears a cone that owns an edge passing the silhouette
// predicate (geom.hpp), for leaves and for merged cones, seen from random
// points near and far.  Prints the number of trials, of clears, and of wrong
// clears.
#define __host__
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_sqrtf(x) std::sqrt(x)
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "../../snch_lbvh_amd/csrc/geom.hpp"

using namespace snch;

struct Edge {
    v3 a, b, n0, n1;
};
struct Node {
    box3 box;
    cone3 cone;
    uint32_t slab;
    std::vector<Edge> edges;
};

static std::mt19937 rng(7);
static float uni(float lo, float hi) { return std::uniform_real_distribution<float>(lo, hi)(rng); }

// the height field of a patch: curved or rough
static v3 surf(float x, float y, float k, float rough, v3 off)
{
    return mk(off.x + x, off.y + y, off.z + k * (x * x + y * y) + rough * std::sin(37.0f * x + 53.0f * y));
}

static Node leaf_of(const v3 (&p)[4])
{
    // triangle p0 p1 p2 owning the edge (p0, p2), whose other face is p0 p2 p3
    Node n;
    n.box = box_of_point(p[0]);
    box_expand(n.box, p[1]);
    box_expand(n.box, p[2]);
    const v3 c = box_centroid(n.box);
    Edge e{p[0], p[2], normalize3(cross3(sub(p[1], p[0]), sub(p[2], p[0]))),
           normalize3(cross3(sub(p[2], p[0]), sub(p[3], p[0])))};
    n.cone.axis = normalize3(mk(e.n0.x + e.n1.x, e.n0.y + e.n1.y, e.n0.z + e.n1.z));
    n.cone.half_angle = dm::acosf_(clamp11(smin(dot3(n.cone.axis, e.n0), dot3(n.cone.axis, e.n1))));
    n.cone.radius = smax(len3(sub(e.a, c)), len3(sub(e.b, c)));
    float h[3];
    for (int k = 0; k < 3; ++k)
        h[k] = dot3(n.cone.axis, sub(p[k], c));
    n.slab = pack_slab(smin(h[0], smin(h[1], h[2])), smax(h[0], smax(h[1], h[2])), n.cone.radius,
                       1e-6f * (smax(dm::fabs_(c.x), smax(dm::fabs_(c.y), dm::fabs_(c.z))) + n.cone.radius));
    n.edges = {e};
    return n;
}

static Node merge(const Node& a, const Node& b)
{
    Node n;
    n.box = box_merge(a.box, b.box);
    n.cone = cone_merge(a.cone, b.cone, box_centroid(a.box), box_centroid(b.box), box_centroid(n.box), true);
    n.slab = slab_merge(n.cone, n.box, a.cone, a.slab, a.box, b.cone, b.slab, b.box);
    n.edges = a.edges;
    n.edges.insert(n.edges.end(), b.edges.begin(), b.edges.end());
    return n;
}

int main()
{
    long trials = 0, clears = 0, wrong = 0;
    const float offs[3] = {0.0f, 3.0f, 50.0f};
    for (int t = 0; t < 4000; ++t) {
        const float k = uni(-2.0f, 2.0f), rough = t % 3 == 0 ? uni(0.0f, 0.01f) : 0.0f, s = std::pow(10.0f, uni(-3.0f, 0.0f));
        const v3 off = mk(offs[t % 3], -offs[t % 3], 0.5f * offs[t % 3]);
        std::vector<Node> level;
        const int m = 4;
        for (int i = 0; i < m; ++i)
            for (int j = 0; j < m; ++j) {
                const float x = s * i / m, y = s * j / m, d = s / m;
                const v3 p[4] = {surf(x, y, k, rough, off), surf(x + d, y, k, rough, off),
                                 surf(x + d, y + d, k, rough, off), surf(x, y + d, k, rough, off)};
                level.push_back(leaf_of(p));
            }
        std::vector<Node> all = level;
        while (level.size() > 1) {
            std::vector<Node> up;
            for (size_t i = 0; i + 1 < level.size(); i += 2)
                up.push_back(merge(level[i], level[i + 1]));
            all.insert(all.end(), up.begin(), up.end());
            level = up;
        }
        for (int q = 0; q < 200; ++q) {
            const float r = s * std::pow(10.0f, uni(-2.0f, 2.0f));
            const v3 o = mk(off.x + 0.5f * s + uni(-r, r), off.y + 0.5f * s + uni(-r, r), off.z + uni(-r, r));
            for (const Node& n : all) {
                float sn, cs;
                dm::sincosf_(n.cone.half_angle, &sn, &cs);
                ++trials;
                if (!cone_slab_clear(n.cone.axis, n.cone.half_angle, sn, cs, n.cone.radius, n.slab, o, n.box))
                    continue;
                ++clears;
                for (const Edge& e : n.edges)
                    for (int flip = 0; flip < 2; ++flip) {
                        v3 cp;
                        const float d = closest_point_segment(e.a, e.b, o, cp);
                        wrong += is_silhouette_edge(e.a, e.b, e.n0, e.n1, sub(o, cp), d, flip != 0) ? 1 : 0;
                    }
            }
        }
    }
    std::printf("%ld %ld %ld\n", trials, clears, wrong);
    return 0;
}
