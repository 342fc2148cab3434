// cone_slab_clear (geom.hpp) where some leaves own no edges: a cone merged with
// an empty one keeps its radius while its box, and the centre that everything
// is measured from, change.  Prints the number of trials, of clears, and of
// cleared cones' edges that pass the silhouette predicate.
#define main slab_check_main
#include "slab_check.cpp"
#undef main

int main()
{
    long trials = 0, clears = 0, wrong = 0;
    for (int t = 0; t < 3000; ++t) {
        const float k = uni(-2.0f, 2.0f), rough = t % 3 == 0 ? uni(0.0f, 0.01f) : 0.0f, s = std::pow(10.0f, uni(-3.0f, 0.0f));
        const float empty = t % 2 ? 0.3f : 0.8f;
        std::vector<Node> level;
        for (int q = 0; q < 64; ++q) { // cells of an 8 x 8 patch in Morton order
            const int i = (q & 1) | (q >> 1 & 2) | (q >> 2 & 4), j = (q >> 1 & 1) | (q >> 2 & 2) | (q >> 3 & 4);
            const float d = s / 8, x = d * i, y = d * j;
            const v3 off = mk(0.0f, 0.0f, 0.0f);
            const v3 p[4] = {surf(x, y, k, rough, off), surf(x + d, y, k, rough, off), surf(x + d, y + d, k, rough, off),
                             surf(x, y + d, k, rough, off)};
            Node n = leaf_of(p);
            if (uni(0.0f, 1.0f) < empty) { // a triangle, maybe a longer one, whose edges others own
                const float g = uni(0.0f, 1.0f) < 0.3f ? uni(0.0f, 3.0f) : 0.0f;
                n.cone = cone3{mk(0.0f, 0.0f, 0.0f), -F_PI, 0.0f};
                n.slab = SLAB_ALL;
                n.edges.clear();
                n.box.hi = mk(n.box.hi.x + g * d, n.box.hi.y, n.box.hi.z + 0.1f * g * d);
                n.box.lo.y -= g * d;
            }
            level.push_back(n);
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
            v3 o = mk(0.5f * s + uni(-r, r), 0.5f * s + uni(-r, r), uni(-r, r));
            if (q % 2) // near the patch's plane
                o.z = 0.5f * k * s * s + uni(-0.1f, 0.1f) * r;
            for (const Node& n : all) {
                if (!cone_valid(n.cone.half_angle))
                    continue;
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
