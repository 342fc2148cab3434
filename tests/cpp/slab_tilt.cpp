// cone_slab_clear (geom.hpp) where chains of merges lose small angles: patches of
// 2^14 leaves, each tilted by a few units of 3e-4 radians (the set bits of its
// number), and gently curved ones, seen along the faces that lie farthest
// outside their cones.  Prints the number of trials, of clears, of cleared
// cones' edges that pass the silhouette predicate, and the largest excess of a
// normal over its cone's half angle in units of 1e-6.
#define main slab_check_main
#include "slab_check.cpp"
#undef main

static double angle_to(v3 a, v3 n)
{
    const v3 c = cross3(a, n);
    return std::atan2(std::sqrt((double)c.x * c.x + (double)c.y * c.y + (double)c.z * c.z),
                      (double)a.x * n.x + (double)a.y * n.y + (double)a.z * n.z);
}

int main()
{
    constexpr int K = 14, side = 1 << (K / 2);
    long trials = 0, clears = 0, wrong = 0;
    double worst = 0.0;
    const float tilts[] = {2.5e-4f, 3e-4f, 3.1e-4f, 3.4e-4f, 5e-4f, 0.0f, 0.0f, 0.0f};
    const float curves[] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.01f, 0.03f, 0.3f};
    for (int m = 0; m < 8; ++m) {
        std::vector<Node> leaves;
        for (int i = 0; i < 1 << K; ++i) {
            int x = 0, y = 0;
            for (int b = 0; b < K / 2; ++b) {
                x |= (i >> (2 * b) & 1) << b;
                y |= (i >> (2 * b + 1) & 1) << b;
            }
            const float s = 1.0f / side, X = x * s, Y = y * s, k = curves[m];
            const float slope = std::tan(tilts[m] * __builtin_popcount(i));
            v3 p[4] = {mk(X, Y, 0), mk(X + s, Y, 0), mk(X + s, Y + s, 0), mk(X, Y + s, 0)};
            for (v3& v : p)
                v.z = (v.x - X - 0.5f * s) * slope + k * (v.x * v.x + v.y * v.y);
            if (k == 0.0f) {
                p[1].z -= 2e-4f * s;
                p[3].z -= 2e-4f * s;
            }
            leaves.push_back(leaf_of(p));
            float s2 = 0.0f; // the leaf's own excess, as the build takes it
            for (v3 n : {leaves.back().edges[0].n0, leaves.back().edges[0].n1})
                s2 = smax(s2, sqlen3(cross3(leaves.back().cone.axis, n)));
            leaves.back().slab |= excess_units(asin_bound(std::sqrt(s2)) - leaves.back().cone.half_angle + 1e-6f) << 13;
        }
        std::vector<Node> level = leaves;
        for (auto& n : level)
            n.edges.clear();
        for (int l = 1; level.size() > 1; ++l) {
            std::vector<Node> up;
            for (size_t i = 0; i + 1 < level.size(); i += 2)
                up.push_back(merge(level[i], level[i + 1]));
            level = up;
            for (size_t k = 0; k < level.size(); ++k) {
                const Node& n = level[k];
                double far = -1.0;
                const Edge* e = nullptr;
                for (size_t i = k << l; i < (k + 1) << l; ++i)
                    for (const Edge& x : leaves[i].edges)
                        for (v3 nn : {x.n0, x.n1}) {
                            const double a = angle_to(n.cone.axis, nn) - n.cone.half_angle;
                            if (a > far) {
                                far = a;
                                e = &x;
                            }
                        }
                worst = std::max(worst, far);
                if (l < 4 || k >= 64)
                    continue;
                float sn, cs;
                dm::sincosf_(n.cone.half_angle, &sn, &cs);
                for (int q = 0; q < 200; ++q) { // views along the faces of that edge
                    const v3 nm = normalize3(mk(e->n0.x + e->n1.x, e->n0.y + e->n1.y, e->n0.z + e->n1.z));
                    const v3 mid = mk(0.5f * (e->a.x + e->b.x), 0.5f * (e->a.y + e->b.y), 0.5f * (e->a.z + e->b.z));
                    v3 t = mk(uni(-1, 1), uni(-1, 1), 0.0f);
                    const float tn = dot3(t, nm), R = std::pow(10.0f, uni(-1.0f, 3.0f)), up1 = uni(-1e-4f, 1e-4f) * R;
                    t = normalize3(mk(t.x - tn * nm.x, t.y - tn * nm.y, t.z - tn * nm.z));
                    const v3 o = mk(mid.x + R * t.x + up1 * nm.x, mid.y + R * t.y + up1 * nm.y, mid.z + R * t.z + up1 * nm.z);
                    ++trials;
                    if (!cone_slab_clear(n.cone.axis, n.cone.half_angle, sn, cs, n.cone.radius, n.slab, o, n.box))
                        continue;
                    ++clears;
                    for (int flip = 0; flip < 2; ++flip) {
                        v3 cp;
                        const float d = closest_point_segment(e->a, e->b, o, cp);
                        wrong += is_silhouette_edge(e->a, e->b, e->n0, e->n1, sub(o, cp), d, flip != 0) ? 1 : 0;
                    }
                }
                // and views from anywhere, which clear most of such patches
                for (int q = 0; q < 20; ++q, ++trials)
                    clears += cone_slab_clear(n.cone.axis, n.cone.half_angle, sn, cs, n.cone.radius, n.slab,
                                              mk(uni(-3, 3), uni(-3, 3), uni(-3, 3)), n.box)
                                  ? 1
                                  : 0;
            }
        }
    }
    std::printf("%ld %ld %ld %ld\n", trials, clears, wrong, std::lround(1e6 * worst));
    return 0;
}
