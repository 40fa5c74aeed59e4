// instance_bounds_driver.cpp - the host builder's instance boxes
// (transformed_bounds in psx_bvh.cpp): they hold every transformed vertex, are
// exact while the search may open what it needs, and whatever the mesh the
// search ends within its budget.  Prints "ok".
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "psx_bvh.h"

namespace {

std::mt19937 generator(7);
float normal() { return std::normal_distribution<float>()(generator); }

struct Mesh {
    std::vector<psx::Node4> nodes;
    std::vector<psx::LeafTri> tris;
};

// a sphere (the worst case: many nodes reach equally far), a ball of
// triangles, or a flat sheet
Mesh make(int kind, int count) {
    std::vector<psx::BuildItem> items;
    std::vector<psx::LeafTri> all;
    for (int i = 0; i < count; ++i) {
        float centre[3] = {normal(), kind == 2 ? 0.0f : normal(), normal()}, p[3][3];
        const float size = kind == 0 ? 2.0f / std::sqrt(static_cast<float>(count)) : 0.05f;
        auto project = [&](float *v) {
            const float l = std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
            for (int a = 0; kind == 0 && a < 3; ++a) v[a] /= l;
        };
        project(centre);
        psx::BuildItem item;
        for (int a = 0; a < 3; ++a) {
            item.lo[a] = HUGE_VALF;
            item.hi[a] = -HUGE_VALF;
        }
        for (auto &v : p) {
            for (int a = 0; a < 3; ++a) v[a] = centre[a] + (kind == 2 && a == 1 ? 0.0f : size * normal());
            project(v);
            for (int a = 0; a < 3; ++a) {
                item.lo[a] = std::min(item.lo[a], v[a]);
                item.hi[a] = std::max(item.hi[a], v[a]);
            }
        }
        items.push_back(item);
        all.push_back(psx::LeafTri{p[0][0], p[0][1], p[0][2], 0u, p[1][0], p[1][1], p[1][2], 0u, p[2][0], p[2][1], p[2][2],
                                   0u});
    }
    psx::Bvh4 tree = psx::build_bvh4(items, 0u, 2u, 4u);
    Mesh m;
    m.nodes = tree.nodes;
    for (uint32_t i : tree.order) m.tris.push_back(all[i]);
    return m;
}

}  // namespace

int main() {
    for (int kind = 0; kind < 3; ++kind)
        for (int count : {1, 2, 7, 500, 20000}) {
            const Mesh mesh = make(kind, count);
            for (uint32_t budget : {1u, 16u, 100u, 1u << 20})
                for (int turn = 0; turn < 20; ++turn) {
                    float m[16] = {};
                    for (int i = 0; i < 15; ++i) m[i] = i % 4 == 3 ? 0.0f : normal();
                    m[15] = 1.0f;
                    double lo[3], hi[3];
                    const uint32_t opened =
                        psx::transformed_bounds(mesh.nodes, mesh.tris, 0u, m, budget, lo, hi);
                    if (opened > 6ull * budget) return 1;
                    for (int a = 0; a < 3; ++a) {
                        double least = HUGE_VAL, most = -HUGE_VAL;
                        for (const psx::LeafTri &t : mesh.tris)
                            for (const float *v : {&t.p0x, &t.p1x, &t.p2x}) {
                                const double at = static_cast<double>(m[a]) * v[0] + static_cast<double>(m[4 + a]) * v[1] +
                                                  static_cast<double>(m[8 + a]) * v[2] + m[12 + a];
                                least = std::min(least, at);
                                most = std::max(most, at);
                            }
                        // what the search may leave: 1e-4 of the extent and
                        // 4e-5 of the magnitude of the largest box under the root
                        double exact = 0.0;
                        for (int o = 0; o < 3; ++o) {
                            float low = HUGE_VALF, high = -HUGE_VALF;
                            for (const psx::LeafTri &t : mesh.tris)
                                for (const float *v : {&t.p0x, &t.p1x, &t.p2x}) {
                                    low = std::min(low, v[o]);
                                    high = std::max(high, v[o]);
                                }
                            exact += std::fabs(m[4 * o + a]) * (1.01e-4 * (high - low) +
                                                                4.1e-5 * std::max(std::fabs(low), std::fabs(high)));
                        }
                        if (lo[a] > least + 1.0e-12 * std::fabs(least) || hi[a] < most - 1.0e-12 * std::fabs(most)) return 1;
                        if (budget > 1000u && (least - lo[a] > exact || hi[a] - most > exact)) return 1;
                    }
                }
        }
    std::printf("ok\n");
    return 0;
}
