// psx_bvh.h - host builder of BVH4 trees (see psx_bvh.cpp).
#pragma once

#include <cstdint>
#include <vector>

#include "psx_device.h"

namespace psx {

struct BuildItem {
    float lo[3];
    float hi[3];
    // an instance makes a leaf of its own and weighs as many triangles as
    // entering it costs; 0: a triangle
    uint32_t instance_weight = 0;
};

struct Bvh4 {
    std::vector<Node4> nodes;     // node 0 is the root; inner child indices are
                                  // offset by the node_base passed to the build
    std::vector<uint32_t> order;  // leaf item order -> input item index
    float lo[3] = {0, 0, 0};
    float hi[3] = {0, 0, 0};
    uint32_t depth = 0;           // number of 4-wide levels
};

// max_leaf: largest number of items per leaf (1..4); width: children per
// node (2..4; the 4-wide record keeps unused slots empty).
Bvh4 build_bvh4(const std::vector<BuildItem> &items, uint32_t node_base, uint32_t max_leaf, uint32_t width = 4u);

// The traversal form of a node array: node i becomes QNode4 i with 8-bit
// outward-rounded child bounds and child references encoded as traversal
// entries.
std::vector<QNode4> quantize_nodes(const std::vector<Node4> &nodes);

QNode4 quantize_node(const Node4 &n);

// Bounds of the triangles under `root` (leaves hold triangles only) after the
// affine map `transform` (column-major 4x4), in double precision: six support
// searches that open the nodes whose boxes reach past the best vertex so far,
// the furthest first and at most `budget` of them each; where more are left the
// bound is the box of the furthest.  Returns how many were opened.  A box of
// eight transformed corners is up to sqrt(3) times as wide for a rotated
// instance.
uint32_t transformed_bounds(const std::vector<Node4> &nodes, const std::vector<LeafTri> &tris, uint32_t root,
                            const float *transform, uint32_t budget, double lo[3], double hi[3]);

}  // namespace psx
