// Host-side binned-SAH BVH builder (replaces Embree's BVH build,
// src/embreeaccelerator.cxx:36-84, and Scene::BuildAccelStructure,
// src/scene.cxx:116-141).  Produces the GPU layout of device_scene.hpp.
#pragma once
#include <cstdint>
#include <vector>

namespace ttgpu {

struct BuildPrim {
  float lo[3], hi[3];
};

struct BuiltBvh {
  // Node array in the device layout (BvhNode, 16 floats each).
  std::vector<float> nodes;      // 16 * num_nodes
  std::vector<uint32_t> order;   // leaf-order position -> input primitive index
  int num_nodes = 0;
  int max_depth = 0;
  float root_lo[3] = {0, 0, 0}, root_hi[3] = {0, 0, 0};
};

// SAH with 32 bins per axis, leaves of at most `max_leaf` primitives.
BuiltBvh BuildBvh(const std::vector<BuildPrim> &prims, int max_leaf = 4, int num_threads = 0);

// 4-wide BVH collapsed from a BVH2: every node takes its BVH2 node's two children and then opens the
// inner child of largest surface area until it has four.  Leaves keep the BVH2's primitive ranges (same
// leaf order).  32 words per node: rows of four (one word per child) of lo.x, hi.x, lo.y, hi.y, lo.z,
// hi.z, then the children (>= 0 inner node, < 0 leaf ~first primitive) and their leaves' primitive
// counts (0 with a leaf: empty slot, planes at infinity).
struct BuiltBvh4 {
  std::vector<float> nodes;      // 32 * num_nodes
  int num_nodes = 0;
  int max_depth = 0;             // depth of the deepest node (root = 0)
};
BuiltBvh4 CollapseToBvh4(const BuiltBvh &b2);

// The tree as the device traverses it (device layout TravNode, 16 words per node): inner children of
// a node consecutive and in its first slots, the primitives of its leaves consecutive.  Planes are
// quantized anew: each lies outside the child's box by a margin of 2^-12 of the grid step plus 4
// units in the last place of the coordinates.  The slab test evaluates plane * inv - org * inv as
// q * (step * inv) + (origin * inv - org * inv): against exact arithmetic that is off by the
// rounding of the second term, at most 2^-24 (|t| + 255 step |inv|), so by less than 2^-16 step in
// the plane beside the relative error that the decoded form has too.
struct PackedBvh {
  std::vector<uint32_t> nodes;   // 16 * num_nodes
  std::vector<uint32_t> prims;   // traversal order -> leaf-order index of BuiltBvh
  int num_nodes = 0;
};
// Throws if a node's leaves hold more than 31 primitives or an extent exceeds 255 x 2^127.
PackedBvh PackTraversal(const BuiltBvh4 &b4);

}  // namespace ttgpu
