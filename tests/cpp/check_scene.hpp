// Scenes and records of the host checks of the surface BVH (packed_traversal_check.cpp,
// watertight_check.cpp): the traversal tree and the per-axis record copies as the library uploads them.
#pragma once
#include "../../naivetrace_amd/csrc/bvh_build.hpp"
#include "../../naivetrace_amd/csrc/device_scene.hpp"
#include "../../naivetrace_amd/csrc/trace.hpp"
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

namespace check {
using namespace ttgpu;

struct Prim {
  float3 v[3];      // triangle, or v[0] = centre
  float radius = 0.f;  // > 0: sphere
};

inline BuildPrim bounds(const Prim &p) {
  BuildPrim b;
  for (int k = 0; k < 3; ++k) {
    const float x = comp3(p.v[0], k), y = comp3(p.v[1], k), z = comp3(p.v[2], k);
    b.lo[k] = p.radius > 0.f ? x - p.radius : std::min(x, std::min(y, z));
    b.hi[k] = p.radius > 0.f ? x + p.radius : std::max(x, std::max(y, z));
  }
  return b;
}

// A bumpy heightfield of grid x grid cells, plus small random triangles floating above it.
inline std::vector<Prim> heightfield(int grid, float off, std::mt19937 &rng) {
  std::uniform_real_distribution<float> U(0.f, 1.f);
  std::vector<Prim> out;
  std::vector<float> h((grid + 1) * (grid + 1));
  for (int i = 0; i <= grid; ++i)
    for (int j = 0; j <= grid; ++j) h[i * (grid + 1) + j] = 3.f * sinf(i * 0.13f) * cosf(j * 0.07f) + 0.3f * U(rng);
  for (int i = 0; i < grid; ++i)
    for (int j = 0; j < grid; ++j) {
      auto at = [&](int a, int b) { return mk(i + a + off, h[(i + a) * (grid + 1) + j + b], j + b); };
      out.push_back({{at(0, 0), at(1, 0), at(0, 1)}});
      out.push_back({{at(1, 0), at(1, 1), at(0, 1)}});
    }
  for (int k = 0; k < grid * grid / 2; ++k) {
    const float x = U(rng) * grid + off, y = 4 + 10 * U(rng), z = U(rng) * grid;
    const float3 c = mk(x, y, z);
    const float a = U(rng), b = U(rng), d = U(rng), e = U(rng);
    out.push_back({{c, c + mk(a, b, 0), c + mk(0, d, e)}});
  }
  return out;
}

// Spheres of 0.02 to 2 units above the heightfield, some of them overlapping.
inline void add_spheres(std::vector<Prim> &out, int count, int grid, float off, std::mt19937 &rng) {
  std::uniform_real_distribution<float> U(0.f, 1.f);
  for (int k = 0; k < count; ++k) {
    const float x = U(rng) * grid + off, y = 12.f * U(rng), z = U(rng) * grid;
    out.push_back({{mk(x, y, z), mk(0, 0, 0), mk(0, 0, 0)}, 0.02f * std::pow(100.f, U(rng))});
  }
}

// Thin triangles stacked along the x axis whose boxes all contain the axis while the triangles leave it
// free, so that rays along (and near) the axis visit every node -- the deepest stacks a tree of this size
// can need, beyond the LDS part of the traversal stack into its private spill area.  Tooth k at
// x = off + 0.01 (g^k - 1) / (g - 1) (spacing growing geometrically, e^4 over the comb, so the binned
// SAH splits unevenly and the tree is deep): (y, z) corners (1, -1), (1, 1), (-0.8, 1), each turned by
// a small random angle about x.
inline std::vector<Prim> comb(int teeth, float off, std::mt19937 &rng) {
  std::uniform_real_distribution<float> U(0.f, 1.f);
  std::vector<Prim> out;
  const double g = 1.0 + 4.0 / teeth;
  for (int k = 0; k < teeth; ++k) {
    const float a = 0.2f * (U(rng) - 0.5f), ca = cosf(a), sa = sinf(a);
    const float x = off + (float)(0.01 * (std::pow(g, (double)k) - 1.0) / (g - 1.0));
    auto yz = [&](float y, float z) { return mk(x + 0.004f * (y + 1.f), ca * y - sa * z, sa * y + ca * z); };
    out.push_back({{yz(1.f, -1.f), yz(1.f, 1.f), yz(-0.8f, 1.f)}});
  }
  return out;
}

struct Tree {
  BuiltBvh b2;
  BuiltBvh4 b4;
  PackedBvh packed;
  std::vector<PrimRecord> recs;  // leaf order
  // Three copies in the packed order (copy k: triangle vertices in the order ((k+1) mod 3, (k+2) mod 3, k),
  // w of the first = leaf-order index).
  std::vector<PrimRecord> per_axis;
  const TravNode *nodes() const { return (const TravNode *)packed.nodes.data(); }
  int size() const { return (int)recs.size(); }
};

inline Tree build(const std::vector<Prim> &prims) {
  Tree t;
  std::vector<BuildPrim> bp;
  for (const Prim &p : prims) bp.push_back(bounds(p));
  t.b2 = BuildBvh(bp, 4, 0);
  t.b4 = CollapseToBvh4(t.b2);
  t.packed = PackTraversal(t.b4);
  const int n = (int)prims.size();
  t.recs.resize(n);
  for (int k = 0; k < n; ++k) {
    const Prim &p = prims[t.b2.order[k]];
    const int kind = p.radius > 0.f;
    auto row = [](float3 v) { return make_float4(v.x, v.y, v.z, 0.f); };
    t.recs[k].a = row(p.v[0]);
    t.recs[k].b = kind ? make_float4(p.radius, 0.f, 0.f, as_float(kind)) : row(p.v[1]);
    t.recs[k].c = kind ? make_float4(0.f, 0.f, 0.f, 0.f) : row(p.v[2]);
  }
  t.per_axis.resize(3 * (size_t)n);
  for (int k = 0; k < 3; ++k)
    for (int i = 0; i < n; ++i) {
      auto perm = [&](float4 v) {
        const float c[3] = {v.x, v.y, v.z};
        return make_float4(c[(k + 1) % 3], c[(k + 2) % 3], c[k], v.w);
      };
      PrimRecord r = t.recs[t.packed.prims[i]];
      const int index = (int)t.packed.prims[i];
      std::memcpy(&r.a.w, &index, 4);
      if (as_int(r.b.w) == 0) {
        r.a = perm(r.a);
        r.b = perm(r.b);
        r.c = perm(r.c);
      }
      t.per_axis[(size_t)k * n + i] = r;
    }
  return t;
}

// Nearest hit by a loop over every primitive: leaf-order index or -1.
inline int brute_force(const Tree &t, const Ray &ray, float &best) {
  const RayPre pp = precompute(ray);
  int index = -1;
  best = ray.tmax;
  for (int k = 0; k < t.size(); ++k) {
    float th, u, v;
    if (intersect_prim(t.recs[k], pp, ray, best, th, u, v)) {
      best = th;
      index = k;
    }
  }
  return index;
}

// Nearest hit by a plain descent of the tree with its float planes (the slab test of the intermediate
// precision: plane * inv - origin * inv), which loses a hit only where that test does.
inline int float_planes(const Tree &t, const Ray &ray, float &best) {
  const RayPre p = precompute(ray);
  int index = -1;
  best = ray.tmax;
  std::vector<int> stack{0};
  while (!stack.empty()) {
    const float *n = &t.b4.nodes[32 * (size_t)stack.back()];
    stack.pop_back();
    int child[4], count[4];
    std::memcpy(child, n + 24, sizeof(child));
    std::memcpy(count, n + 28, sizeof(count));
    for (int c = 0; c < 4; ++c) {
      if (child[c] < 0 && count[c] == 0) continue;
      float tn = 0.f, tf = best;
      const float inv[3] = {p.inv.x, p.inv.y, p.inv.z}, on[3] = {p.onear.x, p.onear.y, p.onear.z}, of[3] = {p.ofar.x, p.ofar.y, p.ofar.z};
      for (int k = 0; k < 3; ++k) {
        const float lo = n[4 * (2 * k) + c], hi = n[4 * (2 * k + 1) + c];
        tn = fmaxf(tn, (inv[k] < 0.f ? hi : lo) * inv[k] - on[k]);
        tf = fminf(tf, (inv[k] < 0.f ? lo : hi) * inv[k] - of[k]);
      }
      if (!(tn <= tf * 1.0000004f)) continue;
      if (child[c] >= 0) {
        stack.push_back(child[c]);
        continue;
      }
      for (int k = ~child[c]; k < ~child[c] + count[c]; ++k) {
        float th, u, v;
        if (intersect_prim(t.recs[k], p, ray, best, th, u, v)) {
          best = th;
          index = k;
        }
      }
    }
  }
  return index;
}

}  // namespace check
