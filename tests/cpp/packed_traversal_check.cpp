// Host-side check of the packed traversal tree (TravNode), running the traversal code of
// naivetrace_amd/csrc/trace.hpp (compiled for the host, the same source the kernels use):
//   * every packed child box, evaluated in exact (double) arithmetic, contains the child's true box
//     with room to spare, slots are inner children first, and every primitive is in one leaf;
//   * closest-hit distance and primitive and the any-hit answer equal a brute-force loop over all
//     primitives for random, axis-parallel and vertex-aimed rays (a primitive may differ on an
//     exactly equal distance).
// Usage: packed_traversal_check <grid> <x offset> <rays> [comb]; prints a summary; exit status 1
// when a box or the layout is wrong or a stack overflowed.  "comb" as in bvh_quantized_check.cpp.
static long g_overflows = 0;
#define TTGPU_STACK_OVERFLOW() (++g_overflows)
#include "../../naivetrace_amd/csrc/bvh_build.hpp"
#include "../../naivetrace_amd/csrc/device_scene.hpp"
#include "../../naivetrace_amd/csrc/trace.hpp"
#include <cstdio>
#include <cmath>
#include <cstring>
#include <string>
#include <random>
#include <vector>
using namespace ttgpu;

// The traversal's three copies of the records in the packed order (copy k: triangle vertices in the
// order ((k+1) mod 3, (k+2) mod 3, k), w of the first = leaf-order index), as the library uploads them.
static std::vector<ttgpu::PrimRecord> per_axis_copies(const std::vector<ttgpu::PrimRecord> &recs, const std::vector<uint32_t> &order) {
  std::vector<ttgpu::PrimRecord> out(3 * recs.size());
  for (int k = 0; k < 3; ++k)
    for (size_t i = 0; i < recs.size(); ++i) {
      auto perm = [&](float4 v) {
        const float c[3] = {v.x, v.y, v.z};
        return make_float4(c[(k + 1) % 3], c[(k + 2) % 3], c[k], v.w);
      };
      ttgpu::PrimRecord r = recs[order[i]];
      const int index = (int)order[i];
      std::memcpy(&r.a.w, &index, 4);
      r.a = perm(r.a); r.b = perm(r.b); r.c = perm(r.c);
      out[k * recs.size() + i] = r;
    }
  return out;
}


int main(int argc, char **argv) {
  const int grid = argc > 1 ? atoi(argv[1]) : 100;
  const float off = argc > 2 ? (float)atof(argv[2]) : 0.f;
  const int rays = argc > 3 ? atoi(argv[3]) : 50000;
  const bool comb = argc > 4 && std::string(argv[4]) == "comb";
  std::mt19937 rng(7);
  std::uniform_real_distribution<float> U(0.f, 1.f);
  // A bumpy heightfield of grid x grid cells plus small random triangles floating above it.
  std::vector<float3> v0, v1, v2;
  std::vector<float> h((grid + 1) * (grid + 1));
  if (comb) {
    // Tooth k at x = off + 0.01 (g^k - 1) / (g - 1) (spacing growing geometrically, e^4 over the
    // comb, so the binned SAH splits unevenly and the tree is deep): (y, z) corners (1, -1), (1, 1),
    // (-0.8, 1), each turned by a small random angle about x; the axis (y = z = 0) passes beside
    // every tooth, inside its box.
    const int nt = grid * 1000;
    const double g = 1.0 + 4.0 / nt;
    for (int k = 0; k < nt; ++k) {
      const float a = 0.2f * (U(rng) - 0.5f), ca = cosf(a), sa = sinf(a);
      const float x = off + (float)(0.01 * (std::pow(g, (double)k) - 1.0) / (g - 1.0));
      auto yz = [&](float y, float z) { return mk(x + 0.004f * (y + 1.f), ca * y - sa * z, sa * y + ca * z); };
      v0.push_back(yz(1.f, -1.f)); v1.push_back(yz(1.f, 1.f)); v2.push_back(yz(-0.8f, 1.f));
    }
  }
  for (int i = 0; i <= grid && !comb; ++i)
    for (int j = 0; j <= grid; ++j) h[i * (grid + 1) + j] = 3.f * sinf(i * 0.13f) * cosf(j * 0.07f) + 0.3f * U(rng);
  for (int i = 0; i < grid && !comb; ++i)
    for (int j = 0; j < grid; ++j) {
      const float3 a = mk(i + off, h[i * (grid + 1) + j], j), b = mk(i + 1 + off, h[(i + 1) * (grid + 1) + j], j);
      const float3 c = mk(i + off, h[i * (grid + 1) + j + 1], j + 1), d = mk(i + 1 + off, h[(i + 1) * (grid + 1) + j + 1], j + 1);
      v0.push_back(a); v1.push_back(b); v2.push_back(c);
      v0.push_back(b); v1.push_back(d); v2.push_back(c);
    }
  for (int k = 0; k < (comb ? 0 : grid * grid / 2); ++k) {
    const float3 c = mk(U(rng) * grid + off, 4 + 10 * U(rng), U(rng) * grid);
    v0.push_back(c); v1.push_back(c + mk(U(rng), U(rng), 0)); v2.push_back(c + mk(0, U(rng), U(rng)));
  }
  const int n = (int)v0.size();
  float comb_end = off;
  for (const float3 &p : v0) comb_end = std::max(comb_end, p.x + 0.01f);
  std::vector<BuildPrim> bp(n);
  for (int i = 0; i < n; ++i)
    for (int k = 0; k < 3; ++k) {
      const float a = comp3(v0[i], k), b = comp3(v1[i], k), c = comp3(v2[i], k);
      bp[i].lo[k] = std::min(a, std::min(b, c));
      bp[i].hi[k] = std::max(a, std::max(b, c));
    }
  const BuiltBvh b2 = BuildBvh(bp, 4, 0);
  const BuiltBvh4 b4 = CollapseToBvh4(b2);
  const PackedBvh pk = PackTraversal(b4);
  const TravNode *qn = (const TravNode *)pk.nodes.data();
  long bad_box = 0, bad_layout = pk.num_nodes != b4.num_nodes;
  std::vector<int> seen(n, 0);
  // Walk both trees together.
  std::vector<std::pair<int, int>> todo{{0, 0}};
  while (!todo.empty()) {
    const auto [i, j] = todo.back();
    todo.pop_back();
    const float *f = &b4.nodes[32 * (size_t)i];
    int child[4], count[4], slot[4], num = 0, inner = 0;
    std::memcpy(child, f + 24, 16);
    std::memcpy(count, f + 28, 16);
    for (int c = 0; c < 4; ++c) if (child[c] >= 0) slot[num++] = c;
    inner = num;
    for (int c = 0; c < 4; ++c) if (child[c] < 0 && count[c] > 0) slot[num++] = c;
    const TravNode &q = qn[j];
    const uint32_t e = as_uint(q.origin.w);
    const double st[3] = {std::ldexp(1.0, (int8_t)e), std::ldexp(1.0, (int8_t)(e >> 8)), std::ldexp(1.0, (int8_t)(e >> 16))};
    const uint32_t rows[6] = {q.qxy.x, q.qxy.y, q.qxy.z, q.qxy.w, q.qlz, q.qhz};
    const double o[3] = {q.origin.x, q.origin.y, q.origin.z};
    const uint32_t leaf[4] = {q.leaf.x, q.leaf.y, q.leaf.z, q.leaf.w};
    for (int c = 0; c < 4; ++c) {
      if (c >= num) { bad_layout += leaf[c] != 0x80000000u; continue; }
      for (int k = 0; k < 3; ++k) {
        const double lo = o[k] + ((rows[2 * k] >> (8 * c)) & 255u) * st[k], hi = o[k] + ((rows[2 * k + 1] >> (8 * c)) & 255u) * st[k];
        bad_box += !(lo <= f[4 * (2 * k) + slot[c]] - st[k] * 0x1p-13) || !(hi >= f[4 * (2 * k + 1) + slot[c]] + st[k] * 0x1p-13);
      }
      if (c < inner) {
        bad_layout += leaf[c] != 0u;
        todo.push_back({child[slot[c]], q.child_base + c});
      } else {
        bad_layout += !(leaf[c] >> 31) || __builtin_popcount(leaf[c] & 0x7fffffffu) != count[slot[c]];
        for (int b = 0; b < 31; ++b)
          if ((leaf[c] >> b) & 1u) {
            const int p = (int)pk.prims[q.prim_base + b];
            bad_layout += p < ~child[slot[c]] || p >= ~child[slot[c]] + count[slot[c]];
            seen[p]++;
          }
      }
    }
  }
  for (int k = 0; k < n; ++k) bad_layout += seen[k] != 1;
  std::vector<PrimRecord> recs(n);
  for (int k = 0; k < n; ++k) {
    const int p = (int)b2.order[k];
    recs[k].a = make_float4(v0[p].x, v0[p].y, v0[p].z, 0.f);
    recs[k].b = make_float4(v1[p].x, v1[p].y, v1[p].z, 0.f);
    recs[k].c = make_float4(v2[p].x, v2[p].y, v2[p].z, 0.f);
  }
  const std::vector<PrimRecord> kzrecs = per_axis_copies(recs, pk.prims);
  std::vector<int> stack(kLdsStack * kTraceBlock);
  long diff = 0, any_diff = 0, prim_diff = 0, checked = 0, hits = 0;
  int max_sp = 0;
  const int every = (n <= 2000 || comb) ? 1 : 16;
  for (int r = 0; r < rays; ++r) {
    Ray ray;
    ray.org = mk(U(rng) * grid + off, 2 + 15 * U(rng), U(rng) * grid);
    float3 d = mk(U(rng) - 0.5f, U(rng) - 0.7f, U(rng) - 0.5f);
    if (r % 7 == 0) d = mk(1.f, 0.f, 0.f);
    if (r % 11 == 0) d = mk(0.f, -1.f, 0.f);
    if (comb) {
      // Along the axis from before the first tooth (every fourth ray exactly on it, the others
      // up to 0.02 off, some of those tilted enough to hit a tooth further on), or backwards.
      const bool on_axis = r % 4 == 0;
      ray.org = mk(off - 1.f, on_axis ? 0.f : 0.04f * (U(rng) - 0.5f), on_axis ? 0.f : 0.04f * (U(rng) - 0.5f));
      d = mk(1.f, on_axis ? 0.f : 4e-3f * (U(rng) - 0.5f), on_axis ? 0.f : 4e-3f * (U(rng) - 0.5f));
      if (r % 3 == 1) {
        ray.org.x = comb_end + 1.f;
        d.x = -1.f;
      }
    }
    if (!comb && r % 5 == 0) {  // at a vertex shared by several triangles, from above
      const float3 v = v0[(size_t)(U(rng) * 2 * grid * grid)];
      d = v - ray.org;
    }
    ray.dir = normalize(d);
    ray.tmax = 3e38f;
    if (r % every) continue;
    HitRec hq, aq;
    {
      // The closest hit, step by step, to record the deepest stack.
      int spill[kSpillStack];
      Trav t;
      trav_init(t, ray, n, false, stack.data());
      while (t.active()) {
        trav_advance(t, qn, kzrecs.data(), stack.data(), spill);
        max_sp = std::max(max_sp, t.sp / kTraceBlock);
      }
      hq = t.hit;
    }
    const bool oq = traverse<true>(qn, kzrecs.data(), n, ray, stack.data(), aq);
    const RayPre pp = precompute(ray);
    float best = 3e38f;
    int bi = -1;
    for (int k = 0; k < n; ++k) {
      float th, u, v;
      if (intersect_prim(recs[k], pp, ray, best, th, u, v)) { best = th; bi = k; }
    }
    checked++;
    hits += bi >= 0;
    diff += (hq.prim >= 0) != (bi >= 0) || (bi >= 0 && hq.t != best);
    if (bi >= 0 && hq.prim >= 0 && hq.prim != bi) {  // only on an exactly equal distance
      float th, u, v;
      prim_diff += !(intersect_prim(recs[hq.prim], pp, ray, 3e38f, th, u, v) && th == best);
    }
    any_diff += oq != (bi >= 0);
  }
  printf("prims %d nodes %d depth %d box_errors %ld layout_errors %ld rays %ld hits %ld closest_diff %ld prim_diff %ld anyhit_diff %ld "
         "max_stack %d lds_stack %d overflows %ld\n",
         n, b4.num_nodes, b4.max_depth, bad_box, bad_layout, checked, hits, diff, prim_diff, any_diff, max_sp, kLdsStack, g_overflows);
  return (bad_box || bad_layout || g_overflows) ? 1 : 0;
}
