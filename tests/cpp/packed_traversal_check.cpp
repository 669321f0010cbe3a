// Host-side check of the surface BVH as the device traverses it (TravNode), running the traversal code
// of naivetrace_amd/csrc/trace.hpp (compiled for the host, the same source the kernels use):
//   * every packed child box, evaluated in exact (double) arithmetic, contains the child's true box
//     with room to spare, slots are inner children first, and every primitive is in one leaf;
//   * closest-hit distance and primitive and the any-hit answer equal a brute-force loop over all
//     primitives (every ray when the scene is small, every 16th otherwise) for random, axis-parallel
//     and vertex-aimed rays (a primitive may differ on an exactly equal distance: ties on shared edges);
//   * a plain descent of the tree's float planes (check_scene.hpp) is compared the same way.
// Far from the origin the slab test (plane / dir - org / dir, as in Embree's non-robust mode that the
// reference uses) cancels and loses some grazing hits; the caller decides what to require there.
// Usage: packed_traversal_check <grid> <x offset> <rays> [comb | spheres]; prints a summary; exit status
// 1 when a box or the layout is wrong or a stack overflowed.  "comb": grid x 1000 teeth of
// check::comb instead of the heightfield; "spheres": grid spheres over the heightfield.
static long g_overflows = 0;
#define TTGPU_STACK_OVERFLOW() (++g_overflows)
#include "check_scene.hpp"
#include <cstdio>
#include <cstdlib>
#include <string>
using namespace check;

int main(int argc, char **argv) {
  const int grid = argc > 1 ? atoi(argv[1]) : 100;
  const float off = argc > 2 ? (float)atof(argv[2]) : 0.f;
  const int rays = argc > 3 ? atoi(argv[3]) : 50000;
  const std::string kind = argc > 4 ? argv[4] : "";
  const bool teeth = kind == "comb";
  std::mt19937 rng(7);
  std::uniform_real_distribution<float> U(0.f, 1.f);
  std::vector<Prim> prims = teeth ? comb(grid * 1000, off, rng) : heightfield(grid, off, rng);
  const int ground = teeth ? 0 : 2 * grid * grid;
  if (kind == "spheres") add_spheres(prims, grid, grid, off, rng);
  const int n = (int)prims.size();
  float comb_end = off;
  for (const Prim &p : prims) comb_end = std::max(comb_end, p.v[0].x + 0.01f);
  const Tree tree = build(prims);
  const PackedBvh &pk = tree.packed;
  const TravNode *qn = tree.nodes();
  long bad_box = 0, bad_layout = pk.num_nodes != tree.b4.num_nodes;
  std::vector<int> seen(n, 0);
  // Walk both trees together.
  std::vector<std::pair<int, int>> todo{{0, 0}};
  while (!todo.empty()) {
    const auto [i, j] = todo.back();
    todo.pop_back();
    const float *f = &tree.b4.nodes[32 * (size_t)i];
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
  std::vector<int> stack(kLdsStack * kTraceBlock);
  long diff = 0, any_diff = 0, prim_diff = 0, full_diff = 0, short_diff = 0, checked = 0, hits = 0, sphere_hits = 0;
  int max_sp = 0;
  const int every = (n <= 2000 || teeth) ? 1 : 16;
  for (int r = 0; r < rays; ++r) {
    Ray ray;
    ray.org.x = U(rng) * grid + off;
    ray.org.y = 2 + 15 * U(rng);
    ray.org.z = U(rng) * grid;
    float3 d;
    d.x = U(rng) - 0.5f;
    d.y = U(rng) - 0.7f;
    d.z = U(rng) - 0.5f;
    if (r % 7 == 0) d = mk(1.f, 0.f, 0.f);
    if (r % 11 == 0) d = mk(0.f, -1.f, 0.f);
    if (teeth) {
      // Along the axis from before the first tooth (every fourth ray exactly on it, the others
      // up to 0.02 off, some of those tilted enough to hit a tooth further on), or backwards.
      const bool on_axis = r % 4 == 0;
      ray.org = mk(off - 1.f, on_axis ? 0.f : 0.04f * (U(rng) - 0.5f), on_axis ? 0.f : 0.04f * (U(rng) - 0.5f));
      d = mk(1.f, on_axis ? 0.f : 4e-3f * (U(rng) - 0.5f), on_axis ? 0.f : 4e-3f * (U(rng) - 0.5f));
      if (r % 3 == 1) {
        ray.org.x = comb_end + 1.f;
        d.x = -1.f;
      }
    } else if (r % 5 == 0) {  // at a vertex shared by several triangles, from above
      d = prims[(size_t)(U(rng) * ground)].v[0] - ray.org;
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
        trav_advance(t, qn, tree.per_axis.data(), stack.data(), spill);
        max_sp = std::max(max_sp, t.sp / kTraceBlock);
      }
      hq = t.hit;
    }
    const bool oq = traverse<true>(qn, tree.per_axis.data(), n, ray, stack.data(), aq);
    // The camera connections keep fewer stack entries in LDS.
    HitRec hs, as;
    traverse<false, 13>(qn, tree.per_axis.data(), n, ray, stack.data(), hs);
    const bool os = traverse<true, 13>(qn, tree.per_axis.data(), n, ray, stack.data(), as);
    short_diff += hs.prim != hq.prim || (hq.prim >= 0 && hs.t != hq.t) || os != oq;
    float best, full;
    const int bi = brute_force(tree, ray, best), fi = float_planes(tree, ray, full);
    checked++;
    hits += bi >= 0;
    sphere_hits += bi >= 0 && as_int(tree.recs[bi].b.w) != 0;
    diff += (hq.prim >= 0) != (bi >= 0) || (bi >= 0 && hq.t != best);
    full_diff += (fi >= 0) != (bi >= 0) || (bi >= 0 && full != best);
    if (bi >= 0 && hq.prim >= 0 && hq.prim != bi) {  // only on an exactly equal distance
      float th, u, v;
      prim_diff += !(intersect_prim(tree.recs[hq.prim], precompute(ray), ray, 3e38f, th, u, v) && th == best);
    }
    any_diff += oq != (bi >= 0);
  }
  printf("prims %d nodes %d depth %d box_errors %ld layout_errors %ld rays %ld hits %ld sphere_hits %ld closest_diff %ld prim_diff %ld "
         "anyhit_diff %ld full_closest_diff %ld short_stack_diff %ld max_stack %d lds_stack %d overflows %ld\n",
         n, pk.num_nodes, tree.b4.max_depth, bad_box, bad_layout, checked, hits, sphere_hits, diff, prim_diff, any_diff, full_diff, short_diff,
         max_sp, kLdsStack, g_overflows);
  return (bad_box || bad_layout || g_overflows) ? 1 : 0;
}
