// Host replay of rays aimed at the shared edges and vertices of a closed mesh through the traversal
// source of the kernels (naivetrace_amd/csrc/trace.hpp, built for the host with the same
// multiply-add contraction as the device code): every ray must hit, as a closest-hit and as an any-hit
// query of the packed tree and in a brute-force loop over the triangles, and the closest hit's distance
// is the loop's.
// Usage: watertight_check <file>; the file holds int32 nv, nt, nr, then float32 vertices (3 nv),
// int32 triangles (3 nt), float32 origins (3 nr) and directions (3 nr).  Prints the miss counts.
#include "check_scene.hpp"
#include <cstdio>
#include <fstream>
using namespace check;

int main(int argc, char **argv) {
  if (argc < 2) return 2;
  std::ifstream in(argv[1], std::ios::binary);
  int nv, nt, nr;
  in.read((char *)&nv, 4);
  in.read((char *)&nt, 4);
  in.read((char *)&nr, 4);
  std::vector<float> v(nv * 3), org(nr * 3), d(nr * 3);
  std::vector<int> f(nt * 3);
  in.read((char *)v.data(), nv * 12);
  in.read((char *)f.data(), nt * 12);
  in.read((char *)org.data(), nr * 12);
  in.read((char *)d.data(), nr * 12);
  if (!in) return 2;
  std::vector<Prim> prims(nt);
  for (int i = 0; i < nt; ++i)
    for (int c = 0; c < 3; ++c) prims[i].v[c] = mk(v[3 * f[3 * i + c]], v[3 * f[3 * i + c] + 1], v[3 * f[3 * i + c] + 2]);
  const Tree tree = build(prims);
  std::vector<int> stack(kLdsStack * kTraceBlock);
  int miss = 0, any_miss = 0, brute_miss = 0, diff = 0;
  for (int r = 0; r < nr; ++r) {
    Ray ray;
    ray.org = mk(org[3 * r], org[3 * r + 1], org[3 * r + 2]);
    ray.dir = mk(d[3 * r], d[3 * r + 1], d[3 * r + 2]);
    ray.tmax = 1e30f;
    HitRec h, a;
    traverse<false>(tree.nodes(), tree.per_axis.data(), nt, ray, stack.data(), h);
    const bool any = traverse<true>(tree.nodes(), tree.per_axis.data(), nt, ray, stack.data(), a);
    float best;
    const int bi = brute_force(tree, ray, best);
    miss += h.prim < 0;
    any_miss += !any;
    brute_miss += bi < 0;
    diff += h.prim >= 0 && h.t != best;
  }
  printf("rays %d packed misses %d anyhit misses %d brute misses %d distance differences %d\n", nr, miss, any_miss, brute_miss, diff);
}
