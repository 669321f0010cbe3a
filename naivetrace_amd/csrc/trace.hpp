// BVH traversal on the GPU: closest hit and any hit, FP32, watertight
// ray/triangle test (Woop, Benthin & Wald 2013) and spheres.  Replaces
// rtcIntersect1 / rtcOccluded1 (src/embreeaccelerator.cxx:111,302).
//
// The traversal stack lives in LDS, one column per lane (bank-conflict free),
// with a small private overflow area for unusually deep trees.
#pragma once
#include "device_math.hpp"

// Called when a push finds the traversal stack full.  The host bounds the tree's depth so that
// this cannot happen; a translation unit that launches traversals defines it to raise a flag the
// host turns into an error (the entry is dropped, so memory accesses stay in bounds).
#ifndef TTGPU_STACK_OVERFLOW
#define TTGPU_STACK_OVERFLOW() ((void)0)
#endif

namespace ttgpu {

#ifndef TTGPU_LDS_STACK
#define TTGPU_LDS_STACK 24
#endif
constexpr int kTraceBlock = 128;                    // threads per block of the trace kernels
constexpr int kLdsStack = TTGPU_LDS_STACK;          // traversal stack entries per lane in LDS
constexpr int kSpillStack = kStackEntries - kLdsStack;  // and in a private overflow area

struct Ray {
  float3 org, dir;
  float tmax;
};

struct HitRec {
  float t, u, v;
  int prim;  // leaf-order primitive, -1 = none
};

struct RayPre {
  float3 inv;
  // org * inv, widened by its rounding error: entry distances are plane * inv - onear, exit
  // distances plane * inv - ofar (see precompute).
  float3 onear, ofar;
  bool negx, negy, negz;  // direction signs: which of a box's two planes per axis is entered first
  int kx, ky, kz;
  float Sx, Sy, Sz;
  float3 orgp;  // the origin's coordinates in the order (kx, ky, kz)
};

TT_HD float comp3(float3 v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : v.z); }

TT_HD RayPre precompute(const Ray &r) {
  RayPre p;
  const float tiny = 1e-30f;
  float dx = fabsf(r.dir.x) > tiny ? r.dir.x : copysignf(tiny, r.dir.x);
  float dy = fabsf(r.dir.y) > tiny ? r.dir.y : copysignf(tiny, r.dir.y);
  float dz = fabsf(r.dir.z) > tiny ? r.dir.z : copysignf(tiny, r.dir.z);
  p.inv = mk(1.f / dx, 1.f / dy, 1.f / dz);
  const float3 oinv = mk(r.org.x * p.inv.x, r.org.y * p.inv.y, r.org.z * p.inv.z);
  // The slab distances plane * inv - oinv carry an absolute error of up to ulp(oinv) beside their
  // relative one (covered by the far bound's 1 + 2 gamma(3) factor).  Where a ray passes through a
  // box's edge or corner -- a ray aimed at a shared vertex of a mesh -- the entry and exit
  // distances are equal, so each axis's interval is widened by 2^-23 |oinv|: entry distances
  // subtract oinv + err, exit distances oinv - err.
  const float e = 1.1920929e-7f;
  const float3 err = mk(fabsf(oinv.x) * e, fabsf(oinv.y) * e, fabsf(oinv.z) * e);
  p.onear = oinv + err;
  p.ofar = oinv - err;
  p.negx = p.inv.x < 0.f;
  p.negy = p.inv.y < 0.f;
  p.negz = p.inv.z < 0.f;
  float ax = fabsf(r.dir.x), ay = fabsf(r.dir.y), az = fabsf(r.dir.z);
  int kz = 0;
  if (ay > ax) kz = 1;
  if (az > fmaxf(ax, ay)) kz = 2;
  // Woop, Benthin & Wald swap kx and ky when the direction's kz component is negative, to keep
  // the winding; the test below is two-sided and symmetric in x and y (U, V, W and det change
  // sign exactly, t and the barycentrics do not change), so the frame stays the cyclic one.
  const int kx = kz == 2 ? 0 : kz + 1, ky = kx == 2 ? 0 : kx + 1;
  float dkz = kz == 0 ? r.dir.x : (kz == 1 ? r.dir.y : r.dir.z);
  float dkx = kx == 0 ? r.dir.x : (kx == 1 ? r.dir.y : r.dir.z);
  float dky = ky == 0 ? r.dir.x : (ky == 1 ? r.dir.y : r.dir.z);
  p.kx = kx; p.ky = ky; p.kz = kz;
  p.Sx = dkx / dkz; p.Sy = dky / dkz; p.Sz = 1.f / dkz;
  p.orgp = mk(comp3(r.org, kx), comp3(r.org, ky), comp3(r.org, kz));
  return p;
}

// Watertight test on vertices already given in the ray's (kx, ky, kz) frame, relative to the
// origin: A = v0 - org, B = v1 - org, C = v2 - org with components (kx, ky, kz).  On a hit within
// (0, tmax) writes t and barycentrics (b1, b2) of v1, v2.
TT_HD bool intersect_triangle_k(const RayPre &p, float3 A, float3 B, float3 C, float tmax, float &t, float &b1, float &b2) {
  // No fused multiply-adds in this test: the edge functions must be antisymmetric
  // (U(B,C) == -U(C,B) bit for bit) so that a ray through a shared edge or vertex is
  // accepted by at least one of the triangles that share it.  fma(Cx, By, -Cy*Bx) rounds
  // the two products differently from fma(Bx, Cy, -By*Cx) and breaks that.
#pragma clang fp contract(off)
  const float Akz = A.z, Bkz = B.z, Ckz = C.z;
  const float Ax = A.x - p.Sx * Akz, Ay = A.y - p.Sy * Akz;
  const float Bx = B.x - p.Sx * Bkz, By = B.y - p.Sy * Bkz;
  const float Cx = C.x - p.Sx * Ckz, Cy = C.y - p.Sy * Ckz;
  float U = Cx * By - Cy * Bx;
  float V = Ax * Cy - Ay * Cx;
  float W = Bx * Ay - By * Ax;
  // Comparisons through minima and maxima (exact; NaNs end at the determinant): a third of the
  // instructions of one compare per edge and sign.
  if (fminf(fminf(fabsf(U), fabsf(V)), fabsf(W)) == 0.f) {
    U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
    V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
    W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
  }
  if (fminf(fminf(U, V), W) < 0.f && fmaxf(fmaxf(U, V), W) > 0.f) return false;
  const float det = U + V + W;
  if (det == 0.f) return false;
  const float Az = p.Sz * Akz, Bz = p.Sz * Bkz, Cz = p.Sz * Ckz;
  const float T = U * Az + V * Bz + W * Cz;
  const float inv = 1.f / det;
  const float tt = T * inv;
  if (!(tt > 0.f && tt < tmax)) return false;
  // Conservative lower bound on t (PBRT-v3 Triangle::Intersect): rays leaving a surface do not
  // re-hit it at a distance below the rounding error of t.
  {
    constexpr float e = kFltEps;
    const float g2 = 2.f * e / (1.f - 2.f * e), g3 = 3.f * e / (1.f - 3.f * e), g5 = 5.f * e / (1.f - 5.f * e);
    const float maxZt = fmaxf(fabsf(Az), fmaxf(fabsf(Bz), fabsf(Cz)));
    const float maxXt = fmaxf(fabsf(Ax), fmaxf(fabsf(Bx), fabsf(Cx)));
    const float maxYt = fmaxf(fabsf(Ay), fmaxf(fabsf(By), fabsf(Cy)));
    const float deltaZ = g3 * maxZt, deltaX = g5 * (maxXt + maxZt), deltaY = g5 * (maxYt + maxZt);
    // Grouped so that exchanging x and y leaves the bound unchanged bit for bit.
    const float deltaE = 2.f * (g2 * (maxXt * maxYt) + (deltaY * maxXt + deltaX * maxYt));
    const float maxE = fmaxf(fabsf(U), fmaxf(fabsf(V), fabsf(W)));
    const float deltaT = 3.f * (g3 * maxE * maxZt + deltaE * maxZt + deltaZ * maxE) * fabsf(inv);
    if (tt <= deltaT) return false;
  }
  t = tt;
  b1 = V * inv;
  b2 = W * inv;
  return true;
}

// The same test on world-space vertices.
TT_HD bool intersect_triangle(const RayPre &p, float3 org, float3 v0, float3 v1, float3 v2, float tmax, float &t,
                              float &b1, float &b2) {
#pragma clang fp contract(off)
  const float3 A = v0 - org, B = v1 - org, C = v2 - org;
  return intersect_triangle_k(p, mk(comp3(A, p.kx), comp3(A, p.ky), comp3(A, p.kz)),
                              mk(comp3(B, p.kx), comp3(B, p.ky), comp3(B, p.kz)),
                              mk(comp3(C, p.kx), comp3(C, p.ky), comp3(C, p.kz)), tmax, t, b1, b2);
}

// Sphere: nearest root in (eps, tmax), numerically stable form, in FP64 so that spheres of
// planetary size (thousands of scene units) keep their hit distances and inside/outside
// decisions exact to well below the self-intersection offset.  The lower bound eps is
// 1e-9 of the sphere's extent and absorbs the residual root of a ray leaving the surface.
TT_HD bool intersect_sphere(float3 org, float3 dir, float4 cr, float tmax, float &t) {
  const double ox = (double)org.x - cr.x, oy = (double)org.y - cr.y, oz = (double)org.z - cr.z;
  const double dx = dir.x, dy = dir.y, dz = dir.z, r = cr.w;
  const double a = dx * dx + dy * dy + dz * dz;
  const double b = ox * dx + oy * dy + oz * dz;
  const double s = b / a;
  const double qx = ox - dx * s, qy = oy - dy * s, qz = oz - dz * s;
  const double disc = a * (r * r - (qx * qx + qy * qy + qz * qz));
  if (disc < 0.) return false;
  const double sd = sqrt(disc);
  const double q = b > 0. ? -b - sd : -b + sd;
  const double c = ox * ox + oy * oy + oz * oz - r * r;
  double t0 = q != 0. ? c / q : 0., t1 = q / a;
  if (t0 > t1) { double x = t0; t0 = t1; t1 = x; }
  const double eps = 1e-9 * ((double)fabsf(cr.x) + fabsf(cr.y) + fabsf(cr.z) + r);
  if (t0 > eps && t0 < (double)tmax) { t = (float)t0; return true; }
  if (t1 > eps && t1 < (double)tmax) { t = (float)t1; return true; }
  return false;
}

TT_HD bool intersect_prim(const PrimRecord &pr, const RayPre &p, const Ray &r, float tmax, float &t, float &u, float &v) {
  if (as_int(pr.b.w) == 0)
    return intersect_triangle(p, r.org, xyz(pr.a), xyz(pr.b), xyz(pr.c), tmax, t, u, v);
  u = v = 0.f;
  return intersect_sphere(r.org, r.dir, make_float4(pr.a.x, pr.a.y, pr.a.z, pr.b.x), tmax, t);
}

// The same on a record of DeviceScene::prims_kz's copy p.kz (triangle vertices in the ray's frame).
TT_HD bool intersect_prim_k(const PrimRecord &pr, const RayPre &p, const Ray &r, float tmax, float &t, float &u, float &v) {
#pragma clang fp contract(off)
  if (as_int(pr.b.w) == 0)
    return intersect_triangle_k(p, xyz(pr.a) - p.orgp, xyz(pr.b) - p.orgp, xyz(pr.c) - p.orgp, tmax, t, u, v);
  u = v = 0.f;
  return intersect_sphere(r.org, r.dir, make_float4(pr.a.x, pr.a.y, pr.a.z, pr.b.x), tmax, t);
}

// Slab test of both children; returns entry distances (or +inf when missed).  Per axis the plane
// the ray enters first is the lower one for a positive direction and the upper one otherwise.
TT_HD void box2(const BvhNode &n, const RayPre &p, float tmax, float &tl, float &tr) {
  const float lxn = p.negx ? n.lxy.y : n.lxy.x, lxf = p.negx ? n.lxy.x : n.lxy.y;
  const float lyn = p.negy ? n.lxy.w : n.lxy.z, lyf = p.negy ? n.lxy.z : n.lxy.w;
  const float lzn = p.negz ? n.lrz.y : n.lrz.x, lzf = p.negz ? n.lrz.x : n.lrz.y;
  const float rxn = p.negx ? n.rxy.y : n.rxy.x, rxf = p.negx ? n.rxy.x : n.rxy.y;
  const float ryn = p.negy ? n.rxy.w : n.rxy.z, ryf = p.negy ? n.rxy.z : n.rxy.w;
  const float rzn = p.negz ? n.lrz.w : n.lrz.z, rzf = p.negz ? n.lrz.z : n.lrz.w;
  // Conservative far bound (1 + 2 gamma(3)) so grazing hits are not lost (Ize 2013).
  const float pad = 1.0000004f;
  const float lmin = fmaxf(fmaxf(lxn * p.inv.x - p.onear.x, lyn * p.inv.y - p.onear.y), fmaxf(lzn * p.inv.z - p.onear.z, 0.f));
  const float lmax = fminf(fminf(lxf * p.inv.x - p.ofar.x, lyf * p.inv.y - p.ofar.y), fminf(lzf * p.inv.z - p.ofar.z, tmax)) * pad;
  const float rmin = fmaxf(fmaxf(rxn * p.inv.x - p.onear.x, ryn * p.inv.y - p.onear.y), fmaxf(rzn * p.inv.z - p.onear.z, 0.f));
  const float rmax = fminf(fminf(rxf * p.inv.x - p.ofar.x, ryf * p.inv.y - p.ofar.y), fminf(rzf * p.inv.z - p.ofar.z, tmax)) * pad;
  tl = lmin <= lmax ? lmin : as_float(0x7f800000);
  tr = rmin <= rmax ? rmin : as_float(0x7f800000);
}

// ---- traversal of the packed nodes ------------------------------------------------------------
// Issue-bound as one ray per lane with nodes of decoded 8-bit planes (VALU work in 95-100 % of SIMD cycles,
// 5.4e8 instructions per launch of the 1080p benchmark): what counted was instructions per step times
// the steps a wave makes, which its busiest lanes set.  Now 2.9e8 instructions, VALU busy 78 % and the
// vector-memory return path 84 % (a scattered 16-byte load of 32 lanes takes 30 cycles of it, so a
// node step's four take 120 of the 173 x 4 its arithmetic takes on each of the four SIMDs).  Three
// things keep both low:
//  * the packed layout.  Child boxes take two instructions per plane (byte to float, fma onto
//    per-node constants); entry distances carry the slot in their low two bits, so sorting the four
//    is five integer min / max pairs and a child's index one addition; entered leaves are bits of
//    one mask.  A node step is 173 VALU instructions, with the decoded planes, compare-and-swap pairs
//    and leaf list of such nodes it was 233.
//  * one kind of step per iteration.  Lanes with primitives to test and lanes with a node to visit
//    do not advance together: the wave takes the kind of step that more of its lanes wait for, and
//    the others wait (their fetch is on its way meanwhile).  A model of 64-lane waves over the
//    benchmark scene's rays counted 146 issued instructions per ray for this, 173 for both kinds in
//    every iteration.
//  * waves take new rays as theirs end (k_trace).
// `node` is the node to visit next and `pmask` the primitives to test before.  A step loads what it
// works on when it starts: with four or five waves per SIMD the others' arithmetic covers the
// latency.  Fetching a step ahead kept 28 more registers alive across the loop, and the copies that
// merged them between the two kinds of step waited for the fetch anyway.
struct Trav {
  RayPre p;
  float3 org, dir;
  float tmax;
  HitRec hit;
  int sp;            // stack top, in entries x kTraceBlock
  int node;          // -1: none
  uint32_t pmask;
  int pbase;         // record of pmask's bit 0
  int kofs;          // p.kz x the number of primitives: this ray's copy of the records
  bool any;          // any-hit query: finished at the first hit
  TT_HD bool wants_prim() const { return pmask != 0; }
  TT_HD bool wants_node() const { return pmask == 0 && node >= 0; }
  TT_HD bool active() const { return pmask != 0 || node >= 0; }
};

TT_HD int first_bit(uint32_t m) { return __builtin_ctz(m); }
TT_HD void sort2(uint32_t &a, uint32_t &b) {
  const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
  a = lo;
  b = hi;
}

TT_HD void trav_init(Trav &t, const Ray &r, int num_prims, bool any_hit, int *stack) {
  t.any = any_hit;
  t.p = precompute(r);
  t.kofs = t.p.kz * num_prims;
  t.org = r.org;
  t.dir = r.dir;
  t.tmax = r.tmax;
  t.hit.prim = -1;
  stack[0] = -1;  // popped when the tree is exhausted
  t.sp = kTraceBlock;
  t.node = 0;
  t.pmask = 0;
  t.pbase = 0;
}

// Primitive step: tests the first primitive of the mask.
TT_HD void trav_prim(Trav &t, const PrimRecord *prims) {
  PrimRecord cur = prims[t.pbase + first_bit(t.pmask)];
  t.pmask &= t.pmask - 1u;
#if defined(__HIP_DEVICE_COMPILE__)
  // The whole record in three wide loads at once, rather than its kind first and the rest in pieces
  // behind the branch on it.
  asm volatile("" : "+v"(cur.a.x), "+v"(cur.a.y), "+v"(cur.a.z), "+v"(cur.a.w), "+v"(cur.b.x), "+v"(cur.b.y), "+v"(cur.b.z),
                    "+v"(cur.b.w), "+v"(cur.c.x), "+v"(cur.c.y), "+v"(cur.c.z), "+v"(cur.c.w));
#endif
  Ray r;
  r.org = t.org;
  r.dir = t.dir;
  float th, u, v;
  if (intersect_prim_k(cur, t.p, r, t.tmax, th, u, v)) {
    t.tmax = th;
    t.hit.t = th; t.hit.u = u; t.hit.v = v; t.hit.prim = as_int(cur.a.w);
    if (t.any) {
      t.pmask = 0;
      t.node = -1;
    }
  }
}

// Node step: slab test of the four children; inner children sorted by entry distance, the nearest
// visited next and the others pushed far to near; the mask of the entered leaves' primitives.  The first
// kLds stack entries are in LDS.
template <int kLds>
TT_HD void trav_node(Trav &t, const TravNode *nodes, int *stack, int *spill) {
  const TravNode n = nodes[t.node];
  const uint32_t e = as_uint(n.origin.w);
  const float ax = ldexpf(t.p.inv.x, (int)(int8_t)e), ay = ldexpf(t.p.inv.y, (int)(int8_t)(e >> 8)),
              az = ldexpf(t.p.inv.z, (int)(int8_t)(e >> 16));
  const float bnx = fmaf(n.origin.x, t.p.inv.x, -t.p.onear.x), bfx = fmaf(n.origin.x, t.p.inv.x, -t.p.ofar.x);
  const float bny = fmaf(n.origin.y, t.p.inv.y, -t.p.onear.y), bfy = fmaf(n.origin.y, t.p.inv.y, -t.p.ofar.y);
  const float bnz = fmaf(n.origin.z, t.p.inv.z, -t.p.onear.z), bfz = fmaf(n.origin.z, t.p.inv.z, -t.p.ofar.z);
  // Rows of the planes the ray enters and leaves by, per axis.
  const uint32_t nx = t.p.negx ? n.qxy.y : n.qxy.x, fx = t.p.negx ? n.qxy.x : n.qxy.y;
  const uint32_t ny = t.p.negy ? n.qxy.w : n.qxy.z, fy = t.p.negy ? n.qxy.z : n.qxy.w;
  const uint32_t nz = t.p.negz ? n.qhz : n.qlz, fz = t.p.negz ? n.qlz : n.qhz;
  const uint32_t leaf[4] = {n.leaf.x, n.leaf.y, n.leaf.z, n.leaf.w};
  const float pad = 1.0000004f;  // conservative far bound, 1 + 2 gamma(3) (Ize 2013)
  uint32_t key[4], mask = 0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    auto q = [c](uint32_t row) { return (float)((row >> (8 * c)) & 0xffu); };
    const float tn = fmaxf(fmaxf(fmaf(q(nx), ax, bnx), fmaf(q(ny), ay, bny)), fmaxf(fmaf(q(nz), az, bnz), 0.f));
    const float tf = fminf(fminf(fmaf(q(fx), ax, bfx), fmaf(q(fy), ay, bfy)), fminf(fmaf(q(fz), az, bfz), t.tmax)) * pad;
    const bool ok = tn <= tf;
    // Distance with the slot in its low bits; leaf and empty slots (bit 31 of their word) and
    // missed children sort behind every inner one, as negative integers.
    const uint32_t k = (as_uint(tn) & ~3u) | (uint32_t)c;
    key[c] = ok ? (k > leaf[c] ? k : leaf[c]) : 0xffffffffu;
    mask |= ok ? leaf[c] : 0u;
  }
  sort2(key[0], key[1]);
  sort2(key[2], key[3]);
  sort2(key[0], key[2]);
  sort2(key[1], key[3]);
  sort2(key[1], key[2]);
  const int base = n.child_base;
  if (t.sp + 3 * kTraceBlock <= kLds * kTraceBlock) {
    // All three writes land in the LDS part: each writes at the top and only a child moves it, so
    // an absent child's write is overwritten or left above the top.
#pragma unroll
    for (int c = 3; c >= 1; --c) {
      stack[t.sp] = base + (int)(key[c] & 3u);
      t.sp += (int)key[c] >= 0 ? kTraceBlock : 0;
    }
  } else {
#pragma unroll
    for (int c = 3; c >= 1; --c) {
      if ((int)key[c] < 0) continue;
      const int id = base + (int)(key[c] & 3u), k = t.sp / kTraceBlock;
      if (k < kLds) stack[t.sp] = id;
      else if (k < kStackEntries) spill[k - kLds] = id;
      if (k < kStackEntries) t.sp += kTraceBlock;
      else TTGPU_STACK_OVERFLOW();
    }
  }
  int next = base + (int)(key[0] & 3u);
  if ((int)key[0] < 0) {
    t.sp -= kTraceBlock;
    // An LDS read (the top's entry, or the last LDS entry when the top lies in the spill part)
    // rather than one generic load through a selected address space.
    const int top = t.sp;
    next = stack[top < (kLds - 1) * kTraceBlock ? top : (kLds - 1) * kTraceBlock];
    if (top >= kLds * kTraceBlock) next = spill[top / kTraceBlock - kLds];
  }
  t.pmask = mask & 0x7fffffffu;
  t.pbase = t.kofs + n.prim_base;
  t.node = next;
}

// One iteration of the wave: the kind of step more of its lanes wait for.
template <int kLds = kLdsStack>
TT_HD void trav_advance(Trav &t, const TravNode *nodes, const PrimRecord *prims, int *stack, int *spill) {
  const bool wp = t.wants_prim(), wn = t.wants_node();
#if defined(__HIP_DEVICE_COMPILE__)
  const bool take_node = (int)__popcll(__builtin_amdgcn_ballot_w64(wn)) >= (int)__popcll(__builtin_amdgcn_ballot_w64(wp));
#else
  const bool take_node = wn;
#endif
  if (take_node) {
    if (wn) trav_node<kLds>(t, nodes, stack, spill);
  } else {
    if (wp) trav_prim(t, prims);
  }
}

// Whole traversal of one ray (closest hit, or any hit with kAnyHit); true if something was hit.
template <bool kAnyHit, int kLds = kLdsStack>
TT_HD bool traverse(const TravNode *__restrict__ nodes, const PrimRecord *__restrict__ prims, int num_prims, const Ray &r, int *stack,
                    HitRec &hit) {
  int spill[kStackEntries - kLds];
  Trav t;
  trav_init(t, r, num_prims, kAnyHit, stack);
  while (t.active()) trav_advance<kLds>(t, nodes, prims, stack, spill);
  hit = t.hit;
  return t.hit.prim >= 0;
}

}  // namespace ttgpu
