// Host side of the C ABI (include/ttgpu.h): scene validation and flattening,
// BVH build, device upload, the pass schedule of PathTracingAlgo2::Run
// (src/renderingalgorithms_pathtracing2.cxx:269-295) and the wavefront loop.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "../../include/ttgpu.h"
#include "bvh_build.hpp"
#include "device_scene.hpp"
#include "guide_fit.hpp"
#include "guiding.hpp"
#include "idle_stages.hpp"
#include "kernels.hpp"
#include "media.hpp"
#include "scene_file.hpp"
#include "nn_host.hpp"

#include "spectral_tables.inc"

using namespace ttgpu;

namespace {

constexpr double kPiD = 3.14159265358979323846;

struct HipError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

void Check(hipError_t e, const char *what) {
  if (e != hipSuccess) throw HipError(std::string(what) + ": " + hipGetErrorString(e));
}

// A device array freed when it goes out of scope (entry points that stage their inputs).
template <class T> struct DevBuffer {
  T *p = nullptr;
  explicit DevBuffer(size_t n) { Check(hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T)), "hipMalloc"); }
  ~DevBuffer() { (void)hipFree(p); }
  DevBuffer(const DevBuffer &) = delete;
  DevBuffer &operator=(const DevBuffer &) = delete;
};

struct V3d {
  double x, y, z;
};
V3d operator-(V3d a, V3d b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
V3d operator+(V3d a, V3d b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
V3d operator*(V3d a, double s) { return {a.x * s, a.y * s, a.z * s}; }
double Dot(V3d a, V3d b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
V3d Cross(V3d a, V3d b) { return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
V3d Normalized(V3d a) { return a * (1.0 / std::sqrt(Dot(a, a))); }
float3 F3(V3d a) { return make_float3((float)a.x, (float)a.y, (float)a.z); }

struct Frame3 {
  V3d x, y, z;
};
Frame3 FrameZ(V3d n) {  // Duff et al. 2017
  double sign = std::copysign(1.0, n.z);
  const double a = -1.0 / (sign + n.z);
  const double b = n.x * n.y * a;
  return {{1.0 + sign * n.x * n.x * a, sign * b, -sign * n.x}, {b, sign + n.y * n.y * a, -n.y}, n};
}

}  // namespace

namespace {
void *ScratchOnCurrentDevice();
}

struct ttgpu_handle {
  std::string err;
  ttgpu_params params{};
  int device = 0;  // the device current at ttgpu_create; the handle's stream and buffers live there
  hipStream_t stream = nullptr;
  DeviceScene dsc{};
  PathQueues q{};
  std::vector<void *> allocs;
  double *fb = nullptr, *fb_sq = nullptr;
  void *select_temp = nullptr;  // storage of the slot-ordered queue selection
  BdptWork bdpt{};              // bdpt only
  InferSort infer_sort{};       // learned guide: sort of the inference queue by hit point
  bool infer_sorted = false;
  std::vector<uint64_t> pixel_spp;
  uint64_t total_spp = 0;    // all samples per pixel rendered (the RNG sample index base)
  uint64_t sched_total = 0;  // samples per pixel of the current schedule (capped by max spp)
  int sched_spp = 1;
  std::atomic<bool> stop{false}, interrupt{false};
  ttgpu_pass_callback cb = nullptr;
  void *cb_user = nullptr;
  ttgpu_stats stats{};
  bool timing = false;
  struct Timed {
    double ms = 0;
    int64_t launches = 0;
  };
  std::map<std::string, Timed> timers;
  std::vector<std::pair<std::string, std::pair<hipEvent_t, hipEvent_t>>> pending_events;
  std::vector<hipEvent_t> event_pool;
  size_t event_next = 0;
  // page-locked records the device writes: the progress of even and odd iterations, and the
  // counters at the end of a pass
  struct Pinned {
    PassProgress poll[2];
    PassReport report;
  } *pinned = nullptr, *pinned_dev = nullptr;
  ProgressRecords progress;
  int npix = 0;
  uint32_t capacity = 0;
  // host copies needed later
  std::vector<float> host_area;
  int num_triangles = 0;
  // guided integrator
  bool guided = false, trained = false;
  std::unique_ptr<guide::Recorder> recorder;       // vMF-tree or quadtree guide
  std::unique_ptr<nn::NeuralGuide> net;            // learned guide
  bool learned = false;
  int train_rounds = 0;
  float last_loss = 0.f;
  void *d_guide_nodes = nullptr, *d_guide_cells = nullptr;
  void *d_guide_qnodes = nullptr, *d_guide_qcells = nullptr;
  size_t guide_qnodes_cap = 0, guide_qcells_cap = 0;  // allocated element counts
  int64_t records_last_pass = 0, records_dropped = 0;
  // The recorder's per-pass fit on the device (vMF tree and quadtree): buffers that grow with the
  // records and cells, the quadtree's host-node -> slot maps of the uploaded trees, and whether
  // the passes fit on the host instead (TTGPU_GUIDE_HOST_FIT=1, for comparisons).
  struct GpuFit {
    GuideFitBuffers buf{};
    int64_t entries_cap = 0;
    int cells_cap = 0;
    int64_t slots_cap = 0, roots_cap = 0;
    void *temp = nullptr;
    size_t temp_bytes = 0;
    std::vector<int> fit_root, branch_end;
    std::vector<std::vector<int>> slot_of_node;
    int num_branches = 0;
    bool host = false;
    std::vector<void *> owned;
  } fit;

  template <class T> T *Alloc(size_t n) {
    void *p = nullptr;
    if (n == 0) n = 1;
    Check(hipMalloc(&p, n * sizeof(T)), "hipMalloc");
    allocs.push_back(p);
    return (T *)p;
  }
  template <class T> T *Upload(const T *src, size_t n) {
    T *d = Alloc<T>(n);
    if (n) Check(hipMemcpy(d, src, n * sizeof(T), hipMemcpyHostToDevice), "hipMemcpy H2D");
    return d;
  }
  hipEvent_t NextEvent() {
    if (event_next == event_pool.size()) {
      hipEvent_t e;
      Check(hipEventCreate(&e), "hipEventCreate");
      event_pool.push_back(e);
    }
    return event_pool[event_next++];
  }
  template <class F> void Timed(const char *name, F &&launch) {
    if (!timing) {
      launch();
      return;
    }
    hipEvent_t a = NextEvent(), b = NextEvent();
    Check(hipEventRecord(a, stream), "hipEventRecord");
    launch();
    Check(hipEventRecord(b, stream), "hipEventRecord");
    pending_events.push_back({name, {a, b}});
  }
  void CollectTimers() {
    if (pending_events.empty()) return;
    Check(hipStreamSynchronize(stream), "hipStreamSynchronize");
    for (auto &pe : pending_events) {
      float ms = 0.f;
      Check(hipEventElapsedTime(&ms, pe.second.first, pe.second.second), "hipEventElapsedTime");
      auto &t = timers[pe.first];
      t.ms += ms;
      t.launches += 1;
    }
    pending_events.clear();
    event_next = 0;
  }
  ~ttgpu_handle() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (auto e : event_pool) (void)hipEventDestroy(e);
    if (pinned) (void)hipHostFree(pinned);
    for (void *p : allocs) (void)hipFree(p);
    if (d_guide_nodes) (void)hipFree(d_guide_nodes);
    if (d_guide_cells) (void)hipFree(d_guide_cells);
    if (d_guide_qnodes) (void)hipFree(d_guide_qnodes);
    if (d_guide_qcells) (void)hipFree(d_guide_qcells);
    for (void *p : fit.owned) (void)hipFree(p);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

thread_local std::string g_create_error;
std::once_flag g_tables_once;
hipError_t g_tables_err = hipSuccess;

void EnsureTables() {
  std::call_once(g_tables_once, [] {
    float to_rgb[3 * 36], smits[7 * 36];
    for (int i = 0; i < 3; ++i)
      for (int b = 0; b < 36; ++b) to_rgb[i * 36 + b] = (float)ttgpu_tables::kSpecToRGB[i][b];
    for (int i = 0; i < 7; ++i)
      for (int b = 0; b < 36; ++b) smits[i * 36 + b] = (float)ttgpu_tables::kSmits[i][b];
    g_tables_err = UploadSpectralTables(to_rgb, smits);
  });
  Check(g_tables_err, "upload spectral tables");
}

void Validate(const ttgpu_scene &s, const ttgpu_params &p) {
  auto bad = [](const std::string &m) { throw std::invalid_argument(m); };
  if (p.width <= 0 || p.height <= 0) bad("width and height must be positive");
  if ((int64_t)p.width * p.height > (int64_t)1 << 31) bad("image too large");
  if (p.max_ray_depth < 2 || p.max_ray_depth > 255) bad("max_ray_depth must be in [2, 255]");
  if (p.num_wavelengths != 0 && p.num_wavelengths != 4) bad("the GPU path traces 4 wavelengths per path");
  if (p.sample_mode < 0 || p.sample_mode > 2) bad("bad sample_mode");
  if (p.algo != TTGPU_ALGO_PT2 && p.algo != TTGPU_ALGO_PTG && p.algo != TTGPU_ALGO_PT && p.algo != TTGPU_ALGO_BDPT)
    bad("unknown algorithm");
  if (p.algo == TTGPU_ALGO_BDPT) {
    if (p.max_ray_depth + 1 > kBdptMaxVertices) bad("bdpt supports max_ray_depth <= 16");
    if (s.camera.kind != TTGPU_CAMERA_PINHOLE) bad("bdpt needs the pinhole camera");
    for (int i = 0; i < s.num_area_emitters; ++i)
      if (s.area_emitters[i].kind != TTGPU_AREA_UNIFORM) bad("bdpt supports uniform area emitters only");
    for (int i = 0; i < s.num_env_lights; ++i)
      if (s.env_lights[i].kind == TTGPU_ENV_DIRECTIONAL) bad("bdpt does not support directional lights");
  }
  if (p.guide_kind < TTGPU_GUIDE_NONE || p.guide_kind > TTGPU_GUIDE_QUADTREE) bad("unknown guide kind");
  if (s.num_triangles < 0 || s.num_spheres < 0 || s.num_vertices < 0) bad("negative counts");
  if (s.num_triangles > 0 && (!s.vertices || !s.indices || !s.tri_material)) bad("triangles need vertices, indices, materials");
  if (s.num_spheres > 0 && (!s.spheres || !s.sphere_material)) bad("spheres need data and materials");
  // Traversal queues leaves as first << 3 | count in an int.
  if (s.num_triangles + s.num_spheres >= ((int64_t)1 << 28)) bad("too many primitives (at most 2^28 - 1)");
  for (int64_t i = 0; i < 3 * s.num_triangles; ++i)
    if (s.indices[i] >= (uint64_t)s.num_vertices) bad("triangle vertex index out of range");
  auto check_mat = [&](int m) {
    if (m < 0 || m >= s.num_materials) bad("primitive material out of range");
  };
  for (int64_t i = 0; i < s.num_triangles; ++i) check_mat(s.tri_material[i]);
  for (int64_t i = 0; i < s.num_spheres; ++i) check_mat(s.sphere_material[i]);
  for (int i = 0; i < s.num_materials; ++i) {
    const auto &m = s.materials[i];
    if (m.shader >= s.num_shaders || m.medium >= s.num_media || m.outer_medium >= s.num_media || m.emitter >= s.num_area_emitters)
      bad("material references out of range");
    if (m.shader < 0 && m.medium < 0 && m.outer_medium < 0) bad("material without shader and medium");
    if (m.shader < 0 && m.emitter >= 0) bad("emissive volume boundaries are not supported");
  }
  for (int i = 0; i < s.num_shaders; ++i)
    if (s.shaders[i].kind < 0 || s.shaders[i].kind > TTGPU_SHADER_DENSE_DIELECTRIC) bad("unknown shader kind");
  if (s.num_env_lights > kMaxEnvLights) bad("too many environment lights");
  for (int i = 0; i < s.num_env_lights; ++i) {
    const auto &e = s.env_lights[i];
    if (e.kind < 0 || e.kind > TTGPU_ENV_MAP) bad("unknown env light kind");
    if (e.kind == TTGPU_ENV_MAP && (e.tex_width <= 0 || e.tex_height <= 0 || !e.texture_rgb)) bad("env map needs a texture");
  }
  if (s.num_media > kMaxMedia) bad("too many media");
  if (s.num_media > 0 && !s.media) bad("media table missing");
  if (s.empty_space_medium >= s.num_media || s.empty_space_medium < -1) bad("empty_space_medium out of range");
  if (p.algo == TTGPU_ALGO_PTG || p.algo == TTGPU_ALGO_PT || p.algo == TTGPU_ALGO_BDPT) {
    bool any_medium = s.empty_space_medium >= 0;
    for (int i = 0; i < s.num_materials; ++i) any_medium |= s.materials[i].medium >= 0 || s.materials[i].outer_medium >= 0;
    if (any_medium && p.algo != TTGPU_ALGO_PTG) bad("pt and bdpt run on surface scenes (no media); scenes with media use pt2 or ptg");
  }
  for (int i = 0; i < s.num_media; ++i) {
    const auto &m = s.media[i];
    if (m.kind < TTGPU_MEDIUM_VACUUM || m.kind > TTGPU_MEDIUM_ATMOSPHERE_TABULATED) bad("unknown medium kind");
    if (m.kind == TTGPU_MEDIUM_ATMOSPHERE_TABULATED) {
      if (m.table_size < 2 || !(m.table_dh > 0.) || !m.table_sigma_t || !m.table_sigma_s_molecules || !m.table_sigma_s_aerosols ||
          !(m.planet_radius > 0.))
        bad("tabulated atmosphere needs at least two altitudes, a positive step, its three tables and a planet radius");
    }
    if (m.kind == TTGPU_MEDIUM_HOMOGENEOUS && (m.phase_kind < TTGPU_PHASE_UNIFORM || m.phase_kind > TTGPU_PHASE_RAYLEIGH))
      bad("unknown phase function kind");
    if (m.kind == TTGPU_MEDIUM_ATMOSPHERE && !(m.rayleigh_scale_height > 0. && m.mie_scale_height > 0. && m.planet_radius > 0.))
      bad("atmosphere needs positive scale heights and planet radius");
    for (int b = 0; b < kNBins; ++b)
      if (!(m.sigma_s[b] >= 0.f && m.sigma_a[b] >= 0.f)) bad("medium coefficients must be non-negative");
  }
  if (s.camera.kind != TTGPU_CAMERA_PINHOLE && s.camera.kind != TTGPU_CAMERA_FISHEYE) bad("unknown camera kind");
}

float PrimAreaF(const ttgpu_scene &s, int64_t pid) {
  if (pid < s.num_triangles) {
    const float *v = s.vertices;
    const uint32_t *ix = s.indices + 3 * pid;
    float a[3], b[3], c[3];
    for (int k = 0; k < 3; ++k) { a[k] = v[3 * ix[0] + k]; b[k] = v[3 * ix[1] + k]; c[k] = v[3 * ix[2] + k]; }
    float e1[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]}, e2[3] = {c[0] - a[0], c[1] - a[1], c[2] - a[2]};
    float n[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
    return 0.5f * std::sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
  }
  float r = s.spheres[4 * (pid - s.num_triangles) + 3];
  return (float)(r * r * 4. * kPiD);
}

void BuildGeometry(ttgpu_handle *h, const ttgpu_scene &s, const std::vector<int64_t> &ids, bool surfaces) {
  std::vector<BuildPrim> bp(ids.size());
  for (size_t k = 0; k < ids.size(); ++k) {
    int64_t pid = ids[k];
    BuildPrim &b = bp[k];
    if (pid < s.num_triangles) {
      for (int a = 0; a < 3; ++a) { b.lo[a] = 3e38f; b.hi[a] = -3e38f; }
      for (int j = 0; j < 3; ++j) {
        const float *v = s.vertices + 3 * s.indices[3 * pid + j];
        for (int a = 0; a < 3; ++a) { b.lo[a] = std::min(b.lo[a], v[a]); b.hi[a] = std::max(b.hi[a], v[a]); }
      }
    } else {
      const float *sp = s.spheres + 4 * (pid - s.num_triangles);
      for (int a = 0; a < 3; ++a) {
        b.lo[a] = std::nextafter(sp[a] - sp[3], -3e38f);
        b.hi[a] = std::nextafter(sp[a] + sp[3], 3e38f);
      }
    }
  }
  auto t0 = std::chrono::steady_clock::now();
#ifndef TTGPU_MAX_LEAF
#define TTGPU_MAX_LEAF 4
#endif
  BuiltBvh bvh = BuildBvh(bp, TTGPU_MAX_LEAF, h->params.num_threads);
  auto t1 = std::chrono::steady_clock::now();
  h->stats.bvh_build_ms += std::chrono::duration<double, std::milli>(t1 - t0).count();
  if (bvh.max_depth >= 63) throw std::runtime_error("BVH deeper than the traversal stack (63 levels)");
  const size_t n = ids.size();
  std::vector<PrimRecord> recs(std::max<size_t>(n, 1));
  std::vector<int> mats(std::max<size_t>(n, 1), 0);
  std::vector<float> areas(std::max<size_t>(n, 1), 0.f);
  std::vector<float4> normals;
  const bool smooth = surfaces && s.normals != nullptr;
  if (smooth) normals.resize(3 * std::max<size_t>(n, 1));
  for (size_t k = 0; k < n; ++k) {
    int64_t pid = ids[bvh.order[k]];
    PrimRecord r{};
    int orig = (int)pid;
    if (pid < s.num_triangles) {
      const uint32_t *ix = s.indices + 3 * pid;
      const float *v0 = s.vertices + 3 * ix[0], *v1 = s.vertices + 3 * ix[1], *v2 = s.vertices + 3 * ix[2];
      r.a = make_float4(v0[0], v0[1], v0[2], 0.f);
      r.b = make_float4(v1[0], v1[1], v1[2], 0.f);
      r.c = make_float4(v2[0], v2[1], v2[2], 0.f);
      std::memcpy(&r.a.w, &orig, 4);
      int kind = 0;
      std::memcpy(&r.b.w, &kind, 4);
      mats[k] = s.tri_material[pid];
      if (smooth)
        for (int j = 0; j < 3; ++j) {
          const float *nn = s.normals + 3 * ix[j];
          normals[3 * k + j] = make_float4(nn[0], nn[1], nn[2], 0.f);
        }
    } else {
      const float *sp = s.spheres + 4 * (pid - s.num_triangles);
      r.a = make_float4(sp[0], sp[1], sp[2], 0.f);
      r.b = make_float4(sp[3], 0.f, 0.f, 0.f);
      std::memcpy(&r.a.w, &orig, 4);
      int kind = 1;
      std::memcpy(&r.b.w, &kind, 4);
      mats[k] = s.sphere_material[pid - s.num_triangles];
      if (smooth)
        for (int j = 0; j < 3; ++j) normals[3 * k + j] = make_float4(0.f, 0.f, 1.f, 0.f);
    }
    recs[k] = r;
    areas[k] = PrimAreaF(s, pid);
  }
  if (bvh.num_nodes == 0) {
    // No primitives: one node whose two children are empty leaves, so traversal ends at once.
    bvh.nodes.assign(16, 0.f);
    int ch[4] = {~0, ~0, 0, 0};
    std::memcpy(bvh.nodes.data() + 12, ch, sizeof(ch));
    bvh.num_nodes = 1;
  }
  if (surfaces) {
    // Surfaces: the BVH2 collapsed to a 4-wide BVH for traversal.
    const BuiltBvh4 b4 = CollapseToBvh4(bvh);
    if (b4.max_depth > kMaxBvh4Depth)
      throw std::runtime_error("BVH4 deeper than the traversal stack (" + std::to_string(kMaxBvh4Depth) + " levels)");
    const PackedBvh packed = PackTraversal(b4);
    h->dsc.nodes = h->Upload((const TravNode *)packed.nodes.data(), packed.num_nodes);
    h->stats.scene_bytes += packed.nodes.size() * 4;
    h->stats.bvh_nodes = b4.num_nodes;
    h->dsc.prims = h->Upload(recs.data(), recs.size());
    {
      std::vector<PrimRecord> kz(3 * recs.size());
      for (int k = 0; k < 3; ++k) {
        const int kx = (k + 1) % 3, ky = (k + 2) % 3;
        auto perm = [&](float4 v) {
          const float c[3] = {v.x, v.y, v.z};
          return make_float4(c[kx], c[ky], c[k], v.w);
        };
        for (size_t i = 0; i < packed.prims.size(); ++i) {
          PrimRecord r = recs[packed.prims[i]];
          const int index = (int)packed.prims[i];
          std::memcpy(&r.a.w, &index, 4);
          int kind;
          std::memcpy(&kind, &r.b.w, 4);
          if (kind == 0) {
            r.a = perm(r.a);  // keeps w
            r.b = perm(r.b);
            r.c = perm(r.c);
          }
          kz[k * recs.size() + i] = r;
        }
      }
      h->dsc.prims_kz = h->Upload(kz.data(), kz.size());
      h->stats.scene_bytes += kz.size() * sizeof(PrimRecord);
    }
    h->dsc.prim_material = h->Upload(mats.data(), mats.size());
    h->dsc.prim_area = h->Upload(areas.data(), areas.size());
    h->dsc.prim_normals = smooth ? h->Upload(normals.data(), normals.size()) : nullptr;
    h->dsc.num_prims = (int)n;
    h->stats.scene_bytes += recs.size() * sizeof(PrimRecord) + mats.size() * 4 + areas.size() * 4 + normals.size() * sizeof(float4);
    // Area lights: emissive surface primitives.
    std::vector<int> lights;
    for (size_t k = 0; k < n; ++k)
      if (s.materials[mats[k]].emitter >= 0) lights.push_back((int)k);
    h->dsc.area_lights = h->Upload(lights.data(), lights.size());
    h->dsc.num_area_lights = (int)lights.size();
  } else {
    h->dsc.vol_nodes = h->Upload((const BvhNode *)bvh.nodes.data(), bvh.num_nodes);
    h->dsc.vol_prims = h->Upload(recs.data(), recs.size());
    h->dsc.vol_material = h->Upload(mats.data(), mats.size());
    h->dsc.num_vol_prims = (int)n;
  }
}

// MediumTracker::initializePosition (src/rendering_util.cxx:13-37) at the camera, on the host in
// FP64: a probe ray from outside the scene along -x to the camera position, crossing every
// volume boundary and then every surface in order.  Returns the packed tracker
// (current medium in bits 0-7, four slots in bits 32-63).
struct HostTracker {
  int cur;
  int slots[4];
};
void HostGoingThrough(const ttgpu_scene &s, HostTracker &t, V3d dir, V3d n, int material, int empty) {
  const auto &mat = s.materials[material];
  if (mat.medium < 0 && mat.outer_medium < 0) return;
  auto prio = [&](int m) { return m == kVacuum ? -1 : s.media[m].priority; };
  int to_enter = mat.medium, to_exit = mat.outer_medium;
  float d = (float)dir.x * (float)n.x + (float)dir.y * (float)n.y + (float)dir.z * (float)n.z;
  if (d > 0.f) std::swap(to_enter, to_exit);
  if (to_exit >= 0) {
    for (int &sl : t.slots)
      if (sl == to_exit) { sl = kEmptySlot; break; }
    if (to_exit == t.cur) {
      int best = empty;
      for (int sl : t.slots)
        if (sl != kEmptySlot && prio(best) < prio(sl)) best = sl;
      t.cur = best;
    }
  }
  if (to_enter >= 0) {
    bool inserted = false;
    for (int &sl : t.slots)
      if (sl == kEmptySlot) { sl = to_enter; inserted = true; break; }
    if (inserted && prio(to_enter) > prio(t.cur)) t.cur = to_enter;
  }
}
uint64_t PackTracker(const HostTracker &t) {
  uint64_t v = (uint64_t)(uint32_t)t.cur;
  for (int k = 0; k < 4; ++k) v |= (uint64_t)(uint32_t)t.slots[k] << (32 + 8 * k);
  return v;
}
// MediumTracker::initializePosition (rendering_util.cxx:13-37) at `pos`: a probe ray from outside the
// scene box along -x to pos goes through every volume boundary, then every surface, on its way.
uint64_t TrackerAt(const ttgpu_scene &s, int empty, V3d pos) {
  HostTracker t{empty, {kEmptySlot, kEmptySlot, kEmptySlot, kEmptySlot}};
  const int64_t nprim = s.num_triangles + s.num_spheres;
  if (nprim == 0) return PackTracker(t);
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  auto grow = [&](const double p[3], double r) {
    for (int a = 0; a < 3; ++a) { lo[a] = std::min(lo[a], p[a] - r); hi[a] = std::max(hi[a], p[a] + r); }
  };
  for (int64_t p = 0; p < s.num_triangles; ++p)
    for (int j = 0; j < 3; ++j) {
      const float *v = s.vertices + 3 * s.indices[3 * p + j];
      double q[3] = {v[0], v[1], v[2]};
      grow(q, 0.);
    }
  for (int64_t p = 0; p < s.num_spheres; ++p) {
    const float *sp = s.spheres + 4 * p;
    double q[3] = {sp[0], sp[1], sp[2]};
    grow(q, sp[3]);
  }
  const double pc[3] = {pos.x, pos.y, pos.z};
  for (int a = 0; a < 3; ++a)
    if (pc[a] < lo[a] || pc[a] > hi[a]) return PackTracker(t);
  const double dist = 2. * std::max({hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2]});
  const V3d org = pos + V3d{dist, 0., 0.}, dir{-1., 0., 0.};
  struct BHit { double t; int material; V3d n; };
  for (int pass = 0; pass < 2; ++pass) {  // volume boundaries first, then surfaces
    std::vector<BHit> hits;
    auto add = [&](double tt, int material, V3d n) {
      if (!(tt > 0. && tt < dist)) return;
      for (const auto &b : hits)
        if (b.t == tt && b.material == material) return;
      hits.push_back({tt, material, n});
    };
    for (int64_t p = 0; p < nprim; ++p) {
      const int m = p < s.num_triangles ? s.tri_material[p] : s.sphere_material[p - s.num_triangles];
      const bool surface = s.materials[m].shader >= 0;
      if (surface != (pass == 1)) continue;
      if (p < s.num_triangles) {
        const uint32_t *ix = s.indices + 3 * p;
        V3d A{s.vertices[3 * ix[0]], s.vertices[3 * ix[0] + 1], s.vertices[3 * ix[0] + 2]};
        V3d B{s.vertices[3 * ix[1]], s.vertices[3 * ix[1] + 1], s.vertices[3 * ix[1] + 2]};
        V3d C{s.vertices[3 * ix[2]], s.vertices[3 * ix[2] + 1], s.vertices[3 * ix[2] + 2]};
        const V3d e1 = B - A, e2 = C - A, pv = Cross(dir, e2);
        const double det = Dot(e1, pv);
        if (det == 0.) continue;
        const double inv = 1. / det;
        const V3d tv = org - A;
        const double u = Dot(tv, pv) * inv;
        if (u < 0. || u > 1.) continue;
        const V3d qv = Cross(tv, e1);
        const double v = Dot(dir, qv) * inv;
        if (v < 0. || u + v > 1.) continue;
        add(Dot(e2, qv) * inv, m, Normalized(Cross(e1, e2)));
      } else {
        const float *sp = s.spheres + 4 * (p - s.num_triangles);
        const V3d c{sp[0], sp[1], sp[2]};
        const V3d oc = org - c;
        const double b = Dot(oc, dir), cc = Dot(oc, oc) - (double)sp[3] * sp[3];
        const double disc = b * b - cc;
        if (disc < 0.) continue;
        const double sd = std::sqrt(disc);
        for (double tt : {-b - sd, -b + sd}) add(tt, m, Normalized(org + dir * tt - c));
      }
    }
    std::stable_sort(hits.begin(), hits.end(), [](const BHit &a, const BHit &b) { return a.t < b.t; });
    for (const auto &b : hits) HostGoingThrough(s, t, dir, b.n, b.material, empty);
  }
  return PackTracker(t);
}

uint64_t CameraTracker(const ttgpu_scene &s, int empty) {
  return TrackerAt(s, empty, V3d{s.camera.pos[0], s.camera.pos[1], s.camera.pos[2]});
}

// Alias table of a discrete distribution p[0..n) (sums to 1), Vose's construction in FP64: entry
// b keeps bucket b with probability thr_b and otherwise yields alias_b, so that every index i is
// drawn with probability p_i.  Entries store {thr, alias (int bits), p_b, p_alias}.
void BuildAlias(const double *p, int n, float4 *out) {
  std::vector<double> scaled(n);
  std::vector<int> small, large, alias(n);
  std::vector<double> thr(n, 1.0);
  for (int i = 0; i < n; ++i) {
    alias[i] = i;
    scaled[i] = p[i] * n;
    (scaled[i] < 1.0 ? small : large).push_back(i);
  }
  while (!small.empty() && !large.empty()) {
    const int s = small.back(), l = large.back();
    small.pop_back();
    thr[s] = scaled[s];
    alias[s] = l;
    scaled[l] = (scaled[l] + scaled[s]) - 1.0;
    if (scaled[l] < 1.0) {
      large.pop_back();
      small.push_back(l);
    }
  }
  // Leftovers carry rounding only: they keep themselves.
  for (int i : small) thr[i] = 1.0;
  for (int i : large) thr[i] = 1.0;
  for (int i = 0; i < n; ++i) {
    int32_t a = alias[i];
    float af;
    std::memcpy(&af, &a, 4);
    out[i] = make_float4((float)thr[i], af, (float)p[i], (float)p[alias[i]]);
  }
}

void BuildTables(ttgpu_handle *h, const ttgpu_scene &s, double bb_diag) {
  std::vector<DevShader> shaders(std::max(1, s.num_shaders));
  for (int i = 0; i < s.num_shaders; ++i) {
    const auto &a = s.shaders[i];
    DevShader &d = shaders[i];
    d.kind = a.kind; d.alpha = a.alpha; d.alpha_min = a.alpha_min; d.ior_ratio = a.ior_ratio;
    d.ior_lambda_coeff = a.ior_lambda_coeff; d.specular = a.specular;
    std::memcpy(d.reflectance, a.reflectance, sizeof(d.reflectance));
  }
  h->dsc.shaders = h->Upload(shaders.data(), shaders.size());
  std::vector<DevMaterial> mats(std::max(1, s.num_materials));
  for (int i = 0; i < s.num_materials; ++i)
    mats[i] = {s.materials[i].shader, s.materials[i].medium, s.materials[i].outer_medium, s.materials[i].emitter};
  h->dsc.materials = h->Upload(mats.data(), mats.size());
  std::vector<DevEmitter> ems(std::max(1, s.num_area_emitters));
  for (int i = 0; i < s.num_area_emitters; ++i) {
    ems[i].kind = s.area_emitters[i].kind;
    // UniformAreaLight: spectrum / (2 pi) is the exitant radiance (src/light.hxx:77-80).
    for (int b = 0; b < kNBins; ++b) ems[i].radiance[b] = (float)(s.area_emitters[i].spectrum[b] / (2. * kPiD));
  }
  h->dsc.emitters = h->Upload(ems.data(), ems.size());
  std::vector<DevPointLight> pts(std::max(1, s.num_point_lights));
  for (int i = 0; i < s.num_point_lights; ++i) {
    const auto &p = s.point_lights[i];
    pts[i].pos = make_float3((float)p.pos[0], (float)p.pos[1], (float)p.pos[2]);
    for (int b = 0; b < kNBins; ++b) pts[i].intensity[b] = (float)(p.spectrum[b] / (4. * kPiD));
  }
  h->dsc.points = h->Upload(pts.data(), pts.size());
  h->dsc.num_points = s.num_point_lights;
  // Environment lights.
  std::vector<DevEnvLight> envs(std::max(1, s.num_env_lights));
  for (int i = 0; i < s.num_env_lights; ++i) {
    const auto &e = s.env_lights[i];
    DevEnvLight &d = envs[i];
    std::memset(&d, 0, sizeof(d));
    d.kind = e.kind;
    V3d dir = Normalized({e.dir[0], e.dir[1], e.dir[2]});
    if (e.kind == TTGPU_ENV_SUN) {
      // Sun(total_power, -direction, opening angle) (src/parse_yaml_scene.cxx:555-562, light.hxx:254-263)
      double cos_open = std::cos(kPiD / 180. * e.opening_angle_deg);
      double pdf = 1. / (2. * kPiD * (1. - cos_open));
      Frame3 f = FrameZ(dir * -1.0);
      d.frame_x = F3(f.x); d.frame_y = F3(f.y); d.frame_z = F3(f.z);
      d.cos_open = (float)cos_open;
      d.pdf = (float)pdf;
      for (int b = 0; b < kNBins; ++b) d.spectrum[b] = (float)(ttgpu_tables::kSunSpectrum[b] * e.total_power * pdf);
    } else if (e.kind == TTGPU_ENV_DOME) {
      Frame3 f = FrameZ(dir * -1.0);
      d.frame_x = F3(f.x); d.frame_y = F3(f.y); d.frame_z = F3(f.z);
      d.dir = F3(dir);
      std::memcpy(d.spectrum, e.spectrum, sizeof(d.spectrum));
    } else if (e.kind == TTGPU_ENV_DIRECTIONAL) {
      d.dir = F3(dir * -1.0);  // direction the light travels
      std::memcpy(d.spectrum, e.spectrum, sizeof(d.spectrum));
    } else {
      Frame3 f = FrameZ(dir);
      d.frame_x = F3(f.x); d.frame_y = F3(f.y); d.frame_z = F3(f.z);
      const int w = e.tex_width, hh = e.tex_height;
      d.tex_w = w; d.tex_h = hh;
      // Row and per-row column probabilities weighted by sin(theta) (the CMFs of
      // src/light.cxx:88-116), sampled through alias tables.
      std::vector<double> prow(hh), pcol((size_t)w * hh);
      double total = 0.;
      for (int y = 0; y < hh; ++y) {
        double row = 0.;
        const double theta = kPiD * (((double)(hh - 1 - y) + 0.5) / hh);
        for (int x = 0; x < w; ++x) {
          const float *px = e.texture_rgb + 3 * ((size_t)y * w + x);
          const double v = std::sin(theta) * ((double)px[0] + px[1] + px[2]) / 3.;
          pcol[(size_t)y * w + x] = v;
          row += v;
        }
        for (int x = 0; x < w; ++x) pcol[(size_t)y * w + x] = row > 0 ? pcol[(size_t)y * w + x] / row : 1. / w;
        prow[y] = row;
        total += row;
      }
      for (int y = 0; y < hh; ++y) prow[y] = total > 0. ? prow[y] / total : 1. / hh;
      std::vector<float4> texel((size_t)w * hh), arows(hh), acols((size_t)w * hh);
      for (size_t k = 0; k < texel.size(); ++k) {
        const float *px = e.texture_rgb + 3 * k;
        texel[k] = make_float4(px[0], px[1], px[2], (float)pcol[k]);
      }
      BuildAlias(prow.data(), hh, arows.data());
      for (int y = 0; y < hh; ++y) BuildAlias(pcol.data() + (size_t)y * w, w, acols.data() + (size_t)y * w);
      d.texel = h->Upload(texel.data(), texel.size());
      d.alias_rows = h->Upload(arows.data(), arows.size());
      d.alias_cols = h->Upload(acols.data(), acols.size());
      h->stats.scene_bytes += (texel.size() + arows.size() + acols.size()) * sizeof(float4);
    }
  }
  h->dsc.envs = h->Upload(envs.data(), envs.size());
  h->dsc.num_envs = s.num_env_lights;
  // Light type selection probabilities proportional to counts (src/lightpicker_trivial.cxx:35-51).
  double counts[4] = {s.num_env_lights ? 1. : 0., (double)h->dsc.num_area_lights, (double)s.num_point_lights, 0.};
  double tot = counts[0] + counts[1] + counts[2] + counts[3];
  for (int k = 0; k < 4; ++k) h->dsc.type_probs[k] = tot > 0 ? (float)(counts[k] / tot) : 0.f;
  h->dsc.area_pick_prob = h->dsc.num_area_lights ? (float)(counts[1] / tot / h->dsc.num_area_lights) : 0.f;
  h->dsc.bb_diag = (float)bb_diag;
  // Media (src/shader.cxx:1162-1316, src/atmosphere.cxx:130-200).
  std::vector<DevMedium> media(std::max(1, s.num_media));
  for (int i = 0; i < s.num_media; ++i) {
    const auto &a = s.media[i];
    DevMedium &d = media[i];
    std::memset(&d, 0, sizeof(d));
    d.kind = a.kind;
    d.priority = a.priority;
    d.phase_kind = a.phase_kind;
    d.phase_g = a.phase_g;
    if (a.kind == TTGPU_MEDIUM_HOMOGENEOUS) {
      for (int b = 0; b < kNBins; ++b) {
        d.sigma_s[b] = a.sigma_s[b];
        d.sigma_t[b] = (float)((double)a.sigma_s[b] + a.sigma_a[b]);
      }
    } else if (a.kind == TTGPU_MEDIUM_ATMOSPHERE) {
      for (int k = 0; k < 3; ++k) d.planet_center[k] = a.planet_center[k];
      d.planet_radius = a.planet_radius;
      d.rayleigh_inv_h = 1.0 / a.rayleigh_scale_height;
      d.mie_inv_h = 1.0 / a.mie_scale_height;
      d.lower_cutoff = std::max(-a.rayleigh_scale_height, -a.mie_scale_height);
      d.mie_g = a.mie_g;
      std::memcpy(d.rayleigh_sigma_s, a.rayleigh_sigma_s, sizeof(d.rayleigh_sigma_s));
      std::memcpy(d.mie_sigma_s, a.mie_sigma_s, sizeof(d.mie_sigma_s));
      std::memcpy(d.mie_sigma_a, a.mie_sigma_a, sizeof(d.mie_sigma_a));
    } else if (a.kind == TTGPU_MEDIUM_ATMOSPHERE_TABULATED) {
      // TabulatedConstituents (src/atmosphere.cxx:219-263): the majorant per altitude is the
      // largest extinction over the wavelengths, then the running maximum from the top down so
      // that the lowest point of a segment bounds the whole segment.
      for (int k = 0; k < 3; ++k) d.planet_center[k] = a.planet_center[k];
      d.planet_radius = a.planet_radius;
      d.mie_g = a.mie_g;
      const int n = a.table_size;
      std::vector<float> rows((size_t)n * 3 * kNBins), maj(n);
      for (int r = 0; r < n; ++r) {
        float mx = 0.f;
        for (int b = 0; b < kNBins; ++b) {
          rows[(size_t)r * 3 * kNBins + b] = a.table_sigma_t[(size_t)r * kNBins + b];
          rows[(size_t)r * 3 * kNBins + kNBins + b] = a.table_sigma_s_molecules[(size_t)r * kNBins + b];
          rows[(size_t)r * 3 * kNBins + 2 * kNBins + b] = a.table_sigma_s_aerosols[(size_t)r * kNBins + b];
          mx = std::max(mx, a.table_sigma_t[(size_t)r * kNBins + b]);
        }
        maj[r] = mx;
      }
      for (int r = n - 2; r >= 0; --r) maj[r] = std::max(maj[r], maj[r + 1]);
      if (maj[0] < maj[n - 1])
        throw std::invalid_argument("tabulated atmosphere: the extinction majorant at the lowest altitude is below the highest one");
      d.table_n = n;
      d.table_h0 = a.table_h0;
      d.table_inv_dh = 1.0 / a.table_dh;
      d.lower_cutoff = a.table_h0;
      d.table = h->Upload(rows.data(), rows.size());
      d.table_majorant = h->Upload(maj.data(), maj.size());
      h->stats.scene_bytes += (rows.size() + maj.size()) * 4;
    }
  }
  h->dsc.media = h->Upload(media.data(), media.size());
  h->dsc.num_media = s.num_media;
  h->dsc.empty_space_medium = s.empty_space_medium >= 0 ? s.empty_space_medium : kVacuum;
  bool any_medium = s.empty_space_medium >= 0;
  for (int i = 0; i < s.num_materials; ++i) any_medium |= s.materials[i].medium >= 0 || s.materials[i].outer_medium >= 0;
  h->dsc.has_media = any_medium ? 1 : 0;
  h->dsc.has_atmosphere = 0;
  for (int i = 0; i < s.num_media; ++i)
    if (s.media[i].kind == TTGPU_MEDIUM_ATMOSPHERE || s.media[i].kind == TTGPU_MEDIUM_ATMOSPHERE_TABULATED) h->dsc.has_atmosphere = 1;
  h->dsc.cam_tracker = CameraTracker(s, h->dsc.empty_space_medium);
  // Camera (src/camera.hxx:43-93, 165-174).
  const auto &c = s.camera;
  V3d up = Normalized({c.up[0], c.up[1], c.up[2]}), dir = Normalized({c.dir[0], c.dir[1], c.dir[2]});
  double r = Dot(dir, up);
  if (std::abs(r) <= 1.0 - 2.220446049250313e-16) up = Normalized(up - dir * r);
  V3d right = Cross(up, dir);
  DevCamera &dc = h->dsc.cam;
  dc.kind = c.kind;
  dc.pos = make_float3((float)c.pos[0], (float)c.pos[1], (float)c.pos[2]);
  dc.right = F3(right); dc.up = F3(up); dc.dir = F3(dir);
  const int W = h->params.width, H = h->params.height;
  double fov = c.fov_deg * kPiD / 180.;
  double a = std::tan(fov * 0.5), b = a * (double)H / W;
  dc.xmin = (float)-a; dc.ymin = (float)-b; dc.xper = (float)(2. * a / W); dc.yper = (float)(2. * b / H);
  dc.fish_delta = (float)(2. / std::min(W, H));
  dc.width = W; dc.height = H;
  // Surface passes trace each iteration's shadow rays in the next closest-hit launch unless
  // TTGPU_SHADOW_IN_TRACE=0.
  const char *sit = std::getenv("TTGPU_SHADOW_IN_TRACE");
  h->dsc.shadow_in_trace = (sit && sit[0] == '0') ? 0 : 1;
  // Shade kernels sort each block's paths by shader class with TTGPU_SORT_SHADE=1.  Since the
  // queues hold their slots in ascending order, shading them unsorted (coalesced path state) is
  // the faster of the two on every workload measured.
  const char *ss = std::getenv("TTGPU_SORT_SHADE");
  h->dsc.sort_shade = (ss && ss[0] == '1') ? 1 : 0;
  h->dsc.sample_mode = h->params.sample_mode;
  h->dsc.mis_mode = h->params.mis_mode;
  h->dsc.max_depth = h->params.max_ray_depth;
  h->dsc.algo_pt = h->params.algo == TTGPU_ALGO_PT ? 1 : 0;
}

void AllocateQueues(ttgpu_handle *h) {
  // bdpt keeps its own workspace instead of the wavefront's path state: of path queues it only
  // uses the counters.
  const bool bdpt = h->params.algo == TTGPU_ALGO_BDPT;
  const uint32_t N = bdpt ? 1u : h->capacity;
  PathQueues &q = h->q;
  q.capacity = (int)N;
  q.org = h->Alloc<float4>(N); q.dir = h->Alloc<float4>(N); q.hit = h->Alloc<float4>(N);
  q.thru = h->Alloc<float4>(N); q.rad = h->Alloc<float4>(N);
  q.bins = h->Alloc<uint32_t>(N); q.pixel = h->Alloc<uint32_t>(N);
  q.rng_state = h->Alloc<uint2>(N); q.rng_inc = h->Alloc<uint2>(N);
  q.flags = h->Alloc<uint32_t>(N); q.last_pdf = h->Alloc<float>(N); q.roughness = h->Alloc<float>(N);
  q.tracker = h->Alloc<uint2>(N);
  q.sh_org = h->Alloc<float4>(N); q.sh_dir = h->Alloc<float4>(N); q.sh_contrib = h->Alloc<float4>(N);
  q.queue_a = h->Alloc<uint32_t>(N); q.queue_b = h->Alloc<uint32_t>(N); q.shadow_queue = h->Alloc<uint32_t>(N);
  q.counters = h->Alloc<uint32_t>(kNumCounters);
  Check(hipMemset(q.counters, 0, kNumCounters * sizeof(uint32_t)), "hipMemset counters");
  // Slot-ordered queues (the next queue selected from per-slot alive flags, in ascending slot
  // order) unless TTGPU_SLOT_ORDER=0 (continuing paths appended per block).
  const char *so = std::getenv("TTGPU_SLOT_ORDER");
  q.alive = q.freed = nullptr;
  q.free_slots = nullptr;
  if (so && so[0] == '0') {
    q.free_slots = h->Alloc<uint32_t>(N);
  } else {
    q.alive = h->Alloc<uint8_t>(N);
    q.freed = h->Alloc<uint8_t>(N);
    Check(hipMemset(q.alive, 0, N), "hipMemset alive flags");
    Check(hipMemset(q.freed, 0, N), "hipMemset freed flags");
    h->select_temp = h->Alloc<uint8_t>(SelectTempBytes(N));
  }
  q.progress = h->Alloc<unsigned long long>(2);
  Check(hipMemset(q.progress, 0, 2 * sizeof(unsigned long long)), "hipMemset progress");
  // Coherent: the host reads the progress while the device runs.
  Check(hipHostMalloc((void **)&h->pinned, sizeof(*h->pinned), hipHostMallocMapped | hipHostMallocCoherent), "hipHostMalloc");
  Check(hipHostGetDevicePointer((void **)&h->pinned_dev, h->pinned, 0), "hipHostGetDevicePointer");
  *h->pinned = {};
  h->progress.Attach(h->pinned->poll, h->pinned_dev->poll);
  q.shadow_in = q.shadow_out = q.counters + kCountShadow;
  if (h->dsc.has_media) {
    q.wt_r = h->Alloc<float4>(N);
    q.wt_c = h->Alloc<float4>(N);
    q.sh_aux = h->Alloc<uint4>(N);
  } else {
    q.wt_r = q.wt_c = nullptr;
    q.sh_aux = nullptr;
  }
  h->stats.state_bytes = (size_t)N * (16 * 8 + 4 * 6 + 8 * 3 + 12 + (h->dsc.has_media ? 48 : 0));
  q.gv_pos_pdf = q.gv_dir_acc = q.gv_thru = q.sh_nee = q.rec_pos_w = q.rec_dir = nullptr;
  q.rec_capacity = 0;
  q.max_vertices = 0;
  if (h->guided) {
    // Per-vertex state of the guided integrator: a path scatters at most max_depth - 1 times.
    const int nvtx = std::max(1, h->params.max_ray_depth - 1);
    q.max_vertices = nvtx;
    q.gv_pos_pdf = h->Alloc<float4>((size_t)N * nvtx);
    q.gv_dir_acc = h->Alloc<float4>((size_t)N * nvtx);
    q.gv_thru = h->Alloc<float4>((size_t)N * nvtx);
    q.sh_nee = h->Alloc<float4>(N);
    q.rec_capacity = (uint32_t)std::min<uint64_t>((uint64_t)h->npix * nvtx, (uint64_t)1 << 25);
    q.rec_pos_w = h->Alloc<float4>(q.rec_capacity);
    q.rec_dir = h->Alloc<float4>(q.rec_capacity);
    h->stats.state_bytes += (size_t)N * (48 * nvtx + 16) + (size_t)q.rec_capacity * 32;
  }
  if (bdpt) {
    // Samples in flight: at every depth the memory that 2^18 samples of the deepest paths take (1.4 GB),
    // up to 2^20 (the connection list's sample field).  Each chunk ends in a drained launch of each
    // kernel and a host wait: with 2^18 samples 1024 x 1024 x 16 spp of the Cornell box took 31.1 ms
    // at depth 2, 42.9 at 3 and 91.1 at 8, with this rule 25.2, 33.1 and 85.8.  Fewer when the caller
    // asks for a smaller wavefront, down to one block of the walk per four CUs (2^13 samples), below
    // which a chunk's launches cost more than its samples.
    BdptWork &w = h->bdpt;
    w.max_nodes = h->params.max_ray_depth + 1;
    auto sample_bytes = [](int nodes) { return BdptVertexBytes(nodes) + 4 * BdptMaxPairs(nodes) + 32; };
    const size_t fit = ((size_t)sample_bytes(kBdptMaxVertices) << 18) / sample_bytes(w.max_nodes);
    w.capacity = std::max(1u << 13, std::min((uint32_t)std::min<size_t>(fit, 1u << 20), h->capacity));
    h->stats.wavefront_paths = (int32_t)w.capacity;
    w.verts = (float4 *)h->Alloc<uint8_t>(w.capacity * BdptVertexBytes(w.max_nodes));
    w.pairs = h->Alloc<uint32_t>(w.capacity * BdptMaxPairs(w.max_nodes));
    w.info = h->Alloc<uint2>(w.capacity);
    w.acc = h->Alloc<double>(3 * (size_t)w.capacity);
    w.count = h->Alloc<uint32_t>(1);
    Check(hipMemset(w.count, 0, sizeof(uint32_t)), "hipMemset bdpt count");
    h->stats.state_bytes += w.capacity * sample_bytes(w.max_nodes);
  }
  q.vt = nullptr;
  q.wtn_r = q.wtn_c = nullptr;
  if (h->guided && h->dsc.has_media) {
    q.vt = h->Alloc<double>(N);
    q.wtn_r = h->Alloc<float4>(N);
    q.wtn_c = h->Alloc<float4>(N);
    h->stats.state_bytes += (size_t)N * 40;
  }
  q.gv_nrm = q.gv_wo = q.rec_nrm = q.rec_wo = q.gmix = nullptr;
  if (h->learned) {
    const int nvtx = q.max_vertices;
    q.gv_nrm = h->Alloc<float4>((size_t)N * nvtx);
    q.gv_wo = h->Alloc<float4>((size_t)N * nvtx);
    q.rec_nrm = h->Alloc<float4>(q.rec_capacity);
    q.rec_wo = h->Alloc<float4>(q.rec_capacity);
    q.gmix = h->Alloc<float4>((size_t)N * (sizeof(nn::Mix16) / sizeof(float4)));
    h->stats.state_bytes += (size_t)N * (32 * nvtx + sizeof(nn::Mix16)) + (size_t)q.rec_capacity * 32;
    // Inference on the queue sorted by hit point unless TTGPU_INFER_SORT=0.
    const char *is = std::getenv("TTGPU_INFER_SORT");
    h->infer_sorted = !(is && is[0] == '0');
    if (h->infer_sorted) {
      h->infer_sort.capacity = N;
      h->infer_sort.keys = h->Alloc<uint32_t>(2 * (size_t)N);
      h->infer_sort.vals = h->Alloc<uint32_t>(2 * (size_t)N);
      h->infer_sort.temp_bytes = std::max<size_t>(InferSortTempBytes(N), 16);
      h->infer_sort.temp = h->Alloc<uint8_t>(h->infer_sort.temp_bytes);
    }
  }
  const size_t npix = (size_t)h->npix;
  h->fb = h->Alloc<double>(3 * npix);
  h->fb_sq = h->Alloc<double>(3 * npix);
  LaunchFill(h->fb, h->fb_sq, 3 * npix, 0.0, h->stream);
  Check(hipGetLastError(), "fill framebuffer");
  Check(hipStreamSynchronize(h->stream), "sync");
}

// Appends the branches of a quadtree (pre-order) to `out` as QuadNodes; `dev` receives each node's
// branch index (-1 for a leaf).  The returned header is what the renderer samples: a tree whose root
// weight is not positive and finite, or with a negative or non-finite weight, becomes the uniform
// distribution (root -1), as such weights do not define a density; its branches are appended all
// the same (the device fit updates their weights).
QuadCell FlattenQuad(const guide::quad::Tree &t, const std::vector<float> &w, std::vector<QuadNode> &out,
                     std::vector<int> &dev) {
  const float wr = w[t.root];
  bool ok = wr > 0.f && std::isfinite(wr);
  for (size_t i = 0; ok && i < w.size(); ++i) ok = w[i] >= 0.f && std::isfinite(w[i]);
  dev.assign(t.NumNodes(), -1);
  if (t.IsLeaf(t.root)) return {-1, 1.f};
  int k = (int)out.size();
  for (int n = 0; n < t.NumNodes(); ++n)
    if (!t.IsLeaf(n)) dev[n] = k++;
  out.resize(k);
  for (int n = 0; n < t.NumNodes(); ++n) {
    if (t.IsLeaf(n)) continue;
    float cw[4];
    int cc[4];
    for (int c = 0; c < 4; ++c) {
      const int ch = t.child[n][c];
      cw[c] = w[ch];
      cc[c] = t.IsLeaf(ch) ? -1 : dev[ch];
    }
    out[dev[n]] = QuadNode{make_float4(cw[0], cw[1], cw[2], cw[3]), make_int4(cc[0], cc[1], cc[2], cc[3])};
  }
  return ok ? QuadCell{dev[t.root], wr} : QuadCell{-1, 1.f};
}

// Uploads `n` elements into a device buffer that grows as needed.
template <class T>
void UploadGrow(void *&buf, size_t &cap, const std::vector<T> &v) {
  if (v.size() > cap || !buf) {
    if (buf) Check(hipFree(buf), "hipFree");
    buf = nullptr;
    cap = std::max<size_t>(1, v.size() + v.size() / 4);
    Check(hipMalloc(&buf, cap * sizeof(T)), "hipMalloc guide");
  }
  if (!v.empty()) Check(hipMemcpy(buf, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice), "upload guide");
}

// Bakes the recorder's kd-tree and current distributions into the device layout (GuideNode and
// GuideCell for vMF mixtures; QuadCell and QuadNode for quadtrees).
void UploadGuide(ttgpu_handle *h) {
  const guide::KdTree &t = h->recorder->tree();
  const auto &cells = h->recorder->cells();
  std::vector<GuideNode> nodes(std::max<size_t>(1, t.nodes.size()));
  for (size_t k = 0; k < t.nodes.size(); ++k) {
    const auto &n = t.nodes[k];
    nodes[k] = {(float)n.pos, n.axis, n.left, n.right};
  }
  if (h->recorder->quadtree()) {
    std::vector<QuadCell> qc(std::max<size_t>(1, cells.size()), QuadCell{-1, 1.f});
    std::vector<QuadNode> qn;
    // The fit's view of the same trees: each cell's root branch and branch range, and the slot of
    // every node (the root: slot c; child k of branch b: slot cells + 4 b + k).
    auto &F = h->fit;
    const int C = (int)cells.size();
    F.fit_root.assign(C, -1);
    F.branch_end.assign(C, 0);
    F.slot_of_node.assign(C, {});
    std::vector<int> dev;
    for (int c = 0; c < C; ++c) {
      const auto &t = cells[c].qcurrent.tree;
      qc[c] = FlattenQuad(t, cells[c].qcurrent.probs, qn, dev);
      F.fit_root[c] = dev[t.root];
      F.branch_end[c] = (int)qn.size();
      auto &sl = F.slot_of_node[c];
      sl.assign(t.NumNodes(), -1);
      sl[t.root] = c;
      for (int n = 0; n < t.NumNodes(); ++n)
        if (!t.IsLeaf(n))
          for (int k = 0; k < 4; ++k) sl[t.child[n][k]] = C + 4 * dev[n] + k;
    }
    F.num_branches = (int)qn.size();
    if (h->d_guide_nodes) Check(hipFree(h->d_guide_nodes), "hipFree");
    h->d_guide_nodes = nullptr;
    Check(hipMalloc(&h->d_guide_nodes, nodes.size() * sizeof(GuideNode)), "hipMalloc guide");
    Check(hipMemcpy(h->d_guide_nodes, nodes.data(), nodes.size() * sizeof(GuideNode), hipMemcpyHostToDevice), "upload guide");
    UploadGrow(h->d_guide_qcells, h->guide_qcells_cap, qc);
    UploadGrow(h->d_guide_qnodes, h->guide_qnodes_cap, qn);
    h->dsc.guide_nodes = (const GuideNode *)h->d_guide_nodes;
    h->dsc.guide_cells = nullptr;
    h->dsc.guide_qcells = (const QuadCell *)h->d_guide_qcells;
    h->dsc.guide_qnodes = (const QuadNode *)h->d_guide_qnodes;
    h->dsc.guide_root = t.root;
    return;
  }
  std::vector<GuideCell> dc(std::max<size_t>(1, cells.size()));
  for (size_t c = 0; c < cells.size(); ++c) {
    const guide::Vmf &m = cells[c].current;
    double acc = 0.;
    for (int k = 0; k < kGuideLobes; ++k) {
      const double kap = m.kappa[k];
      dc[c].lobe[k] = make_float4(m.mu[k][0], m.mu[k][1], m.mu[k][2], m.kappa[k]);
      dc[c].wn[k] = (float)(m.w[k] * kap / (2. * kPiD * -std::expm1(-2. * kap)));
      acc += m.w[k];
      dc[c].cdf[k] = (float)acc;
    }
    dc[c].cdf[kGuideLobes - 1] = 2.f;  // every u in [0, 1) selects a lobe
  }
  if (h->d_guide_nodes) Check(hipFree(h->d_guide_nodes), "hipFree");
  if (h->d_guide_cells) Check(hipFree(h->d_guide_cells), "hipFree");
  h->d_guide_nodes = h->d_guide_cells = nullptr;
  Check(hipMalloc(&h->d_guide_nodes, nodes.size() * sizeof(GuideNode)), "hipMalloc guide");
  Check(hipMalloc(&h->d_guide_cells, dc.size() * sizeof(GuideCell)), "hipMalloc guide");
  Check(hipMemcpy(h->d_guide_nodes, nodes.data(), nodes.size() * sizeof(GuideNode), hipMemcpyHostToDevice), "upload guide");
  Check(hipMemcpy(h->d_guide_cells, dc.data(), dc.size() * sizeof(GuideCell), hipMemcpyHostToDevice), "upload guide");
  h->dsc.guide_nodes = (const GuideNode *)h->d_guide_nodes;
  h->dsc.guide_cells = (const GuideCell *)h->d_guide_cells;
  h->dsc.guide_root = t.root;
}

// ---- the recorder's per-pass fit on the device ----------------------------------------------
// IncrementalFit's weight of a leaf (path_guiding.cxx, RadianceDistributionLearned), as the device
// refresh computes it: for a tree that is a single leaf, which the device keeps no node for.
float QuadLeafWeight(float prior, int64_t n, double mean, double m2, double root_n, double total_flux, double log_round) {
  const double rc = (double)n / root_n;
  const double err = rc * (n >= 2 ? std::sqrt(m2) / (double)(n - 1) : guide::quad::kLargeFloat);
  const double mix = 100. / (100. + (double)std::max<int64_t>(n - 2, 0));
  float p = (float)((double)prior * mix + (rc * mean + err) * (1. - mix));
  p += (float)total_flux * (float)std::sqrt(log_round / (double)(n + 1));
  return p;
}

template <class T>
T *FitBuffer(ttgpu_handle *h, T *old, size_t n) {
  if (old) {
    Check(hipFree(old), "hipFree");
    auto &o = h->fit.owned;
    o.erase(std::remove(o.begin(), o.end(), (void *)old), o.end());
  }
  void *p = nullptr;
  Check(hipMalloc(&p, std::max<size_t>(1, n) * sizeof(T)), "hipMalloc guide fit");
  h->fit.owned.push_back(p);
  return (T *)p;
}

// Uploads the recorder's cells as the device fit state (after the kd-tree and the sampling copies
// were uploaded by UploadGuide): learned mixtures and EM statistics, EM parameters, leaf
// statistics, jitter frames; for the quadtree the node statistics and priors in slot order.
void UploadFit(ttgpu_handle *h) {
  auto &F = h->fit;
  const auto &cells = h->recorder->cells();
  const int C = (int)cells.size();
  if (C > F.cells_cap) {
    F.cells_cap = C + C / 4;
    F.buf.cells = FitBuffer(h, F.buf.cells, F.cells_cap);
    F.buf.cell_begin = FitBuffer(h, F.buf.cell_begin, F.cells_cap);
    F.buf.cell_end = FitBuffer(h, F.buf.cell_end, F.cells_cap);
  }
  F.buf.num_cells = C;
  std::vector<DevFitCell> dc(C);
  for (int c = 0; c < C; ++c) {
    const guide::CellData &cd = cells[c];
    DevFitCell &d = dc[c];
    std::memset(&d, 0, sizeof(d));
    for (int k = 0; k < kFitLobes; ++k) {
      for (int a = 0; a < 3; ++a) {
        d.mu[k][a] = cd.learned.mu[k][a];
        d.pos[k][a] = cd.fit.pos[k][a];
      }
      d.kappa[k] = cd.learned.kappa[k];
      d.w[k] = cd.learned.w[k];
      d.resp[k] = cd.fit.resp[k];
    }
    d.count = cd.fit.count;
    d.weight_mean = cd.fit.weight_mean;
    d.weight_count = cd.fit.weight_count;
    // RadianceDistributionLearned::Parameters (path_guiding.cxx:62-77), as the host fit uses them.
    const double strength = std::max(1., 0.01 * (double)cd.max_num_samples);
    d.prior_strength = (float)strength;
    d.m_step_every = std::max(1, (int)strength * 10);
    d.ln = cd.leaf_stats.n;
    for (int a = 0; a < 3; ++a) {
      d.lmean[a] = cd.leaf_stats.mean[a];
      for (int b = 0; b < 3; ++b) {
        d.lc[a][b] = cd.leaf_stats.c[a][b];
        d.frame[a][b] = (float)cd.cov_frame[a][b];
      }
    }
  }
  Check(hipMemcpy(F.buf.cells, dc.data(), C * sizeof(DevFitCell), hipMemcpyHostToDevice), "upload fit cells");
  if (!h->recorder->quadtree()) return;
  const int64_t S = (int64_t)C + 4 * (int64_t)F.num_branches;
  if (S > F.slots_cap) {
    F.slots_cap = S + S / 4;
    F.buf.qslots = FitBuffer(h, F.buf.qslots, F.slots_cap);
  }
  if (C > (int)F.roots_cap) {
    F.roots_cap = C + C / 4;
    F.buf.qfit_root = FitBuffer(h, (int *)F.buf.qfit_root, F.roots_cap);
    F.buf.qbranch_end = FitBuffer(h, (int *)F.buf.qbranch_end, F.roots_cap);
  }
  std::vector<DevQuadSlot> sl(S);
  std::memset(sl.data(), 0, S * sizeof(DevQuadSlot));
  for (int c = 0; c < C; ++c) {
    const auto &st = cells[c].qlearned.stats;
    const auto &prior = cells[c].qcurrent.prior;
    const auto &map = F.slot_of_node[c];
    for (size_t n = 0; n < map.size(); ++n) {
      DevQuadSlot &x = sl[map[n]];
      x.n = (unsigned long long)st.n[n];
      x.mean = st.mean[n];
      x.m2 = st.m2[n];
      x.prior = prior[n];
    }
  }
  Check(hipMemcpy(F.buf.qslots, sl.data(), S * sizeof(DevQuadSlot), hipMemcpyHostToDevice), "upload fit slots");
  Check(hipMemcpy((void *)F.buf.qfit_root, F.fit_root.data(), C * sizeof(int), hipMemcpyHostToDevice), "upload fit roots");
  Check(hipMemcpy((void *)F.buf.qbranch_end, F.branch_end.data(), C * sizeof(int), hipMemcpyHostToDevice), "upload fit ranges");
  F.buf.qcells = (QuadCell *)h->d_guide_qcells;
  F.buf.qnodes = (QuadNode *)h->d_guide_qnodes;
}

// Reads the device fit state back into the recorder's cells (before the host adapts them).
void DownloadFit(ttgpu_handle *h) {
  auto &F = h->fit;
  auto &cells = h->recorder->mutable_cells();
  const int C = (int)cells.size();
  std::vector<DevFitCell> dc(C);
  Check(hipMemcpy(dc.data(), F.buf.cells, C * sizeof(DevFitCell), hipMemcpyDeviceToHost), "download fit cells");
  for (int c = 0; c < C; ++c) {
    guide::CellData &cd = cells[c];
    const DevFitCell &d = dc[c];
    for (int k = 0; k < kFitLobes; ++k) {
      for (int a = 0; a < 3; ++a) {
        cd.learned.mu[k][a] = d.mu[k][a];
        cd.fit.pos[k][a] = d.pos[k][a];
      }
      cd.learned.kappa[k] = d.kappa[k];
      cd.learned.w[k] = d.w[k];
      cd.fit.resp[k] = d.resp[k];
    }
    cd.fit.count = d.count;
    cd.fit.weight_mean = d.weight_mean;
    cd.fit.weight_count = d.weight_count;
    cd.leaf_stats.n = d.ln;
    for (int a = 0; a < 3; ++a) {
      cd.leaf_stats.mean[a] = d.lmean[a];
      for (int b = 0; b < 3; ++b) cd.leaf_stats.c[a][b] = d.lc[a][b];
    }
  }
  if (!h->recorder->quadtree()) return;
  const int64_t S = (int64_t)C + 4 * (int64_t)F.num_branches;
  std::vector<DevQuadSlot> sl(S);
  std::vector<QuadNode> qn(std::max(1, F.num_branches));
  Check(hipMemcpy(sl.data(), F.buf.qslots, S * sizeof(DevQuadSlot), hipMemcpyDeviceToHost), "download fit slots");
  if (F.num_branches)
    Check(hipMemcpy(qn.data(), F.buf.qnodes, F.num_branches * sizeof(QuadNode), hipMemcpyDeviceToHost), "download quadtrees");
  for (int c = 0; c < C; ++c) {
    auto &st = cells[c].qlearned.stats;
    auto &sm = cells[c].qcurrent;
    const auto &t = sm.tree;
    const auto &map = F.slot_of_node[c];
    for (size_t n = 0; n < map.size(); ++n) {
      const DevQuadSlot &x = sl[map[n]];
      st.n[n] = (int64_t)x.n;
      st.mean[n] = x.mean;
      st.m2[n] = x.m2;
    }
    // The sampled weights the device fit wrote (IncrementalFit's probabilities, propagated); a
    // cell whose root has no count kept its weights.
    if (st.n[t.root] <= 0) continue;
    if (t.IsLeaf(t.root)) {
      // A single leaf (the device keeps no node for it): IncrementalFit's weight with the root's
      // own share (1), which the next adaptation scales into its children's priors.
      sm.probs[t.root] = QuadLeafWeight(sm.prior[t.root], st.n[t.root], st.mean[t.root], st.m2[t.root], (double)st.n[t.root],
                                        st.mean[t.root], 0.);
      continue;
    }
    for (int n = 0; n < t.NumNodes(); ++n) {
      if (t.IsLeaf(n)) continue;
      const QuadNode &nd = qn[(F.slot_of_node[c][t.child[n][0]] - C) / 4];  // the branch of node n
      const float w4[4] = {nd.w.x, nd.w.y, nd.w.z, nd.w.w};
      float sum = 0.f;
      for (int k = 0; k < 4; ++k) {
        sm.probs[t.child[n][k]] = w4[k];
        sum += w4[k];
      }
      sm.probs[n] = sum;
    }
  }
}

// The fit of the pass just rendered, on the device: entries, sort by cell, per-cell fit.
void GpuFitPass(ttgpu_handle *h) {
  auto &F = h->fit;
  const uint32_t *counters = h->pinned->report.counters;  // of the pass just rendered
  const int64_t n = std::min(counters[kCountRecords], h->q.rec_capacity);
  h->records_last_pass = n;
  h->records_dropped += counters[kStatRecordsDropped];
  h->recorder->CountRound();
  if (n == 0) return;
  const int64_t items = 2 * n;
  if (items > F.entries_cap) {
    F.entries_cap = items + items / 4;
    F.buf.ent_pos_w = FitBuffer(h, F.buf.ent_pos_w, F.entries_cap);
    F.buf.ent_dir = FitBuffer(h, F.buf.ent_dir, F.entries_cap);
    F.buf.keys_in = FitBuffer(h, F.buf.keys_in, F.entries_cap);
    F.buf.keys_out = FitBuffer(h, F.buf.keys_out, F.entries_cap);
    F.buf.vals_in = FitBuffer(h, F.buf.vals_in, F.entries_cap);
    F.buf.vals_out = FitBuffer(h, F.buf.vals_out, F.entries_cap);
  }
  const size_t tb = FitSortTempBytes(items, F.buf.num_cells);
  if (tb > F.temp_bytes) {
    F.temp_bytes = tb + tb / 4;
    F.temp = FitBuffer(h, (unsigned char *)F.temp, F.temp_bytes);
  }
  F.buf.rec_pos_w = h->q.rec_pos_w;
  F.buf.rec_dir = h->q.rec_dir;
  const bool quad = h->recorder->quadtree();
  DevVmfPrior prior;
  const guide::Vmf &pv = h->recorder->prior();
  for (int k = 0; k < kFitLobes; ++k) {
    for (int a = 0; a < 3; ++a) prior.mu[k][a] = pv.mu[k][a];
    prior.kappa[k] = pv.kappa[k];
    prior.w[k] = pv.w[k];
  }
  h->Timed("guide_fit", [&] {
    LaunchFitPrepare(h->dsc, F.buf, n, quad, h->params.seed, (uint32_t)h->recorder->round(), h->stream);
    Check(LaunchFitSort(F.buf, items, F.temp, F.temp_bytes, h->stream), "sort records into cells");
    // Every fit of a pass sees round 1 (the reference's sub_round restarts at each pass), so the
    // exploration term log(round) vanishes.
    LaunchFitCells(F.buf, items, quad, prior, 0.f, h->stream);
  });
  Check(hipGetLastError(), "guide fit");
}

// Downloads the records of the pass just rendered and hands them to the recorder.
void CollectRecords(ttgpu_handle *h) {
  const uint32_t *counters = h->pinned->report.counters;  // of the pass just rendered
  const uint32_t n = std::min(counters[kCountRecords], h->q.rec_capacity);
  h->records_last_pass = n;
  h->records_dropped += counters[kStatRecordsDropped];
  std::vector<float4> pw(n), dr(n);
  if (n) {
    Check(hipMemcpy(pw.data(), h->q.rec_pos_w, n * sizeof(float4), hipMemcpyDeviceToHost), "records");
    Check(hipMemcpy(dr.data(), h->q.rec_dir, n * sizeof(float4), hipMemcpyDeviceToHost), "records");
  }
  std::vector<guide::Record> recs(n);
  for (uint32_t k = 0; k < n; ++k) {
    guide::Record &r = recs[k];
    r.pos[0] = pw[k].x; r.pos[1] = pw[k].y; r.pos[2] = pw[k].z;
    r.weight = std::isfinite(pw[k].w) ? pw[k].w : 0.f;
    const float len = std::sqrt(dr[k].x * dr[k].x + dr[k].y * dr[k].y + dr[k].z * dr[k].z);
    r.dir[0] = dr[k].x / len; r.dir[1] = dr[k].y / len; r.dir[2] = dr[k].z / len;
    r.original = true;
  }
  h->recorder->FinalizeRound(recs);
}

// After a recording pass: refit the vMF-tree recorder on the host, or train the network on the
// device records (records stay on the GPU; only their count is read back).
void LearnFromPass(ttgpu_handle *h) {
  ++h->train_rounds;
  if (!h->learned) {
    // The first pass builds the kd-tree on the host (AdaptInitial); later passes fit on the device.
    if (h->recorder->round() == 0 || h->fit.host) CollectRecords(h);
    else GpuFitPass(h);
    return;
  }
  const uint32_t *counters = h->pinned->report.counters;  // of the pass just rendered
  const int64_t n = std::min(counters[kCountRecords], h->q.rec_capacity);
  h->records_last_pass = n;
  h->records_dropped += counters[kStatRecordsDropped];
  h->Timed("train", [&] { h->net->TrainOnRecords(h->q.rec_pos_w, h->q.rec_dir, h->q.rec_nrm, h->q.rec_wo, n, h->stream); });
  h->CollectTimers();
}

}  // namespace

void ttgpu::SetCreateError(const std::string &msg) { g_create_error = msg; }

namespace {

// A traversal that found its stack full dropped a subtree; the host's depth bound should make
// this impossible, so it is an error rather than a silently wrong image.
void CheckTraversal(hipStream_t st) {
  if (TakeStackOverflow(st)) throw std::runtime_error("BVH traversal stack overflow: the tree is deeper than the traversal stack allows");
}

int Fail(ttgpu_handle *h, int code, const std::string &msg) {
  if (h) h->err = msg;
  else g_create_error = msg;  // calls without a handle report through ttgpu_create_error()
  return code;
}

#define TTGPU_GUARD(h, ...)                                               \
  try {                                                                   \
    __VA_ARGS__                                                           \
  } catch (const std::invalid_argument &e) {                              \
    return Fail(h, TTGPU_ERR_INVALID_ARGUMENT, e.what());                 \
  } catch (const HipError &e) {                                           \
    return Fail(h, TTGPU_ERR_DEVICE, e.what());                           \
  } catch (const std::bad_alloc &e) {                                     \
    return Fail(h, TTGPU_ERR_OUT_OF_MEMORY, "host allocation failed");    \
  } catch (const std::exception &e) {                                     \
    return Fail(h, TTGPU_ERR_RUNTIME, e.what());                          \
  }

// Ends a pass: the counters and the traversal's overflow flag come back with the wait for the stream.
void FinishPass(ttgpu_handle *h, hipEvent_t ev1) {
  LaunchReport(h->q, &h->pinned_dev->report, h->stream);
  Check(hipGetLastError(), "kernel launch");
  Check(hipEventRecord(ev1, h->stream), "hipEventRecord");
  Check(hipStreamSynchronize(h->stream), "hipStreamSynchronize");
}
void CheckReport(const ttgpu_handle *h) {
  if (h->pinned->report.stack_overflow)
    throw std::runtime_error("BVH traversal stack overflow: the tree is deeper than the traversal stack allows");
}

// Waits until iteration `seq` has reported its progress.  The stream's state bounds the wait: once
// it has run dry (or failed) no report is on its way.  The wait polls, but where the one before was long
// too (`was_long`, kept over a pass), so that the iteration queued behind this one keeps the GPU busy, it
// leaves the core to others 20 us at a time.  (A wait may be long only because of the work queued before
// the pass: sleeping in it left the GPU idle, 0.4 ms per training sweep of the quadtree guide.)
const PassProgress &WaitProgress(ttgpu_handle *h, unsigned long long seq, bool &was_long) {
  constexpr unsigned kSpins = 8192;  // 0.1 to 0.4 ms, by the processor
  const bool sleep = was_long;
  was_long = false;
  for (unsigned spins = 1; !h->progress.Arrived(seq); ++spins) {
    if (spins % kSpins != 0 && !(sleep && was_long)) {
      __builtin_ia32_pause();
      continue;
    }
    was_long = true;
    const hipError_t e = hipStreamQuery(h->stream);
    if (e != hipErrorNotReady) {
      Check(e, "hipStreamQuery");
      if (!h->progress.Arrived(seq)) throw std::runtime_error("no progress report from the device (internal error)");
      break;
    }
    if (sleep) std::this_thread::sleep_for(std::chrono::microseconds(20));
  }
  return h->progress.Record(seq);
}

void ResetFramebuffer(ttgpu_handle *h) {
  LaunchFill(h->fb, h->fb_sq, 3 * (size_t)h->npix, 0.0, h->stream);
  Check(hipGetLastError(), "fill");
  std::fill(h->pixel_spp.begin(), h->pixel_spp.end(), 0);
}

// Renders `spp` samples per pixel as one stream of npix * spp camera paths through the wavefront:
// the first `capacity` paths start at once, and after every iteration (trace, shade, shadow rays)
// the slots of finished paths take the next camera paths, so launches stay full until the pass's
// last paths drain.  The host runs one iteration ahead of a 16-byte progress read-back.  A stop
// request ends the issuing of new paths; the paths in flight finish.  Returns false after a stop.
// bdpt: chunks of as many samples as the workspace holds; a stop request ends the pass after the
// chunk in flight.
bool RenderPassBdpt(ttgpu_handle *h, int spp) {
  const uint64_t npix = (uint64_t)h->npix;
  const uint64_t total = npix * (uint64_t)spp;
  const uint32_t spp_base = (uint32_t)h->total_spp;
  hipEvent_t ev0 = h->NextEvent(), ev1 = h->NextEvent();
  Check(hipEventRecord(ev0, h->stream), "hipEventRecord");
  uint64_t issued = 0;
  while (issued < total && !h->stop.load()) {
    const uint64_t n = std::min<uint64_t>(h->bdpt.capacity, total - issued);
    h->Timed("bdpt", [&] {
      LaunchBdpt(h->dsc, h->bdpt, issued, (uint32_t)n, (uint32_t)npix, spp_base, h->params.seed, h->fb, h->fb_sq, h->q.counters, h->stream);
    });
    Check(hipGetLastError(), "kernel launch");
    Check(hipStreamSynchronize(h->stream), "hipStreamSynchronize");
    issued += n;
    if (h->interrupt.exchange(false) && h->cb) h->cb(h->cb_user, 0);
  }
  FinishPass(h, ev1);
  const bool complete = issued == total;
  {
    const uint64_t full = issued / npix, rem = issued % npix;
    if (full)
      for (auto &c : h->pixel_spp) c += full;
    for (uint64_t k = 0; k < rem; ++k) h->pixel_spp[k] += 1;
  }
  h->stats.paths_traced += issued;
  float ms = 0.f;
  Check(hipEventElapsedTime(&ms, ev0, ev1), "hipEventElapsedTime");
  h->stats.render_ms = ms;
  h->CollectTimers();
  h->event_next = 0;
  CheckReport(h);
  h->stats.rays_closest = h->pinned->report.counters[kStatClosest];
  h->stats.rays_shadow = h->pinned->report.counters[kStatShadow];
  if (complete) {
    h->total_spp += spp;
    h->sched_total += spp;
  }
  h->stats.total_spp = h->total_spp;
  h->stats.passes += 1;
  return complete;
}

bool RenderPass(ttgpu_handle *h, int spp) {
  if (h->stop.load()) return false;
  if (h->params.algo == TTGPU_ALGO_BDPT) return RenderPassBdpt(h, spp);
  const uint64_t npix = (uint64_t)h->npix;
  const uint64_t total = npix * (uint64_t)spp;
  const uint32_t cap = h->capacity;
  PathQueues &q = h->q;
  hipEvent_t ev0 = h->NextEvent(), ev1 = h->NextEvent();
  Check(hipEventRecord(ev0, h->stream), "hipEventRecord");
  const uint32_t n0 = (uint32_t)std::min<uint64_t>(cap, total);
  const uint32_t spp_base = (uint32_t)h->total_spp;
  h->Timed("raygen", [&] { LaunchRaygen(h->dsc, q, n0, (uint32_t)npix, spp_base, h->params.seed, h->stream); });
  // Every path finishes within max_depth - 1 iterations, and then its slot takes a new path: at
  // most ceil(total / capacity) + 1 rounds of max_depth - 1 iterations.
  const uint64_t max_iter = (total / cap + 2) * (uint64_t)std::max(1, h->params.max_ray_depth) + 8;
  uint64_t limit = total;
  uint32_t *cur_q = q.queue_a, *nxt_q = q.queue_b;
  uint32_t *cur_c = q.counters + kCountA, *nxt_c = q.counters + kCountB;
  uint32_t *shadow_in = q.counters + kCountShadow2, *shadow_out = q.counters + kCountShadow;
  bool stopped = false;
  // Plain surface passes trace each iteration's shadow rays in the next closest-hit launch.
  const bool shadow_in_trace = ShadowInTrace(h->dsc, q);
  const bool slot_order = q.alive != nullptr;
  if (!slot_order) shadow_in = shadow_out;
  // Every queue holds at most the pass's n0 slots; once all paths are issued, at most the work
  // the last known iteration left (the launches' grids; their kernels stride over any count).
  uint32_t bound = n0;
  uint64_t issued = n0;  // as of the last iteration that has reported
  bool was_long = false;
  for (uint64_t it = 0;; ++it) {
    if (it > max_iter) throw std::runtime_error("path regeneration did not drain (internal error)");
    if (!stopped && h->stop.load()) {
      stopped = true;
      limit = 0;  // issue no further camera paths; the paths in flight finish
    }
    q.shadow_in = shadow_in;
    q.shadow_out = shadow_out;
    h->Timed("trace", [&] { LaunchTrace(h->dsc, q, cur_q, cur_c, bound, h->fb, h->fb_sq, shadow_in_trace, h->stream); });
    if (q.vt) h->Timed("media", [&] { LaunchTrackMedia(h->dsc, q, cur_q, cur_c, bound, h->stream); });
    if (h->learned)
      h->Timed("guide", [&] {
        LaunchGuideInfer(h->dsc, q, cur_q, cur_c, h->infer_sorted ? n0 : bound, h->net->View(),
                         h->infer_sorted ? &h->infer_sort : nullptr, h->stream);
      });
    if (!slot_order) {
      LaunchResetCounter(q.counters, (int)(nxt_c - q.counters), h->stream);
      LaunchResetCounter(q.counters, kCountShadow, h->stream);
    }
    h->Timed("shade", [&] { LaunchShade(h->dsc, q, cur_q, cur_c, nxt_q, nxt_c, bound, h->fb, h->fb_sq, h->stream); });
    if (!shadow_in_trace) h->Timed("shadow", [&] { LaunchShadow(h->dsc, q, bound, h->fb, h->fb_sq, h->stream); });
    const unsigned long long seq = h->progress.Next();
    h->Timed("raygen", [&] {
      LaunchRegen(h->dsc, q,
                  RegenArgs{nxt_q, nxt_c, n0, limit, (uint32_t)npix, spp_base, h->params.seed, shadow_in_trace, h->progress.Device(seq), seq,
                            h->select_temp},
                  h->stream);
    });
    Check(hipGetLastError(), "kernel launch");
    std::swap(cur_q, nxt_q);
    std::swap(cur_c, nxt_c);
    if (slot_order) std::swap(shadow_in, shadow_out);
    if (h->interrupt.exchange(false)) {
      Check(hipStreamSynchronize(h->stream), "sync");
      if (h->cb) h->cb(h->cb_user, 0);
    }
    // Wait for the previous iteration (this one is already queued behind it): an empty queue after
    // regeneration means every issued path has finished and none is left to issue.
    if (it > 0) {
      const PassProgress &r = WaitProgress(h, seq - 1, was_long);
      issued = r.issued;
      if (r.queued == 0) break;
      if (r.issued >= limit) bound = (uint32_t)std::min<uint64_t>(n0, r.queued);
    }
  }
  const bool complete = issued == total;
  // pt: the light connection at the camera node of every issued camera sample.
  if (h->dsc.algo_pt && h->dsc.sample_mode != TTGPU_SAMPLE_BSDF && h->dsc.cam.kind == TTGPU_CAMERA_PINHOLE)
    h->Timed("camera", [&] {
      LaunchCameraConnect(h->dsc, 0, issued, (uint32_t)npix, spp_base, h->params.seed, h->fb, h->fb_sq, q.counters, h->stream);
    });
  FinishPass(h, ev1);
  // Per-pixel sample counts: path g of the pass belongs to pixel g % npix.
  {
    const uint64_t full = issued / npix, rem = issued % npix;
    if (full)
      for (auto &c : h->pixel_spp) c += full;
    for (uint64_t k = 0; k < rem; ++k) h->pixel_spp[k] += 1;
  }
  h->stats.paths_traced += issued;
  float ms = 0.f;
  Check(hipEventElapsedTime(&ms, ev0, ev1), "hipEventElapsedTime");
  h->stats.render_ms = ms;
  h->CollectTimers();
  h->event_next = 0;
  CheckReport(h);
  h->stats.rays_closest = h->pinned->report.counters[kStatClosest];
  h->stats.rays_shadow = h->pinned->report.counters[kStatShadow];
  if (complete) {
    h->total_spp += spp;
    h->sched_total += spp;
  }
  h->stats.total_spp = h->total_spp;
  h->stats.passes += 1;
  return complete;
}

// ---- ray queries through page-locked staging ---------------------------------------------
// The caller's rays are copied in chunks into page-locked slots; a kernel takes a slot's rays to
// the device, and the trace writes the results into the slot.  The slots' streams overlap, so the
// host copies one chunk while the GPU fetches and traces others.  With seven hipMalloc / hipFree
// pairs and seven copies of pageable arrays per call, a million closest-hit rays of the 1 M triangle
// terrain took 2.6 ms, of which 0.35 were tracing; now 1.9 ms, bound by the host's copies and the link
// (occlusion: 1.6 and 1.5 ms), and 200,000 took 0.66 ms, now 0.50.  Six slots of 2^16 rays, which take the
// same memory: 1.79 and 1.51 ms for a million, but 0.52 (occlusion 0.45 against 0.40) for 200,000; four
// of 2^16: 2.0 and 1.76 ms; twelve of 2^15: 2.2 and 2.0.  Tracing straight from the page-locked rays took
// 5.2 ms for both queries instead of 3.65.
constexpr int kStageSlots = 3;
constexpr size_t kStageRays = 1 << 17;                // of a slot at most: 2048 waves, 5.8 MB
constexpr size_t kMinStageRays = 1 << 10;
constexpr size_t kRayBytes = 28;                      // origin, direction, tmax
constexpr size_t kStageBytesPerRay = kRayBytes + 16;  // and t, prim, u, v (or occluded)
struct RayStage {
  unsigned char *host = nullptr, *dev = nullptr;  // slots and their device address
  unsigned char *rays = nullptr;                  // device memory: a slot's rays each
  hipStream_t stream[kStageSlots] = {};           // of several slots; a single one uses the handle's
  hipEvent_t done[kStageSlots] = {}, begin = nullptr;
  size_t slot_rays = 0;
  int slots = 0, device = 0;
  void Free() {
    for (auto &e : done)
      if (e) (void)hipEventDestroy(e);
    if (begin) (void)hipEventDestroy(begin);
    for (auto &st : stream)
      if (st) (void)hipStreamDestroy(st);
    if (host) (void)hipHostFree(host);
    if (rays) (void)hipFree(rays);
    *this = RayStage{};
  }
};
// Stages are shared by the process's handles (a query borrows one, so queries of several threads
// each have their own; small ones leave the stages of several slots to the large); at most kMaxIdleStages are kept, and none after the last handle.
constexpr int kMaxIdleStages = 4;
std::mutex g_stage_mu;
IdleStages<RayStage, kMaxIdleStages> g_idle_stages;
int g_handles = 0;

// A stage for `count` rays: one slot of at least that many, or kStageSlots of kStageRays.
RayStage BorrowStage(size_t count) {
  RayStage s;
  Check(hipGetDevice(&s.device), "hipGetDevice");
  s.slots = count > kStageRays ? kStageSlots : 1;
  s.slot_rays = kMinStageRays;
  while (s.slot_rays < std::min(count, kStageRays)) s.slot_rays *= 2;
  {
    std::lock_guard<std::mutex> lock(g_stage_mu);
    const RayStage idle = g_idle_stages.Take(s);
    if (idle.slots) return idle;
  }
  try {
    const size_t rays = s.slots * s.slot_rays;
    Check(hipHostMalloc((void **)&s.host, rays * kStageBytesPerRay), "hipHostMalloc");
    Check(hipHostGetDevicePointer((void **)&s.dev, s.host, 0), "hipHostGetDevicePointer");
    Check(hipMalloc((void **)&s.rays, rays * kRayBytes), "hipMalloc");
    Check(hipEventCreateWithFlags(&s.begin, hipEventDisableTiming), "hipEventCreate");
    for (int k = 0; k < s.slots; ++k) {
      Check(hipEventCreateWithFlags(&s.done[k], hipEventDisableTiming), "hipEventCreate");
      if (s.slots > 1) Check(hipStreamCreateWithFlags(&s.stream[k], hipStreamNonBlocking), "hipStreamCreate");
    }
  } catch (...) {
    s.Free();
    throw;
  }
  return s;
}
void ReturnStage(RayStage s) noexcept {
  {
    std::lock_guard<std::mutex> lock(g_stage_mu);
    if (g_handles > 0) s = g_idle_stages.Put(s);
  }
  if (s.slots) s.Free();
}
void CountHandle(int d) noexcept {
  IdleStages<RayStage, kMaxIdleStages> drop;
  {
    std::lock_guard<std::mutex> lock(g_stage_mu);
    g_handles += d;
    if (g_handles == 0) std::swap(drop, g_idle_stages);
  }
  for (RayStage s = drop.Drop(); s.slots; s = drop.Drop()) s.Free();
}

// Closest hits (t, prim, u, v) or, with `occluded`, occlusion of `count` rays.
void QueryRays(ttgpu_handle *h, size_t count, const float *org, const float *dir, const float *tmax, float *t, int32_t *prim, float *u,
               float *v, int32_t *occluded, int brute) {
  struct Loan {
    hipStream_t own;
    RayStage s;
    ~Loan() {  // no kernel may still use the slots
      (void)hipStreamSynchronize(own);
      for (auto &st : s.stream)
        if (st) (void)hipStreamSynchronize(st);
      ReturnStage(s);
    }
  } loan{h->stream, BorrowStage(count)};
  RayStage &s = loan.s;
  const size_t R = s.slot_rays, chunks = (count + R - 1) / R, slots = (size_t)s.slots;
  // Slot layout: origins (12 R bytes), directions (12 R), tmax (4 R), then four result arrays (4 R each).
  auto in_slot = [&](unsigned char *base, size_t slot, size_t offset) { return base + slot * R * kStageBytesPerRay + offset * R; };
  auto collect = [&](size_t chunk) {
    const size_t slot = chunk % slots, at = chunk * R, n = std::min(R, count - at);
    Check(hipEventSynchronize(s.done[slot]), "hipEventSynchronize");
    if (occluded) {
      std::memcpy(occluded + at, in_slot(s.host, slot, 28), 4 * n);
      return;
    }
    std::memcpy(t + at, in_slot(s.host, slot, 28), 4 * n);
    std::memcpy(prim + at, in_slot(s.host, slot, 32), 4 * n);
    std::memcpy(u + at, in_slot(s.host, slot, 36), 4 * n);
    std::memcpy(v + at, in_slot(s.host, slot, 40), 4 * n);
  };
  if (slots > 1) {
    Check(hipEventRecord(s.begin, h->stream), "hipEventRecord");
    for (auto &st : s.stream) Check(hipStreamWaitEvent(st, s.begin, 0), "hipStreamWaitEvent");
  }
  for (size_t c = 0; c < chunks; ++c) {
    if (c >= slots) collect(c - slots);
    const size_t slot = c % slots, at = c * R, n = std::min(R, count - at);
    std::memcpy(in_slot(s.host, slot, 0), org + 3 * at, 12 * n);
    std::memcpy(in_slot(s.host, slot, 12), dir + 3 * at, 12 * n);
    std::memcpy(in_slot(s.host, slot, 24), tmax + at, 4 * n);
    hipStream_t st = slots > 1 ? s.stream[slot] : h->stream;
    unsigned char *rays = s.rays + slot * R * kRayBytes;
    auto ray = [&](size_t offset) { return reinterpret_cast<const float *>(rays + offset * R); };
    auto out = [&](size_t offset) { return reinterpret_cast<float *>(in_slot(s.dev, slot, offset)); };
    LaunchCopyRays(rays, in_slot(s.dev, slot, 0), n, R, st);
    if (occluded)
      LaunchTraceRays(h->dsc, (int64_t)n, ray(0), ray(12), ray(24), nullptr, nullptr, nullptr, nullptr,
                      reinterpret_cast<int32_t *>(out(28)), 0, st);
    else
      LaunchTraceRays(h->dsc, (int64_t)n, ray(0), ray(12), ray(24), out(28), reinterpret_cast<int32_t *>(out(32)), out(36), out(40),
                      nullptr, brute, st);
    Check(hipGetLastError(), "launch");
    Check(hipEventRecord(s.done[slot], st), "hipEventRecord");
  }
  for (size_t c = chunks > slots ? chunks - slots : 0; c < chunks; ++c) collect(c);
  CheckTraversal(h->stream);  // of every chunk
}

}  // namespace

extern "C" {

int ttgpu_abi_version(void) { return TTGPU_ABI_VERSION; }

const char *ttgpu_device_info(void) {
  static std::string info;
  int dev = 0;
  hipDeviceProp_t p;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&p, dev) != hipSuccess) {
    info = "no HIP device";
  } else {
    info = std::string(p.gcnArchName) + ", " + std::to_string(p.multiProcessorCount) + " CUs, " +
           std::to_string(p.totalGlobalMem >> 30) + " GiB, " + p.name;
  }
  return info.c_str();
}

const char *ttgpu_create_error(void) { return g_create_error.c_str(); }

int ttgpu_create(const ttgpu_scene *scene, const ttgpu_params *params, ttgpu_handle **out) {
  if (!scene || !params || !out) {
    g_create_error = "null argument";
    return TTGPU_ERR_INVALID_ARGUMENT;
  }
  *out = nullptr;
  ttgpu_handle *h = nullptr;
  try {
    Validate(*scene, *params);
    EnsureTables();
    h = new ttgpu_handle();
    h->params = *params;
    if (h->params.num_wavelengths == 0) h->params.num_wavelengths = 4;
    h->npix = params->width * params->height;
    h->pixel_spp.assign(h->npix, 0);
    h->sched_spp = 1;
    Check(hipGetDevice(&h->device), "hipGetDevice");
    Check(hipStreamCreate(&h->stream), "hipStreamCreate");
    ScratchOnCurrentDevice();  // the allocation-free entry point's memory, looked up once per device
    auto t0 = std::chrono::steady_clock::now();
    const ttgpu_scene &s = *scene;
    std::vector<int64_t> surf, vol;
    const int64_t nprim = s.num_triangles + s.num_spheres;
    for (int64_t p = 0; p < nprim; ++p) {
      int m = p < s.num_triangles ? s.tri_material[p] : s.sphere_material[p - s.num_triangles];
      (s.materials[m].shader >= 0 ? surf : vol).push_back(p);
    }
    h->num_triangles = (int)s.num_triangles;
    h->dsc.num_triangles = (int)s.num_triangles;
    BuildGeometry(h, s, surf, true);
    BuildGeometry(h, s, vol, false);
    // Scene bounds over all primitives (src/scene.cxx:139-140).
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int64_t p = 0; p < nprim; ++p) {
      if (p < s.num_triangles) {
        for (int j = 0; j < 3; ++j) {
          const float *v = s.vertices + 3 * s.indices[3 * p + j];
          for (int a = 0; a < 3; ++a) { lo[a] = std::min(lo[a], (double)v[a]); hi[a] = std::max(hi[a], (double)v[a]); }
        }
      } else {
        const float *sp = s.spheres + 4 * (p - s.num_triangles);
        for (int a = 0; a < 3; ++a) { lo[a] = std::min(lo[a], (double)sp[a] - sp[3]); hi[a] = std::max(hi[a], (double)sp[a] + sp[3]); }
      }
    }
    double diag = nprim ? std::sqrt((hi[0] - lo[0]) * (hi[0] - lo[0]) + (hi[1] - lo[1]) * (hi[1] - lo[1]) + (hi[2] - lo[2]) * (hi[2] - lo[2]))
                        : 1.0;
    BuildTables(h, s, diag);
    h->dsc.bb_center = nprim ? make_float3((float)(0.5 * (lo[0] + hi[0])), (float)(0.5 * (lo[1] + hi[1])), (float)(0.5 * (lo[2] + hi[2])))
                             : make_float3(0.f, 0.f, 0.f);
    h->guided = params->algo == TTGPU_ALGO_PTG;
    h->learned = h->guided && params->guide_kind == TTGPU_GUIDE_LEARNED;
    if (h->guided) {
      // The guided integrator's MIS (power heuristic) always includes the light-selection
      // probability in the NEE pdf.
      h->params.mis_mode = TTGPU_MIS_CONSISTENT;
      h->dsc.mis_mode = TTGPU_MIS_CONSISTENT;
    }
    int64_t cap = params->wavefront_paths > 0 ? params->wavefront_paths : (int64_t)1 << 22;
    cap = std::min<int64_t>(cap, (int64_t)1 << 26);
    h->capacity = (uint32_t)cap;
    h->stats.wavefront_paths = (int32_t)cap;
    AllocateQueues(h);
    if (h->learned) {
      const float flo[3] = {(float)lo[0], (float)lo[1], (float)lo[2]}, fhi[3] = {(float)hi[0], (float)hi[1], (float)hi[2]};
      h->net = std::make_unique<nn::NeuralGuide>(nn::NeuralGuideConfig{}, flo, fhi, params->seed);
    } else if (h->guided) {
      const int subdiv = params->guide_subdiv_factor > 0 ? params->guide_subdiv_factor : 100;
      // The quadtree is the reference's active directional model, and the default.
      const bool quadtree = params->guide_kind == TTGPU_GUIDE_QUADTREE || params->guide_kind == TTGPU_GUIDE_NONE;
      h->recorder = std::make_unique<guide::Recorder>(subdiv, params->seed, params->num_threads, quadtree);
      // The per-pass fit runs on the device; TTGPU_GUIDE_HOST_FIT=1 runs it on the host threads.
      const char *hf = std::getenv("TTGPU_GUIDE_HOST_FIT");
      h->fit.host = hf && hf[0] == '1';
      UploadGuide(h);
    }
    auto t1 = std::chrono::steady_clock::now();
    h->stats.upload_ms = std::chrono::duration<double, std::milli>(t1 - t0).count() - h->stats.bvh_build_ms;
    *out = h;
    CountHandle(1);
    return TTGPU_OK;
  } catch (const std::invalid_argument &e) {
    g_create_error = e.what();
    delete h;
    return TTGPU_ERR_INVALID_ARGUMENT;
  } catch (const HipError &e) {
    g_create_error = e.what();
    delete h;
    return TTGPU_ERR_DEVICE;
  } catch (const std::exception &e) {
    g_create_error = e.what();
    delete h;
    return TTGPU_ERR_RUNTIME;
  }
}

void ttgpu_destroy(ttgpu_handle *h) {
  if (!h) return;
  delete h;
  CountHandle(-1);
}

const char *ttgpu_last_error(const ttgpu_handle *h) { return h ? h->err.c_str() : g_create_error.c_str(); }

int ttgpu_request_interrupt(ttgpu_handle *h) {
  if (!h) return TTGPU_ERR_INVALID_ARGUMENT;
  h->interrupt.store(true);
  return TTGPU_OK;
}

int ttgpu_request_stop(ttgpu_handle *h) {
  if (!h) return TTGPU_ERR_INVALID_ARGUMENT;
  h->stop.store(true);
  return TTGPU_OK;
}

int ttgpu_set_pass_callback(ttgpu_handle *h, ttgpu_pass_callback cb, void *user) {
  if (!h) return TTGPU_ERR_INVALID_ARGUMENT;
  h->cb = cb;
  h->cb_user = user;
  return TTGPU_OK;
}

int ttgpu_render_spp(ttgpu_handle *h, int32_t spp) {
  if (!h) return TTGPU_ERR_INVALID_ARGUMENT;
  if (spp <= 0) return Fail(h, TTGPU_ERR_INVALID_ARGUMENT, "spp must be positive");
  TTGPU_GUARD(h, { return RenderPass(h, spp) ? TTGPU_OK : TTGPU_ERR_INTERRUPTED; })
}

int ttgpu_run(ttgpu_handle *h, int32_t max_passes) {
  if (!h) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(h, {
    constexpr int kMaxSppPerIteration = 1024;
    const int max_spp = h->params.max_samples_per_pixel;
    int passes = 0;
    if (h->guided && !h->trained) {
      // Training (guided PathTracingAlgo2::Run, src/renderingalgorithms_pathtracing_guided.cxx:1110-1160):
      // an initial 1-spp pass builds the kd-tree, then sweeps of 2, 4, .. 1-spp passes refit the
      // cells after every pass and split cells / bake mixtures after every sweep.
      h->dsc.guide_record = 1;
      if (!h->stop.load()) {
        RenderPass(h, 1);
        LearnFromPass(h);
        if (!h->learned) {
          UploadGuide(h);
          if (!h->fit.host) UploadFit(h);
        }
        if (h->cb) h->cb(h->cb_user, 1);
      }
      for (int num = 2; !h->stop.load() && num <= h->params.guide_max_spp; num *= 2) {
        ResetFramebuffer(h);
        for (int k = 0; k < num && !h->stop.load(); ++k) {
          RenderPass(h, 1);
          LearnFromPass(h);
          // The quadtree's fit updates the sampled distributions after every pass (in place on
          // the device when the fit runs there).
          if (h->recorder && h->recorder->quadtree() && h->fit.host) UploadGuide(h);
        }
        if (h->cb) h->cb(h->cb_user, 1);
        if (!h->learned) {
          if (!h->fit.host) DownloadFit(h);
          h->recorder->PrepareAdaptedStructures();
          UploadGuide(h);
          if (!h->fit.host) UploadFit(h);
        }
      }
      h->dsc.guide_record = 0;
      if (h->stop.load()) return TTGPU_ERR_INTERRUPTED;
      ResetFramebuffer(h);
      h->trained = true;
      h->sched_total = 0;
      h->sched_spp = 1;
    }
    // SamplesPerPixelSchedule (src/renderingalgorithms_simplebase.hxx:34-62).
    if (max_spp > 0 && (int64_t)h->sched_total + h->sched_spp > max_spp) h->sched_spp = max_spp - (int)h->sched_total;
    while (!h->stop.load() && h->sched_spp > 0 && (max_passes <= 0 || passes < max_passes)) {
      RenderPass(h, h->sched_spp);
      ++passes;
      if (h->cb) h->cb(h->cb_user, 1);
      if (h->sched_spp < kMaxSppPerIteration) h->sched_spp *= 2;
      if (max_spp > 0 && (int64_t)h->sched_total + h->sched_spp > max_spp) h->sched_spp = max_spp - (int)h->sched_total;
    }
    return h->stop.load() ? TTGPU_ERR_INTERRUPTED : TTGPU_OK;
  })
}

int ttgpu_write_image(ttgpu_handle *h, const char *path, int32_t format) {
  if (!h || !path) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(h, {
    const size_t n = (size_t)h->npix;
    std::vector<double> rgb(3 * n);
    Check(hipMemcpy(rgb.data(), h->fb, rgb.size() * sizeof(double), hipMemcpyDeviceToHost), "read framebuffer");
    std::vector<float> img(3 * n);
    for (size_t p = 0; p < n; ++p) {
      const double s = h->pixel_spp[p] ? 1.0 / (double)h->pixel_spp[p] : 0.0;
      for (int c = 0; c < 3; ++c) img[3 * p + c] = (float)(rgb[3 * p + c] * s);
    }
    const int rc = ttgpu_write_rgb_image(img.data(), h->params.width, h->params.height, path, format);
    if (rc != TTGPU_OK) return Fail(h, rc, std::string("could not write ") + path);
    return TTGPU_OK;
  })
}

int ttgpu_reset_framebuffer(ttgpu_handle *h) {
  if (!h) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(h, {
    ResetFramebuffer(h);
    return TTGPU_OK;
  })
}

int ttgpu_read_framebuffer(ttgpu_handle *h, double *rgb, double *rgb_sq, uint64_t *spp) {
  if (!h) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(h, {
    Check(hipStreamSynchronize(h->stream), "sync");
    if (rgb) Check(hipMemcpy(rgb, h->fb, 3 * (size_t)h->npix * sizeof(double), hipMemcpyDeviceToHost), "read fb");
    if (rgb_sq) Check(hipMemcpy(rgb_sq, h->fb_sq, 3 * (size_t)h->npix * sizeof(double), hipMemcpyDeviceToHost), "read fb_sq");
    if (spp) std::memcpy(spp, h->pixel_spp.data(), h->pixel_spp.size() * sizeof(uint64_t));
    return TTGPU_OK;
  })
}

int ttgpu_generate_image(ttgpu_handle *h, uint8_t *rgb8) {
  if (!h || !rgb8) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(h, {
    std::vector<double> fb(3 * (size_t)h->npix);
    Check(hipStreamSynchronize(h->stream), "sync");
    Check(hipMemcpy(fb.data(), h->fb, fb.size() * sizeof(double), hipMemcpyDeviceToHost), "read fb");
    const int W = h->params.width, H = h->params.height;
    // framebuffer::ToImage (src/renderbuffer.hxx:99-125): average, clamp, sRGB, rows flipped.
    for (int y = 0; y < H; ++y)
      for (int x = 0; x < W; ++x) {
        const size_t p = (size_t)y * W + x;
        const double n = (double)h->pixel_spp[p];
        uint8_t *dst = rgb8 + 3 * ((size_t)(H - 1 - y) * W + x);
        for (int c = 0; c < 3; ++c) {
          double v = n > 0 ? fb[3 * p + c] / n : 0.0;
          v = std::min(1.0, std::max(0.0, v));
          if (!h->params.linear_output) v = v <= 0.0031308 ? 12.92 * v : 1.055 * std::pow(v, 1.0 / 2.4) - 0.055;
          dst[c] = (uint8_t)(v * 255.999);
        }
      }
    return TTGPU_OK;
  })
}

int ttgpu_stats_get(ttgpu_handle *h, ttgpu_stats *out) {
  if (!h || !out) return TTGPU_ERR_INVALID_ARGUMENT;
  *out = h->stats;
  return TTGPU_OK;
}

int ttgpu_enable_kernel_timing(ttgpu_handle *h, int32_t enable) {
  if (!h) return TTGPU_ERR_INVALID_ARGUMENT;
  h->timing = enable != 0;
  h->timers.clear();
  return TTGPU_OK;
}

int ttgpu_kernel_time(ttgpu_handle *h, const char *name, double *total_ms, int64_t *launches) {
  if (!h || !name) return TTGPU_ERR_INVALID_ARGUMENT;
  auto it = h->timers.find(name);
  if (total_ms) *total_ms = it == h->timers.end() ? 0.0 : it->second.ms;
  if (launches) *launches = it == h->timers.end() ? 0 : it->second.launches;
  return TTGPU_OK;
}

static int TraceClosestImpl(ttgpu_handle *h, int64_t count, const float *org, const float *dir, const float *tmax, float *t,
                            int32_t *prim, float *u, float *v, int brute) {
  if (!h || count < 0 || (count && (!org || !dir || !tmax || !t || !prim || !u || !v))) return TTGPU_ERR_INVALID_ARGUMENT;
  if (count == 0) return TTGPU_OK;
  TTGPU_GUARD(h, {
    if (h->dsc.num_prims > 0) {
      QueryRays(h, (size_t)count, org, dir, tmax, t, prim, u, v, nullptr, brute);
    } else {
      for (int64_t i = 0; i < count; ++i) { t[i] = INFINITY; prim[i] = -1; u[i] = v[i] = 0.f; }
    }
    return TTGPU_OK;
  })
}

int ttgpu_trace_closest(ttgpu_handle *h, int64_t count, const float *org, const float *dir, const float *tmax, float *t, int32_t *prim,
                        float *u, float *v) {
  return TraceClosestImpl(h, count, org, dir, tmax, t, prim, u, v, 0);
}

// ---- allocation-free closest-hit query ------------------------------------------------
// Staging for the rays and hits of ttgpu_trace_closest_noalloc: TTGPU_NOALLOC_MAX_RAYS rays of
// 44 bytes (origin, direction, tmax in; t, prim, u, v out), 11.5 MB per GPU, held until the
// process ends.  Host code never passes `scratch` itself to a kernel or a copy (its host-side
// name is not a device address): it uses the per-device address from hipGetSymbolAddress.
namespace {
constexpr size_t kNoAllocRays = TTGPU_NOALLOC_MAX_RAYS;
constexpr size_t kNoAllocBytesPerRay = 44;
static __device__ __align__(256) unsigned char scratch[kNoAllocRays * kNoAllocBytesPerRay];
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current device, looked up once per device.
void *ScratchOnCurrentDevice() {
  int dev = -1;
  Check(hipGetDevice(&dev), "hipGetDevice");
  if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("device index out of range for the scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    Check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
    if (!p) throw HipError("hipGetSymbolAddress(scratch) returned a null address");
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}
}  // namespace

int ttgpu_trace_closest_noalloc(ttgpu_handle *h, int64_t count, const float *org, const float *dir, const float *tmax, float *t,
                                int32_t *prim, float *u, float *v) {
  if (!h || count < 0 || (count && (!org || !dir || !tmax || !t || !prim || !u || !v))) return TTGPU_ERR_INVALID_ARGUMENT;
  if (count > (int64_t)kNoAllocRays)
    return Fail(h, TTGPU_ERR_INVALID_ARGUMENT,
                "ttgpu_trace_closest_noalloc: " + std::to_string(count) + " rays exceed the limit of " +
                    std::to_string(kNoAllocRays) + " (TTGPU_NOALLOC_MAX_RAYS); use ttgpu_trace_closest or split the batch");
  TTGPU_GUARD(h, {
    int dev = -1;
    Check(hipGetDevice(&dev), "hipGetDevice");
    if (dev != h->device)
      return Fail(h, TTGPU_ERR_INVALID_ARGUMENT, "ttgpu_trace_closest_noalloc: the handle was created on device " +
                                                   std::to_string(h->device) + " but device " + std::to_string(dev) +
                                                   " is current");
    unsigned char *base = static_cast<unsigned char *>(ScratchOnCurrentDevice());
    if (count == 0) return TTGPU_OK;
    const size_t n = (size_t)count, M = kNoAllocRays;
    float *d_org = reinterpret_cast<float *>(base);
    float *d_dir = reinterpret_cast<float *>(base + 12 * M);
    float *d_tmax = reinterpret_cast<float *>(base + 24 * M);
    float *d_t = reinterpret_cast<float *>(base + 28 * M);
    int32_t *d_prim = reinterpret_cast<int32_t *>(base + 32 * M);
    float *d_u = reinterpret_cast<float *>(base + 36 * M);
    float *d_v = reinterpret_cast<float *>(base + 40 * M);
    if (h->dsc.num_prims == 0) {
      for (size_t i = 0; i < n; ++i) { t[i] = INFINITY; prim[i] = -1; u[i] = v[i] = 0.f; }
      return TTGPU_OK;
    }
    // Every output entry below `count` is written by the kernel, so nothing needs clearing; the
    // copies and the launch are ordered on the handle's stream.
    Check(hipMemcpyAsync(d_org, org, 3 * n * 4, hipMemcpyHostToDevice, h->stream), "H2D");
    Check(hipMemcpyAsync(d_dir, dir, 3 * n * 4, hipMemcpyHostToDevice, h->stream), "H2D");
    Check(hipMemcpyAsync(d_tmax, tmax, n * 4, hipMemcpyHostToDevice, h->stream), "H2D");
    LaunchTraceRays(h->dsc, count, d_org, d_dir, d_tmax, d_t, d_prim, d_u, d_v, nullptr, 0, h->stream);
    Check(hipGetLastError(), "launch");
    Check(hipMemcpyAsync(t, d_t, n * 4, hipMemcpyDeviceToHost, h->stream), "D2H");
    Check(hipMemcpyAsync(prim, d_prim, n * 4, hipMemcpyDeviceToHost, h->stream), "D2H");
    Check(hipMemcpyAsync(u, d_u, n * 4, hipMemcpyDeviceToHost, h->stream), "D2H");
    Check(hipMemcpyAsync(v, d_v, n * 4, hipMemcpyDeviceToHost, h->stream), "D2H");
    Check(hipStreamSynchronize(h->stream), "sync");
    CheckTraversal(h->stream);
    return TTGPU_OK;
  })
}

int ttgpu_trace_closest_bruteforce(ttgpu_handle *h, int64_t count, const float *org, const float *dir, const float *tmax, float *t,
                                   int32_t *prim, float *u, float *v) {
  return TraceClosestImpl(h, count, org, dir, tmax, t, prim, u, v, 1);
}

int ttgpu_media_events(ttgpu_handle *h, const ttgpu_scene *scene, int64_t count, const float *org, const float *dir, const float *tmax,
                       int32_t max_events, int32_t *out_initial, double *out_t, int32_t *out_medium, int32_t *out_count) {
  if (!h || !scene || count < 0 || max_events < 0 ||
      (count && (!org || !dir || !tmax || !out_initial || !out_count || (max_events && (!out_t || !out_medium)))))
    return TTGPU_ERR_INVALID_ARGUMENT;
  if (count == 0) return TTGPU_OK;
  TTGPU_GUARD(h, {
    const size_t n = (size_t)count, ne = n * (size_t)max_events;
    const int empty = h->dsc.empty_space_medium;
    std::vector<uint64_t> init(n);
    auto as_id = [](uint32_t m) { return m == (uint32_t)kVacuum ? -1 : (int32_t)m; };
    for (size_t i = 0; i < n; ++i) {
      init[i] = TrackerAt(*scene, empty, V3d{org[3 * i], org[3 * i + 1], org[3 * i + 2]});
      out_initial[i] = as_id((uint32_t)(init[i] & 0xFFFFFFFFu));
    }
    DevBuffer<float> d_org(3 * n), d_dir(3 * n), d_tmax(n);
    DevBuffer<uint64_t> d_init(n);
    DevBuffer<double> d_t(std::max<size_t>(ne, 1));
    DevBuffer<int32_t> d_med(std::max<size_t>(ne, 1)), d_cnt(n);
    Check(hipMemcpy(d_org.p, org, 3 * n * 4, hipMemcpyHostToDevice), "H2D");
    Check(hipMemcpy(d_dir.p, dir, 3 * n * 4, hipMemcpyHostToDevice), "H2D");
    Check(hipMemcpy(d_tmax.p, tmax, n * 4, hipMemcpyHostToDevice), "H2D");
    Check(hipMemcpy(d_init.p, init.data(), n * 8, hipMemcpyHostToDevice), "H2D");
    LaunchMediaEvents(h->dsc, count, d_org.p, d_dir.p, d_tmax.p, d_init.p, max_events, d_t.p, d_med.p, d_cnt.p, h->stream);
    Check(hipGetLastError(), "launch");
    Check(hipStreamSynchronize(h->stream), "sync");
    Check(hipMemcpy(out_count, d_cnt.p, n * 4, hipMemcpyDeviceToHost), "D2H");
    CheckTraversal(h->stream);
    if (ne) {
      Check(hipMemcpy(out_t, d_t.p, ne * 8, hipMemcpyDeviceToHost), "D2H");
      Check(hipMemcpy(out_medium, d_med.p, ne * 4, hipMemcpyDeviceToHost), "D2H");
    }
    return TTGPU_OK;
  })
}

int ttgpu_trace_occluded(ttgpu_handle *h, int64_t count, const float *org, const float *dir, const float *tmax, int32_t *occluded) {
  if (!h || count < 0 || (count && (!org || !dir || !tmax || !occluded))) return TTGPU_ERR_INVALID_ARGUMENT;
  if (count == 0) return TTGPU_OK;
  TTGPU_GUARD(h, {
    if (h->dsc.num_prims > 0) QueryRays(h, (size_t)count, org, dir, tmax, nullptr, nullptr, nullptr, nullptr, occluded, 0);
    else std::fill(occluded, occluded + count, 0);
    return TTGPU_OK;
  })
}

static DevShader ToDev(const ttgpu_shader &a) {
  DevShader d;
  d.kind = a.kind; d.alpha = a.alpha; d.alpha_min = a.alpha_min; d.ior_ratio = a.ior_ratio;
  d.ior_lambda_coeff = a.ior_lambda_coeff; d.specular = a.specular;
  std::memcpy(d.reflectance, a.reflectance, sizeof(d.reflectance));
  return d;
}

static int SamplerCall(int64_t count, size_t out_floats_per, std::function<void(float *, float *, float *)> launch, float *od, float *ov,
                       float *op, size_t dir_floats, size_t val_floats) {
  float *dd = nullptr, *dv = nullptr, *dp = nullptr;
  size_t n = (size_t)count;
  try {
    EnsureTables();
    if (dir_floats) Check(hipMalloc(&dd, dir_floats * n * 4), "hipMalloc");
    Check(hipMalloc(&dv, val_floats * n * 4), "hipMalloc");
    Check(hipMalloc(&dp, n * 4), "hipMalloc");
    launch(dd, dv, dp);
    Check(hipGetLastError(), "launch");
    Check(hipDeviceSynchronize(), "sync");
    if (dir_floats) Check(hipMemcpy(od, dd, dir_floats * n * 4, hipMemcpyDeviceToHost), "D2H");
    Check(hipMemcpy(ov, dv, val_floats * n * 4, hipMemcpyDeviceToHost), "D2H");
    Check(hipMemcpy(op, dp, n * 4, hipMemcpyDeviceToHost), "D2H");
  } catch (const std::exception &e) {
    g_create_error = e.what();
    if (dd) (void)hipFree(dd);
    if (dv) (void)hipFree(dv);
    if (dp) (void)hipFree(dp);
    return TTGPU_ERR_DEVICE;
  }
  (void)out_floats_per;
  if (dd) (void)hipFree(dd);
  (void)hipFree(dv);
  (void)hipFree(dp);
  return TTGPU_OK;
}

int ttgpu_sample_shader(const ttgpu_shader *shader, const float wi[3], const float ng[3], const float ns[3], const int32_t bins[4],
                        float roughness, uint64_t seed, int64_t count, float *out_dir, float *out_value, float *out_pdf) {
  if (!shader || !wi || !ng || !ns || !bins || count < 0 || (count && (!out_dir || !out_value || !out_pdf)))
    return TTGPU_ERR_INVALID_ARGUMENT;
  for (int i = 0; i < 4; ++i)
    if (bins[i] < 0 || bins[i] >= kNBins) return TTGPU_ERR_INVALID_ARGUMENT;
  if (count == 0) return TTGPU_OK;
  DevShader d = ToDev(*shader);
  uint32_t pb = (uint32_t)bins[0] | ((uint32_t)bins[1] << 8) | ((uint32_t)bins[2] << 16) | ((uint32_t)bins[3] << 24);
  return SamplerCall(count, 8, [&](float *dd, float *dv, float *dp) {
    LaunchSampleShader(d, make_float3(wi[0], wi[1], wi[2]), make_float3(ng[0], ng[1], ng[2]), make_float3(ns[0], ns[1], ns[2]), pb,
                       roughness, seed, count, dd, dv, dp, nullptr);
  }, out_dir, out_value, out_pdf, 3, 4);
}

int ttgpu_eval_shader(const ttgpu_shader *shader, const float wi[3], const float ng[3], const float ns[3], const int32_t bins[4],
                      float roughness, int64_t count, const float *dirs, float *out_value, float *out_pdf) {
  if (!shader || !wi || !ng || !ns || !bins || count < 0 || (count && (!dirs || !out_value || !out_pdf))) return TTGPU_ERR_INVALID_ARGUMENT;
  for (int i = 0; i < 4; ++i)
    if (bins[i] < 0 || bins[i] >= kNBins) return TTGPU_ERR_INVALID_ARGUMENT;
  if (count == 0) return TTGPU_OK;
  DevShader d = ToDev(*shader);
  uint32_t pb = (uint32_t)bins[0] | ((uint32_t)bins[1] << 8) | ((uint32_t)bins[2] << 16) | ((uint32_t)bins[3] << 24);
  float *ddirs = nullptr;
  if (hipMalloc(&ddirs, 3 * (size_t)count * 4) != hipSuccess) return TTGPU_ERR_DEVICE;
  if (hipMemcpy(ddirs, dirs, 3 * (size_t)count * 4, hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipFree(ddirs);
    return TTGPU_ERR_DEVICE;
  }
  int rc = SamplerCall(count, 5, [&](float *, float *dv, float *dp) {
    LaunchEvalShader(d, make_float3(wi[0], wi[1], wi[2]), make_float3(ng[0], ng[1], ng[2]), make_float3(ns[0], ns[1], ns[2]), pb,
                     roughness, count, ddirs, dv, dp, nullptr);
  }, nullptr, out_value, out_pdf, 0, 4);
  (void)hipFree(ddirs);
  return rc;
}

int ttgpu_sample_phase(int32_t phase_kind, float g, const float wi[3], uint64_t seed, int64_t count, float *out_dir, float *out_value,
                       float *out_pdf) {
  if (!wi || count < 0 || (count && (!out_dir || !out_value || !out_pdf))) return TTGPU_ERR_INVALID_ARGUMENT;
  if (phase_kind < 0 || phase_kind > TTGPU_PHASE_RAYLEIGH) return TTGPU_ERR_INVALID_ARGUMENT;
  if (count == 0) return TTGPU_OK;
  return SamplerCall(count, 5, [&](float *dd, float *dv, float *dp) {
    LaunchSamplePhase(phase_kind, g, make_float3(wi[0], wi[1], wi[2]), seed, count, dd, dv, dp, nullptr);
  }, out_dir, out_value, out_pdf, 3, 1);
}

int ttgpu_sample_phase_mixture(const int32_t kinds[2], const float g[2], const float weights[8], const float wi[3], uint64_t seed,
                               int64_t count, float *out_dir, float *out_value, float *out_pdf) {
  if (!kinds || !g || !weights || !wi || count < 0 || (count && (!out_dir || !out_value || !out_pdf))) return TTGPU_ERR_INVALID_ARGUMENT;
  for (int c = 0; c < 2; ++c)
    if (kinds[c] < 0 || kinds[c] > TTGPU_PHASE_RAYLEIGH) return TTGPU_ERR_INVALID_ARGUMENT;
  for (int k = 0; k < 8; ++k)
    if (!(weights[k] >= 0.f)) return TTGPU_ERR_INVALID_ARGUMENT;
  for (int k = 0; k < 4; ++k)  // every wavelength needs a positive total weight (phasefunctions.cxx:219)
    if (!(weights[k] + weights[4 + k] > 0.f)) return TTGPU_ERR_INVALID_ARGUMENT;
  if (count == 0) return TTGPU_OK;
  const PhaseMix m = phase_mix(kinds[0], g[0], make_float4(weights[0], weights[1], weights[2], weights[3]), kinds[1], g[1],
                               make_float4(weights[4], weights[5], weights[6], weights[7]));
  return SamplerCall(count, 8, [&](float *dd, float *dv, float *dp) {
    LaunchSamplePhaseMix(m, make_float3(wi[0], wi[1], wi[2]), seed, count, dd, dv, dp, nullptr);
  }, out_dir, out_value, out_pdf, 3, 4);
}

int ttgpu_pcg32(uint64_t initstate, uint64_t initseq, int64_t count, uint32_t *out) {
  if (count < 0 || (count && !out)) return TTGPU_ERR_INVALID_ARGUMENT;
  if (count == 0) return TTGPU_OK;
  uint32_t *d = nullptr;
  try {
    Check(hipMalloc(&d, (size_t)count * 4), "hipMalloc");
    LaunchPcg32(initstate, initseq, count, d, nullptr);
    Check(hipGetLastError(), "launch");
    Check(hipDeviceSynchronize(), "sync");
    Check(hipMemcpy(out, d, (size_t)count * 4, hipMemcpyDeviceToHost), "D2H");
  } catch (const std::exception &e) {
    g_create_error = e.what();
    if (d) (void)hipFree(d);
    return TTGPU_ERR_DEVICE;
  }
  (void)hipFree(d);
  return TTGPU_OK;
}

}  // extern "C"

static nn::NeuralGuideConfig NnConfig(const ttgpu_nn_config &c) {
  nn::NeuralGuideConfig k;
  k.levels = c.levels;
  k.log2_table = c.log2_table;
  k.base_res = c.base_res;
  k.max_res = c.max_res;
  k.batch = c.batch;
  k.lr = c.lr;
  return k;
}

int64_t ttgpu_nn_param_count(const ttgpu_nn_config *cfg) {
  if (!cfg || cfg->levels < 1 || cfg->levels > nn::kMaxLevels || cfg->log2_table < 4 || cfg->log2_table > 24) return -1;
  return nn::make_layout(cfg->levels, cfg->log2_table).total;
}

namespace {
struct DevBuf {
  void *p = nullptr;
  explicit DevBuf(size_t bytes) { Check(hipMalloc(&p, std::max<size_t>(bytes, 16)), "hipMalloc"); }
  ~DevBuf() { (void)hipFree(p); }
  template <class T> T *as() { return (T *)p; }
};
// n x 3 floats (and an optional n-vector in w) -> device float4 array.
void UploadF4(DevBuf &b, int64_t n, const float *xyz, const float *w) {
  std::vector<float4> v(n);
  for (int64_t i = 0; i < n; ++i) v[i] = make_float4(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], w ? w[i] : 0.f);
  if (n) Check(hipMemcpy(b.p, v.data(), n * sizeof(float4), hipMemcpyHostToDevice), "upload");
}
}  // namespace

extern "C" {

int ttgpu_nn_init_params(const ttgpu_nn_config *cfg, float *params) {
  if (!cfg || !params) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    nn::NeuralGuide g(NnConfig(*cfg), cfg->bb_lo, cfg->bb_hi, cfg->seed);
    g.GetParams(params);
    return TTGPU_OK;
  })
}

int ttgpu_nn_forward(const ttgpu_nn_config *cfg, const float *params, int64_t n, const float *pos, const float *nrm,
                     const float *wo, float *out) {
  if (!cfg || !params || n < 0 || (n > 0 && (!pos || !nrm || !wo || !out))) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    nn::NeuralGuide g(NnConfig(*cfg), cfg->bb_lo, cfg->bb_hi, cfg->seed);
    g.SetParams(params);
    DevBuf dp(n * sizeof(float4)), dn(n * sizeof(float4)), dw(n * sizeof(float4)), dout(n * nn::kOut * sizeof(float));
    UploadF4(dp, n, pos, nullptr);
    UploadF4(dn, n, nrm, nullptr);
    UploadF4(dw, n, wo, nullptr);
    g.Forward(dp.as<float4>(), dn.as<float4>(), dw.as<float4>(), nullptr, n, dout.as<float>(), false, 0);
    Check(hipDeviceSynchronize(), "sync");
    if (n) Check(hipMemcpy(out, dout.p, n * nn::kOut * sizeof(float), hipMemcpyDeviceToHost), "download");
    return TTGPU_OK;
  })
}

int ttgpu_nn_gradient(const ttgpu_nn_config *cfg, const float *params, int64_t n, const float *pos, const float *nrm,
                      const float *wo, const float *wi, const float *weight, float *grad, float *loss) {
  if (!cfg || !params || n <= 0 || !pos || !nrm || !wo || !wi || !weight || !grad || n > cfg->batch)
    return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    nn::NeuralGuide g(NnConfig(*cfg), cfg->bb_lo, cfg->bb_hi, cfg->seed);
    g.SetParams(params);
    DevBuf dp(n * sizeof(float4)), dn(n * sizeof(float4)), dw(n * sizeof(float4)), dd(n * sizeof(float4));
    UploadF4(dp, n, pos, nullptr);
    UploadF4(dn, n, nrm, nullptr);
    UploadF4(dw, n, wo, nullptr);
    UploadF4(dd, n, wi, weight);
    g.ZeroGradient(0);
    g.Step(dp.as<float4>(), dd.as<float4>(), dn.as<float4>(), dw.as<float4>(), nullptr, n, nullptr, 0, false, 0);
    Check(hipDeviceSynchronize(), "sync");
    g.Gradient(grad);
    if (loss) *loss = g.LastLoss();
    return TTGPU_OK;
  })
}

int ttgpu_nn_train(const ttgpu_nn_config *cfg, float *params, int64_t n, const float *pos, const float *nrm, const float *wo,
                   const float *wi, const float *weight, int32_t passes, float *loss_per_pass) {
  if (!cfg || !params || n <= 0 || !pos || !nrm || !wo || !wi || !weight || passes < 0) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    nn::NeuralGuide g(NnConfig(*cfg), cfg->bb_lo, cfg->bb_hi, cfg->seed);
    g.SetParams(params);
    DevBuf dp(n * sizeof(float4)), dn(n * sizeof(float4)), dw(n * sizeof(float4)), dd(n * sizeof(float4));
    std::vector<float> w(weight, weight + n);
    UploadF4(dp, n, pos, w.data());
    UploadF4(dn, n, nrm, nullptr);
    UploadF4(dw, n, wo, nullptr);
    UploadF4(dd, n, wi, w.data());
    for (int k = 0; k < passes; ++k) {
      g.TrainOnRecords(dp.as<float4>(), dd.as<float4>(), dn.as<float4>(), dw.as<float4>(), n, 0);
      Check(hipDeviceSynchronize(), "sync");
      if (loss_per_pass) loss_per_pass[k] = g.LastLoss() / (float)std::max<int64_t>(1, (n + cfg->batch - 1) / cfg->batch);
    }
    g.GetParams(params);
    return TTGPU_OK;
  })
}

int ttgpu_guide_info(ttgpu_handle *h, int32_t *cells, int32_t *rounds, int64_t *records_last_pass, int64_t *records_dropped) {
  if (!h) return TTGPU_ERR_INVALID_ARGUMENT;
  if (!h->guided) return Fail(h, TTGPU_ERR_INVALID_ARGUMENT, "not a guided (TTGPU_ALGO_PTG) handle");
  if (cells) *cells = h->learned ? 0 : (int32_t)h->recorder->cells().size();
  if (rounds) *rounds = h->train_rounds;
  if (records_last_pass) *records_last_pass = h->records_last_pass;
  if (records_dropped) *records_dropped = h->records_dropped;
  return TTGPU_OK;
}

namespace {
// Device scratch of `count` floats per column, freed on scope exit.
struct DeviceFloats {
  std::vector<float *> p;
  ~DeviceFloats() {
    for (float *x : p)
      if (x) (void)hipFree(x);
  }
  float *Get(size_t n) {
    float *x = nullptr;
    Check(hipMalloc(&x, std::max<size_t>(1, n) * sizeof(float)), "hipMalloc");
    p.push_back(x);
    return x;
  }
};
}  // namespace

int ttgpu_guide_pdf(ttgpu_handle *h, int64_t count, const float *pos, const float *dirs, int32_t on_device, float *out_pdf) {
  if (!h || count < 0 || (count > 0 && (!pos || !dirs || !out_pdf))) return TTGPU_ERR_INVALID_ARGUMENT;
  if (!h->guided || h->learned)
    return Fail(h, TTGPU_ERR_INVALID_ARGUMENT, "not a vMF-tree or quadtree guided handle");
  TTGPU_GUARD(h, {
    if (on_device) {
      if (count == 0) return TTGPU_OK;
      DeviceFloats f;
      float *dp = f.Get(3 * count), *dd = f.Get(3 * count), *out = f.Get(count);
      Check(hipMemcpy(dp, pos, 3 * count * sizeof(float), hipMemcpyHostToDevice), "upload");
      Check(hipMemcpy(dd, dirs, 3 * count * sizeof(float), hipMemcpyHostToDevice), "upload");
      LaunchGuidePdfAt(h->dsc, count, dp, dd, out, h->stream);
      Check(hipGetLastError(), "launch");
      Check(hipStreamSynchronize(h->stream), "sync");
      Check(hipMemcpy(out_pdf, out, count * sizeof(float), hipMemcpyDeviceToHost), "download");
      return TTGPU_OK;
    }
    const guide::Recorder &rec = *h->recorder;
    for (int64_t i = 0; i < count; ++i) {
      const double p[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
      const guide::CellData &c = rec.cells()[rec.tree().Lookup(p)];
      out_pdf[i] = rec.quadtree() ? (float)c.qcurrent.Pdf(dirs + 3 * i) : guide::Pdf(c.current, dirs + 3 * i);
    }
    return TTGPU_OK;
  })
}

static void ToVmf(const ttgpu_vmf8 &a, guide::Vmf &m) {
  for (int k = 0; k < guide::kLobes; ++k) {
    for (int c = 0; c < 3; ++c) m.mu[k][c] = a.mu[k][c];
    m.kappa[k] = a.kappa[k];
    m.w[k] = a.w[k];
  }
}
static void FromVmf(const guide::Vmf &m, ttgpu_vmf8 &a) {
  for (int k = 0; k < guide::kLobes; ++k) {
    for (int c = 0; c < 3; ++c) a.mu[k][c] = m.mu[k][c];
    a.kappa[k] = m.kappa[k];
    a.w[k] = m.w[k];
  }
}

int ttgpu_guide_init_vmf(ttgpu_vmf8 *out) {
  if (!out) return TTGPU_ERR_INVALID_ARGUMENT;
  guide::Vmf m;
  guide::InitUnitSphere(m);
  FromVmf(m, *out);
  return TTGPU_OK;
}

int ttgpu_guide_fit_vmf(ttgpu_vmf8 *mix, const float *dirs, const float *weights, int64_t n, int64_t max_num_samples) {
  if (!mix || (n > 0 && (!dirs || !weights)) || n < 0) return TTGPU_ERR_INVALID_ARGUMENT;
  guide::Vmf m, prior;
  ToVmf(*mix, m);
  guide::InitUnitSphere(prior);
  guide::FitParams p;
  const double strength = std::max(1., 0.01 * (double)max_num_samples);
  p.prior_alpha = p.prior_nu = p.prior_tau = (float)strength;
  p.m_step_every = std::max(1, (int)strength * 10);
  p.prior = &prior;
  guide::FitData d;
  for (int64_t i = 0; i < n; ++i)
    if (weights[i] > 0.f) guide::FitSample(m, d, p, dirs + 3 * i, weights[i]);
  FromVmf(m, *mix);
  return TTGPU_OK;
}

namespace {
DevVmfPrior DevPrior() {
  guide::Vmf p;
  guide::InitUnitSphere(p);
  DevVmfPrior d;
  for (int k = 0; k < kFitLobes; ++k) {
    for (int a = 0; a < 3; ++a) d.mu[k][a] = p.mu[k][a];
    d.kappa[k] = p.kappa[k];
    d.w[k] = p.w[k];
  }
  return d;
}

// One cell's samples (direction, weight, original flag) in their order as device entries.
struct OneCellEntries {
  DevBuffer<float4> pos_w, dir;
  DevBuffer<uint32_t> order, begin, end;
  OneCellEntries(const float *dirs, const float *weights, const uint8_t *original, int64_t n, const float *pos = nullptr)
      : pos_w(n), dir(n), order(n), begin(1), end(1) {
    std::vector<float4> pw(n), dr(n);
    std::vector<uint32_t> ord(n);
    for (int64_t i = 0; i < n; ++i) {
      pw[i] = pos ? make_float4(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], weights[i]) : make_float4(0.f, 0.f, 0.f, weights[i]);
      dr[i] = dirs ? make_float4(dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2], original && original[i] ? 1.f : 0.f)
                   : make_float4(0.f, 0.f, 1.f, original && original[i] ? 1.f : 0.f);
      ord[i] = (uint32_t)i;
    }
    const uint32_t b = 0, e = (uint32_t)n;
    Check(hipMemcpy(pos_w.p, pw.data(), n * sizeof(float4), hipMemcpyHostToDevice), "upload");
    Check(hipMemcpy(dir.p, dr.data(), n * sizeof(float4), hipMemcpyHostToDevice), "upload");
    Check(hipMemcpy(order.p, ord.data(), n * sizeof(uint32_t), hipMemcpyHostToDevice), "upload");
    Check(hipMemcpy(begin.p, &b, sizeof(b), hipMemcpyHostToDevice), "upload");
    Check(hipMemcpy(end.p, &e, sizeof(e), hipMemcpyHostToDevice), "upload");
  }
  void Into(GuideFitBuffers &f) const {
    f.ent_pos_w = pos_w.p;
    f.ent_dir = dir.p;
    f.vals_out = order.p;
    f.cell_begin = begin.p;
    f.cell_end = end.p;
    f.num_cells = 1;
  }
};
}  // namespace

int ttgpu_guide_fit_vmf_gpu(ttgpu_vmf8 *mix, const float *dirs, const float *weights, int64_t n, int64_t max_num_samples) {
  if (!mix || (n > 0 && (!dirs || !weights)) || n < 0 || n > ((int64_t)1 << 31)) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    DevFitCell c;
    std::memset(&c, 0, sizeof(c));
    for (int k = 0; k < kFitLobes; ++k) {
      for (int a = 0; a < 3; ++a) c.mu[k][a] = mix->mu[k][a];
      c.kappa[k] = mix->kappa[k];
      c.w[k] = mix->w[k];
    }
    const double strength = std::max(1., 0.01 * (double)max_num_samples);
    c.prior_strength = (float)strength;
    c.m_step_every = std::max(1, (int)strength * 10);
    OneCellEntries ent(dirs, weights, nullptr, n);
    DevBuffer<DevFitCell> cell(1);
    Check(hipMemcpy(cell.p, &c, sizeof(c), hipMemcpyHostToDevice), "upload");
    GuideFitBuffers f{};
    ent.Into(f);
    f.cells = cell.p;
    LaunchFitOneCell(f, false, DevPrior(), 0.f, nullptr);
    Check(hipGetLastError(), "launch");
    Check(hipDeviceSynchronize(), "sync");
    Check(hipMemcpy(&c, cell.p, sizeof(c), hipMemcpyDeviceToHost), "download");
    for (int k = 0; k < kFitLobes; ++k) {
      for (int a = 0; a < 3; ++a) mix->mu[k][a] = c.mu[k][a];
      mix->kappa[k] = c.kappa[k];
      mix->w[k] = c.w[k];
    }
    return TTGPU_OK;
  })
}

int ttgpu_guide_leaf_stats_gpu(const float *pts, int64_t n, int64_t *count, double mean[3], double cov[9]) {
  if (!count || !mean || !cov || n < 0 || n > ((int64_t)1 << 31) || (n > 0 && !pts)) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    // Zero weights: no EM, only the leaf statistics of the (original) records.
    std::vector<float> w(n, 0.f);
    std::vector<uint8_t> orig(n, 1);
    OneCellEntries ent(nullptr, w.data(), orig.data(), n, pts);
    DevFitCell c;
    std::memset(&c, 0, sizeof(c));
    c.m_step_every = 1;
    DevBuffer<DevFitCell> cell(1);
    Check(hipMemcpy(cell.p, &c, sizeof(c), hipMemcpyHostToDevice), "upload");
    GuideFitBuffers f{};
    ent.Into(f);
    f.cells = cell.p;
    LaunchFitOneCell(f, false, DevPrior(), 0.f, nullptr);
    Check(hipGetLastError(), "launch");
    Check(hipDeviceSynchronize(), "sync");
    Check(hipMemcpy(&c, cell.p, sizeof(c), hipMemcpyDeviceToHost), "download");
    *count = c.ln;
    for (int a = 0; a < 3; ++a) {
      mean[a] = c.lmean[a];
      for (int b = 0; b < 3; ++b) cov[3 * a + b] = c.ln > 1 ? c.lc[a][b] / (double)(c.ln - 1) : 0.;
    }
    return TTGPU_OK;
  })
}

int ttgpu_guide_build_kdtree(const double *pts, int64_t n, int32_t min_points, int32_t max_depth, int32_t *leaf_of_point,
                             int32_t *num_leafs) {
  if ((n > 0 && (!pts || !leaf_of_point)) || n < 0 || min_points < 1 || max_depth < 1 || !num_leafs)
    return TTGPU_ERR_INVALID_ARGUMENT;
  std::vector<std::array<double, 3>> p(n);
  for (int64_t i = 0; i < n; ++i) p[i] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
  std::vector<int> order;
  std::vector<std::pair<int, int>> ranges;
  guide::KdTree t = guide::BuildTree(p, min_points, max_depth, order, ranges);
  for (size_t l = 0; l < ranges.size(); ++l)
    for (int k = ranges[l].first; k < ranges[l].second; ++k) leaf_of_point[order[k]] = (int32_t)l;
  *num_leafs = t.num_leafs;
  return TTGPU_OK;
}

static GuideCell BakeCell(const ttgpu_vmf8 &m) {
  GuideCell c;
  double acc = 0.;
  for (int k = 0; k < kGuideLobes; ++k) {
    c.lobe[k] = make_float4(m.mu[k][0], m.mu[k][1], m.mu[k][2], m.kappa[k]);
    c.wn[k] = (float)(m.w[k] * (double)m.kappa[k] / (2. * kPiD * -std::expm1(-2. * (double)m.kappa[k])));
    acc += m.w[k];
    c.cdf[k] = (float)acc;
  }
  c.cdf[kGuideLobes - 1] = 2.f;
  return c;
}

int ttgpu_guide_sample_vmf(const ttgpu_vmf8 *m, uint64_t seed, int64_t count, float *out_dir, float *out_pdf) {
  if (!m || count < 0 || (count > 0 && (!out_dir || !out_pdf))) return TTGPU_ERR_INVALID_ARGUMENT;
  const GuideCell c = BakeCell(*m);
  if (count == 0) return TTGPU_OK;
  float *dd = nullptr, *dp = nullptr;
  if (hipMalloc(&dd, count * 3 * sizeof(float)) != hipSuccess) return TTGPU_ERR_DEVICE;
  if (hipMalloc(&dp, count * sizeof(float)) != hipSuccess) {
    (void)hipFree(dd);
    return TTGPU_ERR_DEVICE;
  }
  int rc = TTGPU_OK;
  LaunchGuideSample(c, seed, count, dd, dp, 0);
  if (hipDeviceSynchronize() != hipSuccess || hipGetLastError() != hipSuccess) rc = TTGPU_ERR_DEVICE;
  if (rc == TTGPU_OK && (hipMemcpy(out_dir, dd, count * 3 * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess ||
                         hipMemcpy(out_pdf, dp, count * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess))
    rc = TTGPU_ERR_DEVICE;
  (void)hipFree(dd);
  (void)hipFree(dp);
  return rc;
}

int ttgpu_guide_pdf_vmf(const ttgpu_vmf8 *m, int64_t count, const float *dirs, float *out_pdf) {
  if (!m || count < 0 || (count > 0 && (!dirs || !out_pdf))) return TTGPU_ERR_INVALID_ARGUMENT;
  const GuideCell c = BakeCell(*m);
  float *dd = nullptr, *dp = nullptr;
  if (count == 0) return TTGPU_OK;
  if (hipMalloc(&dd, count * 3 * sizeof(float)) != hipSuccess) return TTGPU_ERR_DEVICE;
  if (hipMalloc(&dp, count * sizeof(float)) != hipSuccess) {
    (void)hipFree(dd);
    return TTGPU_ERR_DEVICE;
  }
  int rc = TTGPU_OK;
  if (hipMemcpy(dd, dirs, count * 3 * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) rc = TTGPU_ERR_DEVICE;
  if (rc == TTGPU_OK) {
    LaunchGuidePdf(c, count, dd, dp, 0);
    if (hipDeviceSynchronize() != hipSuccess || hipGetLastError() != hipSuccess) rc = TTGPU_ERR_DEVICE;
  }
  if (rc == TTGPU_OK && hipMemcpy(out_pdf, dp, count * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) rc = TTGPU_ERR_DEVICE;
  (void)hipFree(dd);
  (void)hipFree(dp);
  return rc;
}


// ---- quadtree guide building blocks --------------------------------------------------------

static void TreeFromArrays(const int32_t *children, int32_t num_nodes, guide::quad::Tree &t) {
  if (!children || num_nodes <= 0 || num_nodes > guide::quad::kMaxNodes) throw std::invalid_argument("bad quadtree");
  t.child.assign(num_nodes, {-1, -1, -1, -1});
  t.root = 0;
  for (int32_t n = 0; n < num_nodes; ++n) {
    const int32_t *c = children + 4 * (size_t)n;
    const bool leaf = c[0] < 0;
    for (int k = 0; k < 4; ++k) {
      if ((c[k] < 0) != leaf) throw std::invalid_argument("quadtree node with some but not all children");
      if (!leaf && (c[k] <= n || c[k] >= num_nodes)) throw std::invalid_argument("quadtree children must follow their parent (pre-order)");
      t.child[n][k] = c[k];
    }
  }
  // Every node but the root has exactly one parent, and descents are at most 8 levels deep.
  std::vector<int> parents(num_nodes, 0), depth(num_nodes, 0);
  for (int32_t n = 0; n < num_nodes; ++n)
    if (!t.IsLeaf(n))
      for (int k = 0; k < 4; ++k) {
        ++parents[t.child[n][k]];
        depth[t.child[n][k]] = depth[n] + 1;
      }
  for (int32_t n = 1; n < num_nodes; ++n)
    if (parents[n] != 1) throw std::invalid_argument("quadtree node without exactly one parent");
  for (int32_t n = 0; n < num_nodes; ++n)
    if (depth[n] >= guide::quad::kMaxDepth) throw std::invalid_argument("quadtree deeper than 8 levels");
}

static void TreeToArrays(const guide::quad::Tree &t, int32_t *children) {
  for (int n = 0; n < t.NumNodes(); ++n)
    for (int k = 0; k < 4; ++k) children[4 * (size_t)n + k] = t.child[n][k];
}

namespace {
// Device copy of one quadtree for the sampling and pdf entry points.
struct DeviceQuad {
  QuadNode *nodes = nullptr;
  QuadCell cell{-1, 1.f};
  ~DeviceQuad() {
    if (nodes) (void)hipFree(nodes);
  }
};
void UploadQuad(const int32_t *children, const float *probs, int32_t num_nodes, DeviceQuad &d) {
  guide::quad::Tree t;
  TreeFromArrays(children, num_nodes, t);
  if (!probs) throw std::invalid_argument("null weights");
  std::vector<float> w(probs, probs + num_nodes);
  std::vector<QuadNode> nodes;
  std::vector<int> dev;
  d.cell = FlattenQuad(t, w, nodes, dev);
  nodes.resize(std::max<size_t>(1, nodes.size()));
  Check(hipMalloc(&d.nodes, nodes.size() * sizeof(QuadNode)), "hipMalloc");
  Check(hipMemcpy(d.nodes, nodes.data(), nodes.size() * sizeof(QuadNode), hipMemcpyHostToDevice), "upload");
}
}  // namespace

int ttgpu_quadtree_build(const float *uv, const float *weights, int64_t n, float fraction, int32_t capacity,
                         int32_t *children, float *node_weights, int32_t *num_nodes) {
  if (n < 0 || (n > 0 && (!uv || !weights)) || !children || !node_weights || !num_nodes) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    std::vector<guide::quad::Point> pts(n);
    std::vector<float> w(weights, weights + n), nw;
    for (int64_t i = 0; i < n; ++i) pts[i] = {uv[2 * i], uv[2 * i + 1]};
    const guide::quad::Tree t = guide::quad::Build(pts, w, fraction, nw);
    *num_nodes = t.NumNodes();
    if (t.NumNodes() > capacity) return Fail(nullptr, TTGPU_ERR_INVALID_ARGUMENT, "quadtree capacity too small");
    TreeToArrays(t, children);
    std::copy(nw.begin(), nw.end(), node_weights);
    return TTGPU_OK;
  })
}

int ttgpu_quadtree_adapt(const int32_t *children, const float *weights, int32_t num_nodes, float fraction, int32_t capacity,
                         int32_t *out_children, float *out_weights, int32_t *out_old_index, float *out_fraction,
                         int32_t *out_num_nodes) {
  if (!weights || !out_children || !out_weights || !out_old_index || !out_fraction || !out_num_nodes)
    return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    guide::quad::Tree t;
    TreeFromArrays(children, num_nodes, t);
    std::vector<float> w(weights, weights + num_nodes), nw;
    std::vector<guide::quad::NewToOld> map;
    const guide::quad::Tree nt = guide::quad::Adapt(t, w, fraction, nw, map);
    *out_num_nodes = nt.NumNodes();
    if (nt.NumNodes() > capacity) return Fail(nullptr, TTGPU_ERR_INVALID_ARGUMENT, "quadtree capacity too small");
    TreeToArrays(nt, out_children);
    for (int i = 0; i < nt.NumNodes(); ++i) {
      out_weights[i] = nw[i];
      out_old_index[i] = map[i].idx;
      out_fraction[i] = map[i].fractional_size;
    }
    return TTGPU_OK;
  })
}


int ttgpu_quadtree_sample(const int32_t *children, const float *probs, int32_t num_nodes, int64_t count, const float *u,
                          float *out_uv, float *out_dir, float *out_pdf) {
  if (count < 0 || (count > 0 && (!u || !out_uv || !out_dir || !out_pdf))) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    DeviceQuad q;
    UploadQuad(children, probs, num_nodes, q);
    if (count == 0) return TTGPU_OK;
    DeviceFloats f;
    float *du = f.Get(2 * count), *duv = f.Get(2 * count), *dd = f.Get(3 * count), *dp = f.Get(count);
    Check(hipMemcpy(du, u, 2 * count * sizeof(float), hipMemcpyHostToDevice), "upload");
    LaunchQuadSample(q.nodes, q.cell.root, q.cell.w_root, count, du, duv, dd, dp, 0);
    Check(hipGetLastError(), "launch");
    Check(hipDeviceSynchronize(), "sync");
    Check(hipMemcpy(out_uv, duv, 2 * count * sizeof(float), hipMemcpyDeviceToHost), "download");
    Check(hipMemcpy(out_dir, dd, 3 * count * sizeof(float), hipMemcpyDeviceToHost), "download");
    Check(hipMemcpy(out_pdf, dp, count * sizeof(float), hipMemcpyDeviceToHost), "download");
    return TTGPU_OK;
  })
}

int ttgpu_quadtree_pdf(const int32_t *children, const float *probs, int32_t num_nodes, int64_t count, const float *dirs,
                       float *out_pdf) {
  if (count < 0 || (count > 0 && (!dirs || !out_pdf))) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    DeviceQuad q;
    UploadQuad(children, probs, num_nodes, q);
    if (count == 0) return TTGPU_OK;
    DeviceFloats f;
    float *dd = f.Get(3 * count), *dp = f.Get(count);
    Check(hipMemcpy(dd, dirs, 3 * count * sizeof(float), hipMemcpyHostToDevice), "upload");
    LaunchQuadPdf(q.nodes, q.cell.root, q.cell.w_root, count, dd, dp, 0);
    Check(hipGetLastError(), "launch");
    Check(hipDeviceSynchronize(), "sync");
    Check(hipMemcpy(out_pdf, dp, count * sizeof(float), hipMemcpyDeviceToHost), "download");
    return TTGPU_OK;
  })
}

struct ttgpu_qmodel {
  guide::quad::Learned learned;
  guide::quad::Sampled sampled;
};

ttgpu_qmodel *ttgpu_qmodel_create(void) {
  try {
    return new ttgpu_qmodel();
  } catch (...) {
    return nullptr;
  }
}

void ttgpu_qmodel_free(ttgpu_qmodel *m) { delete m; }

static std::vector<guide::quad::Sample1> QSamples(const float *dirs, const float *weights, const uint8_t *original, int64_t n) {
  if (n < 0 || (n > 0 && (!dirs || !weights))) throw std::invalid_argument("bad sample arrays");
  std::vector<guide::quad::Sample1> s(n);
  for (int64_t i = 0; i < n; ++i) s[i] = {dirs + 3 * i, weights[i], original ? original[i] != 0 : true};
  return s;
}

int ttgpu_qmodel_initial_fit(ttgpu_qmodel *m, const float *dirs, const float *weights, int64_t n) {
  if (!m) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    m->learned.InitialFit(QSamples(dirs, weights, nullptr, n));
    return TTGPU_OK;
  })
}

int ttgpu_qmodel_bake(ttgpu_qmodel *m) {
  if (!m) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    m->sampled = m->learned.Bake();
    return TTGPU_OK;
  })
}

int ttgpu_qmodel_incremental_fit(ttgpu_qmodel *m, const float *dirs, const float *weights, const uint8_t *original, int64_t n,
                                 int32_t round) {
  if (!m) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    m->learned.IncrementalFit(QSamples(dirs, weights, original, n), round, m->sampled);
    return TTGPU_OK;
  })
}

int ttgpu_qmodel_incremental_fit_gpu(ttgpu_qmodel *m, const float *dirs, const float *weights, const uint8_t *original, int64_t n,
                                     int32_t round) {
  if (!m || round < 1 || n < 0 || n > ((int64_t)1 << 31) || (n > 0 && (!dirs || !weights))) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    const auto &t = m->learned.tree;
    const int nn = t.NumNodes();
    if ((int)m->sampled.prior.size() != nn || m->sampled.tree.NumNodes() != nn)
      throw std::logic_error("quadtree incremental fit: sampled and learned trees differ");
    // The tree as device branches and its nodes as slots (root: slot 0; child k of branch b:
    // slot 1 + 4 b + k), with the learned statistics and the sampled priors and weights.
    std::vector<QuadNode> qn;
    std::vector<int> dev;
    std::vector<float> w = m->sampled.probs;
    w.resize(nn, 0.f);
    const QuadCell hdr = FlattenQuad(t, w, qn, dev);
    const int B = (int)qn.size();
    std::vector<int> slot(nn, -1);
    slot[t.root] = 0;
    for (int k = 0; k < nn; ++k)
      if (!t.IsLeaf(k))
        for (int c = 0; c < 4; ++c) slot[t.child[k][c]] = 1 + 4 * dev[k] + c;
    std::vector<DevQuadSlot> sl(1 + 4 * (size_t)B);
    std::memset(sl.data(), 0, sl.size() * sizeof(DevQuadSlot));
    for (int k = 0; k < nn; ++k) {
      DevQuadSlot &x = sl[slot[k]];
      x.n = (unsigned long long)m->learned.stats.n[k];
      x.mean = m->learned.stats.mean[k];
      x.m2 = m->learned.stats.m2[k];
      x.prior = m->sampled.prior[k];
    }
    const int fit_root = dev[t.root], branch_end = B;
    DevBuffer<QuadNode> d_nodes(std::max(1, B));
    DevBuffer<QuadCell> d_cell(1);
    DevBuffer<DevQuadSlot> d_slots(sl.size());
    DevBuffer<int> d_root(1), d_end(1);
    DevBuffer<DevFitCell> d_fc(1);
    DevFitCell fc;
    std::memset(&fc, 0, sizeof(fc));
    if (B) Check(hipMemcpy(d_nodes.p, qn.data(), B * sizeof(QuadNode), hipMemcpyHostToDevice), "upload");
    Check(hipMemcpy(d_cell.p, &hdr, sizeof(hdr), hipMemcpyHostToDevice), "upload");
    Check(hipMemcpy(d_slots.p, sl.data(), sl.size() * sizeof(DevQuadSlot), hipMemcpyHostToDevice), "upload");
    Check(hipMemcpy(d_root.p, &fit_root, sizeof(int), hipMemcpyHostToDevice), "upload");
    Check(hipMemcpy(d_end.p, &branch_end, sizeof(int), hipMemcpyHostToDevice), "upload");
    Check(hipMemcpy(d_fc.p, &fc, sizeof(fc), hipMemcpyHostToDevice), "upload");
    OneCellEntries ent(dirs, weights, original, n);
    GuideFitBuffers f{};
    ent.Into(f);
    f.cells = d_fc.p;
    f.qfit_root = d_root.p;
    f.qbranch_end = d_end.p;
    f.qslots = d_slots.p;
    f.qcells = d_cell.p;
    f.qnodes = d_nodes.p;
    LaunchFitOneCell(f, true, DevPrior(), (float)std::log((double)round), nullptr);
    Check(hipGetLastError(), "launch");
    Check(hipDeviceSynchronize(), "sync");
    Check(hipMemcpy(sl.data(), d_slots.p, sl.size() * sizeof(DevQuadSlot), hipMemcpyDeviceToHost), "download");
    if (B) Check(hipMemcpy(qn.data(), d_nodes.p, B * sizeof(QuadNode), hipMemcpyDeviceToHost), "download");
    for (int k = 0; k < nn; ++k) {
      const DevQuadSlot &x = sl[slot[k]];
      m->learned.stats.n[k] = (int64_t)x.n;
      m->learned.stats.mean[k] = x.mean;
      m->learned.stats.m2[k] = x.m2;
    }
    const auto &st = m->learned.stats;
    if (st.n[t.root] > 0 && t.IsLeaf(t.root)) {
      m->sampled.probs.resize(nn);
      m->sampled.probs[t.root] = QuadLeafWeight(m->sampled.prior[t.root], st.n[t.root], st.mean[t.root], st.m2[t.root],
                                                (double)st.n[t.root], st.mean[t.root], std::log((double)round));
    }
    if (st.n[t.root] > 0 && !t.IsLeaf(t.root)) {
      m->sampled.probs.resize(nn);
      for (int k = 0; k < nn; ++k) {
        if (t.IsLeaf(k)) continue;
        const float4 q = qn[dev[k]].w;
        const float w4[4] = {q.x, q.y, q.z, q.w};
        for (int c = 0; c < 4; ++c) m->sampled.probs[t.child[k][c]] = w4[c];
        m->sampled.probs[k] = w4[0] + w4[1] + w4[2] + w4[3];
      }
    }
    return TTGPU_OK;
  })
}

int ttgpu_qmodel_update_and_bake(ttgpu_qmodel *m) {
  if (!m) return TTGPU_ERR_INVALID_ARGUMENT;
  TTGPU_GUARD(nullptr, {
    m->sampled = m->learned.IterationUpdateAndBake(m->sampled);
    return TTGPU_OK;
  })
}

int ttgpu_qmodel_num_nodes(const ttgpu_qmodel *m, int32_t which, int32_t *out) {
  if (!m || !out || (which != 0 && which != 1)) return TTGPU_ERR_INVALID_ARGUMENT;
  *out = which == 0 ? m->learned.tree.NumNodes() : m->sampled.tree.NumNodes();
  return TTGPU_OK;
}

int ttgpu_qmodel_get_learned(const ttgpu_qmodel *m, int32_t *children, int64_t *counts, double *means, double *m2) {
  if (!m || !children || !counts || !means || !m2) return TTGPU_ERR_INVALID_ARGUMENT;
  const auto &l = m->learned;
  TreeToArrays(l.tree, children);
  for (int i = 0; i < l.tree.NumNodes(); ++i) {
    counts[i] = l.stats.n[i];
    means[i] = l.stats.mean[i];
    m2[i] = l.stats.m2[i];
  }
  return TTGPU_OK;
}

int ttgpu_qmodel_get_sampled(const ttgpu_qmodel *m, int32_t *children, double *means, double *stddev, float *probs,
                             float *prior) {
  if (!m || !children || !means || !stddev || !probs || !prior) return TTGPU_ERR_INVALID_ARGUMENT;
  const auto &d = m->sampled;
  TreeToArrays(d.tree, children);
  for (int i = 0; i < d.tree.NumNodes(); ++i) {
    means[i] = d.means[i];
    stddev[i] = d.stddev[i];
    probs[i] = d.probs[i];
    prior[i] = d.prior[i];
  }
  return TTGPU_OK;
}

int ttgpu_qmodel_filter_direction(const ttgpu_qmodel *m, const float *dir, double u0, double u1, float *out) {
  if (!m || !dir || !out) return TTGPU_ERR_INVALID_ARGUMENT;
  m->sampled.FilterDirection(dir, u0, u1, out);
  return TTGPU_OK;
}

}  // extern "C"
