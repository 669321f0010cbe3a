// Wavefront kernels of the MI355X path tracer (pt2 semantics).
//
// One bounce of every path in flight is:  trace (closest hit)  ->  shade
// (emission with MIS, next-event estimation, BSDF sampling)  ->  shadow (any
// hit of the compacted NEE rays, accumulate).  Path state is structure-of-
// arrays in HBM; queues are compacted with wave-level ballot + one atomic per
// wave.  The reference's per-path loop is
// src/renderingalgorithms_pathtracing2.cxx:338-443.
#include <hip/hip_runtime.h>
#include <hipcub/device/device_radix_sort.hpp>

#include <stdexcept>
#include <string>

// Traversal stack overflow flag (see trace.hpp): raised by any traversal in this module's
// kernels, read and cleared by the host after every pass and query.
__device__ unsigned int g_stack_overflow;
#if defined(__HIP_DEVICE_COMPILE__)
#define TTGPU_STACK_OVERFLOW() atomicOr(&g_stack_overflow, 1u)
#endif

#include "device_math.hpp"
#include "shading.hpp"
#include "trace.hpp"
#include "media.hpp"
#include "guide_vmf.hpp"
#include "guide_quad.hpp"
#include "nn_device.hpp"
#include "kernels.hpp"

// Minimum waves per SIMD asked of the register allocator for the shade and traversal kernels.
#ifndef TTGPU_SHADE_WAVES
#define TTGPU_SHADE_WAVES 1
#endif
#ifndef TTGPU_TRACE_WAVES
#define TTGPU_TRACE_WAVES 1
#endif

namespace ttgpu {

// ---- wave-aggregated queue append ----------------------------------------
__device__ __forceinline__ uint32_t wave_append(uint32_t *counter, bool pred) {
  const uint64_t mask = __ballot(pred);
  const uint64_t active = __ballot(1);
  const int lane = __lane_id();
  const int leader = __ffsll((unsigned long long)active) - 1;
  uint32_t base = 0;
  if (lane == leader && mask) base = atomicAdd(counter, (uint32_t)__popcll(mask));
  base = __shfl(base, leader);
  return base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
}

// Adds every lane's count with one atomic per wave (called by whole waves).
__device__ __forceinline__ void wave_stat(uint32_t *counter, uint32_t n) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
  if ((threadIdx.x & 63) == 0 && n) atomicAdd(counter, n);
}

__device__ __forceinline__ uint32_t grid_stride() { return gridDim.x * blockDim.x; }
__device__ __forceinline__ uint32_t gtid() { return blockIdx.x * blockDim.x + threadIdx.x; }

__global__ void k_reset_counter(uint32_t *counters, int which) {
  if (threadIdx.x == 0 && blockIdx.x == 0) counters[which] = 0;
}
__global__ void k_fill_f64(double *p, double *p2, size_t n, double v) {
  for (size_t i = gtid(); i < n; i += grid_stride()) p[i] = p2[i] = v;
}

// ---- camera (src/camera.hxx:105-124, 176-210) ----------------------------
// Pinhole direction pdf over solid angle at image-plane point (x, y): |(x, y, 1)|^3 / pixel area
// (PixelPdfWrtSolidAngle, camera.hxx:88-96).
__device__ __forceinline__ float camera_pdf(const DevCamera &c, float x, float y) {
  const float l = sqrtf(x * x + y * y + 1.f);
  return l * l * l / (c.xper * c.yper);
}

__device__ __forceinline__ bool camera_ray(const DevCamera &c, int px, int py, float r0, float r1, float3 &dir,
                                           float *pdf = nullptr) {
  if (c.kind == TTGPU_CAMERA_PINHOLE) {
    const float x = c.xmin + (r0 + px) * c.xper, y = c.ymin + (r1 + py) * c.yper;
    float3 v = normalize(mk(x, y, 1.f));
    dir = c.right * v.x + c.up * v.y + c.dir * v.z;
    if (pdf) *pdf = camera_pdf(c, x, y);
    return true;
  }
  float u = (r0 + px) * c.fish_delta - 1.f, v = (r1 + py) * c.fish_delta - 1.f;
  float rho = u * u + v * v;
  float3 w = mk(2.f * u, 2.f * v, rho - 1.f) * (1.f / (1.f + rho));
  w.z = -w.z;
  if (rho <= 1.f) {
    dir = c.right * w.x + c.up * w.y + c.dir * w.z;
    return true;
  }
  dir = c.dir;
  return false;
}

// Camera path of (pixel, sample) in path slot i.
// Lambda selection: LambdaSelectionStrategy::WithWeights (src/shader_util.hxx:83-91) with 4 strata.
__device__ __forceinline__ void init_camera_path(const DeviceScene &sc, const PathQueues &q, uint32_t i, uint32_t pixel, uint64_t sample,
                                                 uint32_t npix, uint64_t seed) {
  Pcg rng;
  rng.seed(seed, sample * npix + pixel);
  int main_idx = (int)rng.bounded(kStrata);
  int idx[4] = {main_idx, main_idx + kStrata, main_idx + 2 * kStrata, main_idx + 3 * kStrata};
  int rot = (int)rng.bounded(4);
  int t = idx[0]; idx[0] = idx[rot]; idx[rot] = t;
  const float lambda0 = 370.f + 10.f * idx[0] + 10.f * rng.uniform();
  rng.uniform(); rng.uniform(); rng.uniform();  // the other three jittered wavelengths (unused)
  uint32_t bins = (uint32_t)idx[0] | ((uint32_t)idx[1] << 8) | ((uint32_t)idx[2] << 16) | ((uint32_t)idx[3] << 24);
  const int px = pixel % sc.cam.width, py = pixel / sc.cam.width;
  float r0 = rng.uniform(), r1 = rng.uniform();
  float3 dir;
  float cam_pdf = 0.f;
  bool ok = camera_ray(sc.cam, px, py, r0, r1, dir, &cam_pdf);
  q.org[i] = make_float4(sc.cam.pos.x, sc.cam.pos.y, sc.cam.pos.z, lambda0);
  q.dir[i] = make_float4(dir.x, dir.y, dir.z, 0.f);
  q.thru[i] = ok ? f4((float)kStrata) : f4(0.f);
  q.rad[i] = f4(0.f);
  q.bins[i] = bins;
  q.pixel[i] = pixel;
  q.rng_state[i] = make_uint2((uint32_t)rng.state, (uint32_t)(rng.state >> 32));
  q.rng_inc[i] = make_uint2((uint32_t)rng.inc, (uint32_t)(rng.inc >> 32));
  q.flags[i] = 2u;  // node count 2: camera position and direction nodes (pt2.cxx:388-406)
  q.last_pdf[i] = 0.f;
  if (sc.algo_pt) {
    // pt weighs emission seen by camera rays against light connections to the camera with the
    // camera's direction pdf; the fisheye's direction sample is flagged as a pmf (camera.hxx:191-209).
    q.flags[i] = 2u | kFlagHasLastPdf | (sc.cam.kind == TTGPU_CAMERA_PINHOLE ? 0u : kFlagLastPdfDelta);
    q.last_pdf[i] = cam_pdf;
  }
  q.roughness[i] = 0.f;
  q.tracker[i] = make_uint2((uint32_t)sc.cam_tracker, (uint32_t)(sc.cam_tracker >> 32));
  if (q.wt_r) {
    q.wt_r[i] = f4(1.f);
    q.wt_c[i] = f4(1.f);
  }
}

// The first `count` camera paths of a pass fill slots [0, count): path g is sample
// spp_base + g / npix of pixel g % npix.  Also sets up the pass's counters (which this kernel does
// not read): queue A is 0, 1, .., count - 1.
__global__ void __launch_bounds__(256) k_raygen(DeviceScene sc, PathQueues q, uint32_t count, uint32_t npix, uint32_t spp_base,
                                                uint64_t seed) {
  if (gtid() == 0) {
    q.counters[kCountA] = count;
    q.counters[kCountB] = 0;
    q.counters[kCountShadow] = 0;
    q.counters[kCountShadow2] = 0;
    q.counters[kCountFree] = 0;
    q.counters[kSlotTicket] = 0;
    q.counters[kIdentA] = 1;
    q.counters[kIdentB] = 0;
    if (sc.guide_record) {
      q.counters[kCountRecords] = 0;
      q.counters[kStatRecordsDropped] = 0;
    }
    q.progress[0] = count;
    q.progress[1] = count;
  }
  for (uint32_t i = gtid(); i < count; i += grid_stride()) {
    init_camera_path(sc, q, i, i % npix, (uint64_t)spp_base + i / npix, npix, seed);
    q.queue_a[i] = i;
    if (q.alive) {
      q.alive[i] = 1;
      q.freed[i] = 0;
    }
  }
}

// Waits until this wave's stores have arrived where their scope is coherent, and keeps the compiler
// from moving memory accesses across.  Together with relaxed atomics of that scope it orders two
// accesses without a fence, which would write the whole L2 back (buffer_wbl2): one such fence per
// wave made k_slot_select 74 us instead of 12.
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ void report_progress(PassProgress *host, unsigned long long issued, unsigned long long queued,
                                                unsigned long long seq) {
  __hip_atomic_store(&host->issued, issued, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&host->queued, queued, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  wait_stores();
  __hip_atomic_store(&host->seq, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Path regeneration (appended queues): the slots freed in this iteration take the next camera
// paths of the pass (up to `limit` paths in total), queued after the surviving paths.
__device__ __forceinline__ uint32_t regen_count(uint32_t freed, uint64_t limit, uint64_t issued) {
  const uint64_t left = limit > issued ? limit - issued : 0;
  return (uint32_t)min((uint64_t)freed, left);
}
__global__ void __launch_bounds__(256) k_regen(DeviceScene sc, PathQueues q, uint32_t *__restrict__ queue_out,
                                               const uint32_t *__restrict__ count_out, uint64_t limit, uint32_t npix,
                                               uint32_t spp_base, uint64_t seed) {
  const uint64_t issued = q.progress[0];
  const uint32_t n = regen_count(q.counters[kCountFree], limit, issued);
  const uint32_t out0 = *count_out;
  for (uint32_t k = gtid(); k < n; k += grid_stride()) {
    const uint32_t slot = q.free_slots[k];
    const uint64_t g = issued + k;
    init_camera_path(sc, q, slot, (uint32_t)(g % npix), spp_base + g / npix, npix, seed);
    queue_out[out0 + k] = slot;
  }
}
// Runs after k_regen (same stream): commits the issued paths and the queue length.  progress[1],
// which the host polls to end the pass, is the work of the next trace launch: the queue, plus the
// shadow rays queued for it when it takes them (with_shadow).
__global__ void k_regen_commit(PathQueues q, uint32_t *count_out, uint64_t limit, int with_shadow, PassProgress *host,
                               unsigned long long seq) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    const uint64_t issued = q.progress[0];
    const uint32_t n = regen_count(q.counters[kCountFree], limit, issued);
    const uint32_t total = *count_out + n;
    *count_out = total;
    // A queue of every slot is read as slot k = entry k (coalesced path-state accesses).
    count_out[kIdentOffset] = total == (uint32_t)q.capacity ? 1u : 0u;
    q.progress[0] = issued + n;
    q.progress[1] = total + (with_shadow ? *q.shadow_out : 0u);
    q.counters[kCountFree] = 0;
    report_progress(host, q.progress[0], q.progress[1], seq);
  }
}

// ---- slot-ordered queues -------------------------------------------------------------
// The next queue lists, in ascending slot order, the alive slots (paths that continue) and the
// freed slots the regeneration refills (the first min(freed, paths left) of the freed slots in
// ascending order): slot k lands at (alive slots before k) + min(freed slots before k, refilled).
// Two launches per iteration.  k_slot_select counts the flags of each chunk of kSlotBlock slots
// (one wave per chunk, 16 flags of each kind per lane in two 16-byte loads); its last block turns
// the counts into prefix sums, commits the pass's progress and reports it to the host.
// k_slot_scatter writes the queue and starts the new camera paths in their slots.  Both are bound
// by launch latency below a million slots (6 + 5 us); over 4 M slots they take 12 + 46 us, where
// separate count, scan, scatter, regeneration and commit kernels, the clears of the counters and
// the progress copy took 13 + 8 + 17 + 37 + 5 + 9 + 4 us in nine launches (1080p benchmark, average
// launch).
constexpr int kSlotBlock = 1024;

// Storage of the selection: the plan, the chunks' packed counts, and their prefix sums.
struct SlotTemp {
  SlotPlan plan;
  uint32_t counts[1];  // nb packed counts (alive | freed << 16), then nb alive and nb freed prefix sums
};

__global__ void __launch_bounds__(kSlotBlock) k_slot_select(PathQueues q, uint32_t n, uint32_t nb, SlotTemp *__restrict__ tmp,
                                                            uint32_t *count_out, uint64_t limit, uint32_t npix, uint32_t spp_base,
                                                            int with_shadow, PassProgress *host, unsigned long long seq) {
  constexpr int kWaves = kSlotBlock / 64;
  __shared__ uint32_t s_part[2][kWaves];
  __shared__ int s_last;
  const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
  uint32_t *counts = tmp->counts;
  const uint32_t chunk = blockIdx.x * kWaves + wave;
  if (chunk < nb) {
    const uint32_t base = chunk * kSlotBlock + 16u * lane;
    uint32_t c = 0;
    if (base + 16u <= n) {
      const uint4 a = *reinterpret_cast<const uint4 *>(q.alive + base), f = *reinterpret_cast<const uint4 *>(q.freed + base);
      c = (uint32_t)(__popc(a.x) + __popc(a.y) + __popc(a.z) + __popc(a.w)) +
          ((uint32_t)(__popc(f.x) + __popc(f.y) + __popc(f.z) + __popc(f.w)) << 16);
    } else {
      for (uint32_t k = base; k < n; ++k) c += (uint32_t)q.alive[k] + ((uint32_t)q.freed[k] << 16);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if (lane == 0) {
      __hip_atomic_store(counts + chunk, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      wait_stores();
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) s_last = atomicAdd(q.counters + kSlotTicket, 1u) == gridDim.x - 1u;
  __syncthreads();
  if (!s_last) return;
  // The last block to arrive: every chunk's count is in memory.
  const uint32_t per = (nb + kSlotBlock - 1) / kSlotBlock, b0 = min(threadIdx.x * per, nb), b1 = min(b0 + per, nb);
  uint32_t *pa = counts + nb, *pf = counts + 2 * (size_t)nb;
  uint32_t ta = 0, tf = 0;
  for (uint32_t b = b0; b < b1; ++b) {
    const uint32_t c = __hip_atomic_load(counts + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    ta += c & 0xffffu;
    tf += c >> 16;
  }
  uint32_t ia = ta, jf = tf;  // inclusive sums over the wave's threads
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t va = __shfl_up(ia, o), vf = __shfl_up(jf, o);
    ia += lane >= o ? va : 0u;
    jf += lane >= o ? vf : 0u;
  }
  if (lane == 63) {
    s_part[0][wave] = ia;
    s_part[1][wave] = jf;
  }
  __syncthreads();
  uint32_t before_a = 0, before_f = 0, all_a = 0, all_f = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) {
      before_a += s_part[0][w];
      before_f += s_part[1][w];
    }
    all_a += s_part[0][w];
    all_f += s_part[1][w];
  }
  uint32_t ra = before_a + ia - ta, rf = before_f + jf - tf;
  for (uint32_t b = b0; b < b1; ++b) {
    const uint32_t c = __hip_atomic_load(counts + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    pa[b] = ra;
    pf[b] = rf;
    ra += c & 0xffffu;
    rf += c >> 16;
  }
  if (threadIdx.x == 0) {
    const uint64_t issued = q.progress[0];
    const uint32_t refill = regen_count(all_f, limit, issued);
    const uint32_t total = all_a + refill;
    tmp->plan = SlotPlan{spp_base + issued / npix, (uint32_t)(issued % npix), refill};
    *count_out = total;
    // A queue of every slot of the pass is read as slot k = entry k (coalesced path-state accesses).
    count_out[kIdentOffset] = total == n ? 1u : 0u;
    q.progress[0] = issued + refill;
    q.progress[1] = total + (with_shadow ? *q.shadow_out : 0u);
    *q.shadow_in = 0;  // read by this iteration's trace launch; the next shade launch appends there
    q.counters[kSlotTicket] = 0;
    report_progress(host, q.progress[0], q.progress[1], seq);
  }
}

__global__ void __launch_bounds__(kSlotBlock) k_slot_scatter(DeviceScene sc, PathQueues q, uint32_t n, uint32_t nb,
                                                             const SlotTemp *__restrict__ tmp, uint32_t npix, uint64_t seed,
                                                             uint32_t *__restrict__ queue_out) {
  __shared__ uint32_t s[2][kSlotBlock / 64];
  if (tmp->counts[blockIdx.x] == 0) return;  // no slot of the chunk is alive or freed
  const uint32_t k = blockIdx.x * kSlotBlock + threadIdx.x;
  const bool a = k < n && q.alive[k] != 0, f = k < n && q.freed[k] != 0;
  const uint64_t ma = __ballot(a), mf = __ballot(f);
  const int w = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
  if (lane == 0) {
    s[0][w] = (uint32_t)__popcll(ma);
    s[1][w] = (uint32_t)__popcll(mf);
  }
  __syncthreads();
  uint32_t ra = tmp->counts[nb + blockIdx.x], rf = tmp->counts[2 * (size_t)nb + blockIdx.x];
  for (int i = 0; i < w; ++i) {
    ra += s[0][i];
    rf += s[1][i];
  }
  const uint64_t below = (1ull << lane) - 1ull;
  ra += (uint32_t)__popcll(ma & below);
  rf += (uint32_t)__popcll(mf & below);
  const SlotPlan plan = tmp->plan;
  const bool refilled = f && rf < plan.refill;
  if (a || refilled) queue_out[ra + min(rf, plan.refill)] = k;
  if (refilled) {
    // pixel0 + rf stays below 2^32: fewer than 2^31 pixels, at most 2^26 slots.
    const uint32_t g = plan.pixel0 + rf;
    init_camera_path(sc, q, k, g % npix, plan.sample0 + g / npix, npix, seed);
    q.alive[k] = 1;
    q.freed[k] = 0;
  }
}

__global__ void k_report(PathQueues q, PassReport *host) {
  if (threadIdx.x < kNumCounters) host->counters[threadIdx.x] = q.counters[threadIdx.x];
  if (threadIdx.x == 0) {
    const unsigned int v = g_stack_overflow;
    host->stack_overflow = v;
    if (v) g_stack_overflow = 0;
  }
}

// ---- closest hit --------------------------------------------------------------
__device__ __forceinline__ void finalize_path(const PathQueues &q, double *fb, double *fb_sq, uint32_t i, float4 rad);
__device__ __forceinline__ float4 add_rgb(float4 rad, float3 c);
__device__ void shadow_done_guided(const DeviceScene &sc, const PathQueues &q, uint32_t i, bool occluded, double *fb, double *fb_sq);

// What k_shadow (kShadow 1) or k_shadow_guided (2) do with a traced shadow ray of path i.
template <int kShadow>
__device__ __forceinline__ void shadow_done(const DeviceScene &sc, const PathQueues &q, uint32_t i, bool occluded, double *fb,
                                            double *fb_sq) {
  if (kShadow == 2) {
    shadow_done_guided(sc, q, i, occluded, fb, fb_sq);
    return;
  }
  float4 rad = q.rad[i];
  if (!occluded) rad = add_rgb(rad, xyz(q.sh_contrib[i]));
  if (q.flags[i] & kFlagFinalizeAfterShadow) finalize_path(q, fb, fb_sq, i, rad);
  else q.rad[i] = rad;
}

// Work entry k of a trace launch: entries below the closest-hit count are closest-hit rays of the
// queue; with kShadow, the entries after them are the shadow rays the previous shade launch queued.
template <int kShadow>
__device__ __forceinline__ Ray trace_entry(const PathQueues &q, const uint32_t *queue, bool ident, uint32_t ccount, uint32_t k,
                                           uint32_t &i, bool &shadow) {
  Ray r;
  shadow = kShadow && k >= ccount;
  if (!shadow) {
    i = ident ? k : queue[k];
    r.org = xyz(q.org[i]);
    r.dir = xyz(q.dir[i]);
    r.tmax = 3.0e38f;
  } else {
    i = q.shadow_queue[k - ccount];
    const float4 o = q.sh_org[i];
    r.org = xyz(o);
    r.dir = xyz(q.sh_dir[i]);
    r.tmax = o.w;
  }
  return r;
}

// Rays of a trace launch: each wave owns a run of consecutive entries and takes new ones from it
// into its idle lanes whenever at most kRefill lanes still have a ray, so that long rays do not
// leave the wave nearly empty (a model of the benchmark scene's rays: 35 % of the lanes busy in node
// steps with one ray per lane, 47-54 % with runs of 256 rays).  Runs need no counter (a returning
// atomic per refill cost more than the idle lanes), and finished rays' results are written together
// at the next refill.  1080p benchmark, trace per 8-spp pass: one ray per lane with the decoded
// quantized nodes 20.6 ms; this kernel 17.0 / 16.4 / 16.4 / 16.5 / 17.0 ms refilling at 24 / 32 /
// 40 / 48 / 56 lanes; Cornell box 64 spp 2.76 ms, then 2.34 / 2.40 / 2.48 / 2.59 / 2.76.
constexpr int kRefill = 32;

// With kShadow (1: plain, 2: guided) the launch also traces the shadow rays of the previous shade
// launch (entries after the closest-hit queue), so that they need no launch of their own.
template <int kShadow>
__global__ void __launch_bounds__(kTraceBlock, TTGPU_TRACE_WAVES) k_trace(DeviceScene sc, PathQueues q, const uint32_t *__restrict__ queue,
                                                       const uint32_t *__restrict__ count_ptr, uint32_t *stats, double *fb,
                                                       double *fb_sq) {
  __shared__ int lds_stack[kLdsStack * kTraceBlock];
  int *stack = lds_stack + threadIdx.x;
  int spill[kSpillStack];
  const uint32_t ccount = *count_ptr;
  const uint32_t scount = kShadow ? *q.shadow_in : 0u;
  const uint32_t count = ccount + scount;
  const bool ident = count_ptr[kIdentOffset] != 0;
  const uint32_t waves = gridDim.x * (kTraceBlock / 64), wave = blockIdx.x * (kTraceBlock / 64) + (threadIdx.x >> 6);
  const uint32_t run = max(64u, ((count + waves - 1) / waves + 63u) & ~63u);
  uint32_t next = __builtin_amdgcn_readfirstlane((uint32_t)min((uint64_t)wave * run, (uint64_t)count));
  const uint32_t end = min(next + run, count);
  const uint64_t below = (1ull << __lane_id()) - 1ull;
  Trav t;
  t.node = -1;
  t.pmask = 0;
  bool loaded = false, shadow = false;  // loaded: the lane has a ray whose result is not written yet
  uint32_t i = 0;
  for (;;) {
    const bool idle = !t.active();
    if (idle && loaded) {
      if (kShadow && shadow) shadow_done<kShadow>(sc, q, i, t.hit.prim >= 0, fb, fb_sq);
      else q.hit[i] = t.hit.prim >= 0 ? make_float4(t.hit.t, t.hit.u, t.hit.v, as_float(t.hit.prim)) : make_float4(0.f, 0.f, 0.f, as_float(-1));
      loaded = false;
    }
    const uint64_t free_lanes = __ballot(idle);
    if (next < end) {
      const uint32_t k = next + (uint32_t)__popcll(free_lanes & below);
      if (idle && k < end) {
        const Ray r = trace_entry<kShadow>(q, queue, ident, ccount, k, i, shadow);
        trav_init(t, r, sc.num_prims, shadow, stack);
        loaded = true;
      }
      next = min(next + (uint32_t)__popcll(free_lanes), end);
    } else if (free_lanes == ~0ull) {
      break;
    }
    const int stop = next < end ? kRefill : 0;
    while ((int)__popcll(__builtin_amdgcn_ballot_w64(t.active())) > stop) trav_advance(t, sc.nodes, sc.prims_kz, stack, spill);
  }
  if (gtid() == 0) {
    atomicAdd(stats + kStatClosest, ccount);
    if (kShadow) atomicAdd(stats + kStatShadow, scount);
  }
}

// ---- environment lights (src/light.hxx:148-288, src/light.cxx:29-189) -------------
// Alias-table draw (Walker 1977, Vose 1991): bucket from u, kept when coin < threshold, else its
// alias; one load gives the index and its probability.
__device__ __forceinline__ uint32_t alias_pick(const float4 *t, uint32_t n, float u, float coin, float &p) {
  const uint32_t b = min((uint32_t)(u * (float)n), n - 1u);
  const float4 e = t[b];
  const bool keep = coin < e.x;
  p = keep ? e.z : e.w;
  return keep ? b : (uint32_t)as_int(e.y);
}

__device__ __forceinline__ void env_map_pixel(const DevEnvLight &e, float3 dir_out, int &x, int &y) {
  float3 l = mk(dot(e.frame_x, dir_out), dot(e.frame_y, dir_out), dot(e.frame_z, dir_out));
  // KartesianToSpherical (src/vec3f.hxx:298-323): component 2 is the polar axis.
  const float X = l.x, Z = l.y, Y = l.z;
  const float ax = fabsf(X), az = fabsf(Z);
  const float r = sqrtf(X * X + Y * Y + Z * Z);
  float theta = acosf(fminf(1.f, fmaxf(-1.f, Y / r)));
  float phi;
  if (ax > az) {
    phi = atan2f(Z, ax);
    phi = X > 0.f ? phi : kPi - phi;
  } else {
    phi = atan2f(X, az);
    phi = Z > 0.f ? 0.5f * kPi - phi : 1.5f * kPi + phi;
  }
  float u = phi * (0.5f * kInvPi), v = theta * kInvPi;
  u = u - floorf(u);
  v = v - floorf(v);
  if (u > 1.f - kFltEps) u -= kFltEps;
  if (v > 1.f - kFltEps) v -= kFltEps;
  if (!(u >= 0.f)) u = 0.f;  // also catches NaN directions
  if (!(v >= 0.f)) v = 0.f;
  x = max(0, min((int)(u * e.tex_w), e.tex_w - 1));
  y = e.tex_h - 1 - max(0, min((int)(v * e.tex_h), e.tex_h - 1));
}
__device__ __forceinline__ void env_pixel_bounds(const DevEnvLight &e, int x, int y, float &phi0, float &z0, float &phi1, float &z1) {
  float ul = (float)x / e.tex_w, vl = 1.f - (float)y / e.tex_h;
  float uu = ul + 1.f / e.tex_w, vu = 1.f - (float)(y + 1) / e.tex_h;
  phi0 = ul * 2.f * kPi; phi1 = uu * 2.f * kPi;
  z0 = cosf(vl * kPi); z1 = cosf(vu * kPi);
}
__device__ float4 env_eval_one(const DevEnvLight &e, float3 dir_out, uint32_t bins, float *pdf) {
  switch (e.kind) {
    case TTGPU_ENV_SUN: {
      bool in = dot(dir_out, e.frame_z) > e.cos_open;
      *pdf = in ? e.pdf : 0.f;
      return in ? take(e.spectrum, bins) : f4(0.f);
    }
    case TTGPU_ENV_DOME: {
      bool in = dot(dir_out, -e.dir) > 0.f;
      *pdf = in ? 1.f / (2.f * kPi) : 0.f;
      return in ? take(e.spectrum, bins) : f4(0.f);
    }
    case TTGPU_ENV_DIRECTIONAL: *pdf = 0.f; return f4(0.f);
    case TTGPU_ENV_MAP: {
      int x, y;
      env_map_pixel(e, dir_out, x, y);
      const float4 tx = e.texel[(size_t)y * e.tex_w + x];
      const float prow = e.alias_rows[y].z;
      float p0, z0, p1, z1;
      env_pixel_bounds(e, x, y, p0, z0, p1, z1);
      *pdf = prow * tx.w / ((z1 - z0) * (p1 - p0));
      return rgb_to_spectral(mk(tx.x, tx.y, tx.z), bins);
    }
  }
  *pdf = 0.f;
  return f4(0.f);
}
// Sum of all env lights and their average pdf (TotalEnvironmentalRadianceField).
__device__ float4 env_eval(const DeviceScene &sc, float3 dir_out, uint32_t bins, float *pdf) {
  float4 L = f4(0.f);
  float p = 0.f;
  for (int i = 0; i < sc.num_envs; ++i) {
    float pi;
    L = L + env_eval_one(sc.envs[i], dir_out, bins, &pi);
    p += pi;
  }
  *pdf = sc.num_envs ? p / sc.num_envs : 0.f;
  return L;
}
__device__ void env_sample(const DeviceScene &sc, uint32_t bins, Pcg &rng, float3 &dir_out, float4 &val, float &pdf, bool &delta) {
  int i = sc.num_envs > 1 ? (int)rng.bounded(sc.num_envs) : 0;
  const DevEnvLight &e = sc.envs[i];
  delta = false;
  switch (e.kind) {
    case TTGPU_ENV_SUN: {
      float r0 = rng.uniform(), r1 = rng.uniform();
      float3 l = to_sphere_section(e.cos_open, r0, r1);
      dir_out = e.frame_x * l.x + e.frame_y * l.y + e.frame_z * l.z;
      val = take(e.spectrum, bins);
      pdf = e.pdf;
      break;
    }
    case TTGPU_ENV_DOME: {
      float r0 = rng.uniform(), r1 = rng.uniform();
      float3 l = to_uniform_hemisphere(r0, r1);
      dir_out = e.frame_x * l.x + e.frame_y * l.y + e.frame_z * l.z;
      val = take(e.spectrum, bins);
      pdf = 1.f / (2.f * kPi);
      break;
    }
    case TTGPU_ENV_DIRECTIONAL: {
      dir_out = e.dir;
      val = take(e.spectrum, bins);
      pdf = 1.f;
      delta = true;
      break;
    }
    default: {
      // Pixel with probability p_row * p_col (the sin-theta weighted CMFs of src/light.cxx:88-116,
      // drawn from alias tables), then a uniform point of its solid angle.
      const float r0 = rng.uniform(), r1 = rng.uniform(), c0 = rng.uniform(), c1 = rng.uniform();
      float prow, pcol;
      const uint32_t y = alias_pick(e.alias_rows, e.tex_h, r1, c1, prow);
      const uint32_t x = alias_pick(e.alias_cols + (size_t)y * e.tex_w, e.tex_w, r0, c0, pcol);
      const float4 tx = e.texel[(size_t)y * e.tex_w + x];
      float p0, z0, p1, z1;
      env_pixel_bounds(e, x, y, p0, z0, p1, z1);
      float s0 = rng.uniform(), s1 = rng.uniform();
      float3 l = to_sphere_section(s0, s1, p0, z0, p1, z1);
      dir_out = e.frame_x * l.x + e.frame_y * l.y + e.frame_z * l.z;
      val = rgb_to_spectral(mk(tx.x, tx.y, tx.z), bins);
      pdf = prow * pcol / ((z1 - z0) * (p1 - p0));
      break;
    }
  }
  pdf /= (float)sc.num_envs;
}

// ---- surface interaction at a hit ----------------------------------------------
__device__ __forceinline__ SurfHit make_hit(const DeviceScene &sc, int prim, float u, float v, float t, float3 org, float3 dir) {
  SurfHit h;
  const PrimRecord pr = sc.prims[prim];
  h.prim = prim;
  h.material = sc.prim_material[prim];
  if (as_int(pr.b.w) == 0) {
    const float3 v0 = xyz(pr.a), v1 = xyz(pr.b), v2 = xyz(pr.c);
    const float b0 = 1.f - u - v;
    h.pos = v0 * b0 + v1 * u + v2 * v;
    h.ng = normalize(cross(v1 - v0, v2 - v0));
    if (sc.prim_normals) {
      const float4 *nn = sc.prim_normals + 3 * (size_t)prim;
      h.ns = normalize(xyz(nn[0]) * b0 + xyz(nn[1]) * u + xyz(nn[2]) * v);
    } else {
      h.ns = h.ng;
    }
    // PBRT position error bound gamma(7) * sum |b_i p_i| (src/primitive.cxx:291-299), projected on |n|.
    const float g7 = 7.f * kFltEps * 0.5f / (1.f - 7.f * kFltEps * 0.5f);
    float3 e = mk(fabsf(v0.x * b0) + fabsf(v1.x * u) + fabsf(v2.x * v), fabsf(v0.y * b0) + fabsf(v1.y * u) + fabsf(v2.y * v),
                  fabsf(v0.z * b0) + fabsf(v1.z * u) + fabsf(v2.z * v)) * g7;
    h.offset = e.x * fabsf(h.ng.x) + e.y * fabsf(h.ng.y) + e.z * fabsf(h.ng.z);
  } else {
    // FP64 reprojection onto the sphere (Spheres::GetLocalGeometry, src/primitive.cxx:214-223):
    // the position then carries only its final rounding to FP32, which the offset covers.
    const double px = (double)org.x + (double)dir.x * t - pr.a.x, py = (double)org.y + (double)dir.y * t - pr.a.y,
                 pz = (double)org.z + (double)dir.z * t - pr.a.z;
    const double inv = 1.0 / sqrt(px * px + py * py + pz * pz);
    const double nx = px * inv, ny = py * inv, nz = pz * inv, r = pr.b.x;
    h.ng = mk((float)nx, (float)ny, (float)nz);
    h.pos = mk((float)(pr.a.x + nx * r), (float)(pr.a.y + ny * r), (float)(pr.a.z + nz * r));
    h.ns = h.ng;
    const float g5 = 5.f * kFltEps * 0.5f / (1.f - 5.f * kFltEps * 0.5f);
    h.offset = (fabsf(h.pos.x) * fabsf(h.ng.x) + fabsf(h.pos.y) * fabsf(h.ng.y) + fabsf(h.pos.z) * fabsf(h.ng.z)) * g5;
  }
  // Orient towards the incoming ray (SurfaceInteraction::SetOrientedNormals, src/scene.cxx:239-244).
  const float sign = -copysignf(1.f, dot(dir, h.ng));
  h.n = h.ng * sign;
  h.ns = h.ns * sign;
  return h;
}

// Adds a finished path's radiance to its pixel and hands its slot to path regeneration (one
// atomic per wave on the free-slot counter: the lanes finishing here share it).
__device__ __forceinline__ void finalize_path(const PathQueues &q, double *fb, double *fb_sq, uint32_t i, float4 rad) {
  if (q.freed) q.freed[i] = 1;
  else q.free_slots[wave_append(q.counters + kCountFree, true)] = i;
  const uint32_t p = q.pixel[i];
  atomicAdd(fb + 3 * (size_t)p + 0, (double)rad.x);
  atomicAdd(fb + 3 * (size_t)p + 1, (double)rad.y);
  atomicAdd(fb + 3 * (size_t)p + 2, (double)rad.z);
  if (fb_sq) {
    atomicAdd(fb_sq + 3 * (size_t)p + 0, (double)rad.x * rad.x);
    atomicAdd(fb_sq + 3 * (size_t)p + 1, (double)rad.y * rad.y);
    atomicAdd(fb_sq + 3 * (size_t)p + 2, (double)rad.z * rad.z);
  }
}

__device__ __forceinline__ float4 add_rgb(float4 rad, float3 c) { return make_float4(rad.x + c.x, rad.y + c.y, rad.z + c.z, rad.w); }

// ---- light selection and sampling for NEE (pt2.cxx:479-540, lightpicker_trivial.cxx:35-51) ----
struct LightSample {
  float3 dir;     // from the shading point towards the light
  float len;      // distance to the light (environment: 10 x scene diagonal)
  float4 weight;  // light value / (pdf x selection probability), incl. 1/len^2 for positional lights
  float pdf;      // pdf handed to MisWeight (solid angle; selection probability only in consistent mode)
  bool delta, valid;
};

// `fallback_dir` is used when the sampled light point coincides with `here` (SegmentToPoint).
// pt: the pdf always includes the selection probability and the cosine at an area light uses its
// geometry normal (DFactorOf, rendering_randomwalk_impl.hxx:758-769).
template <bool kPt = false>
__device__ __forceinline__ LightSample sample_light(const DeviceScene &sc, float3 here, float3 fallback_dir, uint32_t bins, Pcg &rng) {
  LightSample ls;
  ls.dir = mk(0.f, 0.f, 1.f);
  ls.len = 0.f;
  ls.weight = f4(0.f);
  ls.pdf = 0.f;
  ls.delta = false;
  const float u_type = rng.uniform();
  const float u_idx = rng.uniform();
  int kind = 3;
  {
    float r = u_type;
    while (kind > 0 && r >= sc.type_probs[kind]) { r -= sc.type_probs[kind]; --kind; }
  }
  // A type whose light count is zero can only be reached through float rounding of the
  // selection probabilities; it contributes nothing.
  ls.valid = (kind == 0 && sc.num_envs > 0) || (kind == 1 && sc.num_area_lights > 0) || (kind == 2 && sc.num_points > 0);
  if (!ls.valid) return ls;
  if (kind == 1) {
    const uint32_t li = min((uint32_t)(u_idx * sc.num_area_lights), (uint32_t)sc.num_area_lights - 1u);
    const int lp = sc.area_lights[li];
    const PrimRecord pr = sc.prims[lp];
    const float r0 = rng.uniform(), r1 = rng.uniform();
    float3 lpos, lng, lns;
    if (as_int(pr.b.w) == 0) {
      const float3 v0 = xyz(pr.a), v1 = xyz(pr.b), v2 = xyz(pr.c);
      const float s = sqrtf(r0);
      const float b0 = 1.f - s, b1 = (1.f - r1) * s, b2 = r1 * s;
      lpos = v0 * b0 + v1 * b1 + v2 * b2;
      lng = normalize(cross(v1 - v0, v2 - v0));
      if (sc.prim_normals) {
        const float4 *nn = sc.prim_normals + 3 * (size_t)lp;
        lns = normalize(xyz(nn[0]) * b0 + xyz(nn[1]) * b1 + xyz(nn[2]) * b2);
      } else {
        lns = lng;
      }
    } else {
      lng = to_uniform_sphere(r0, r1);
      lns = lng;
      lpos = xyz(pr.a) + lng * pr.b.x;
    }
    float3 d = lpos - here;
    ls.len = length(d);
    ls.dir = ls.len > 0.f ? d * (1.f / ls.len) : fallback_dir;
    if (!(ls.len > 0.f)) ls.len = 2.220446049250313e-16f;
    const DevEmitter &em = sc.emitters[sc.materials[sc.prim_material[lp]].emitter];
    float4 Le = (em.kind == TTGPU_AREA_UNIFORM && dot(lng, -ls.dir) > 0.f) ? take(em.radiance, bins) : f4(0.f);
    const float area_pdf = 1.f / sc.prim_area[lp];
    const float dfac = fabsf(dot(kPt ? lng : lns, ls.dir));
    ls.weight = (dfac / (area_pdf * sc.area_pick_prob * ls.len * ls.len)) * Le;
    ls.pdf = area_to_solid_angle(ls.len, ls.dir, lng) * area_pdf;
    if (kPt || sc.mis_mode == TTGPU_MIS_CONSISTENT) ls.pdf *= sc.area_pick_prob;
  } else if (kind == 0) {
    float3 dout;
    float4 val;
    float p;
    env_sample(sc, bins, rng, dout, val, p, ls.delta);
    ls.dir = -dout;
    ls.len = 10.f * sc.bb_diag;
    ls.weight = (1.f / (p * sc.type_probs[0])) * val;
    ls.pdf = p * ((kPt || sc.mis_mode == TTGPU_MIS_CONSISTENT) ? sc.type_probs[0] : 1.f);
  } else {
    const uint32_t li = min((uint32_t)(u_idx * sc.num_points), (uint32_t)sc.num_points - 1u);
    const DevPointLight &pl = sc.points[li];
    float3 d = pl.pos - here;
    ls.len = length(d);
    ls.dir = ls.len > 0.f ? d * (1.f / ls.len) : fallback_dir;
    if (!(ls.len > 0.f)) ls.len = 2.220446049250313e-16f;
    const float prob = sc.type_probs[2] / sc.num_points;
    ls.weight = (1.f / (prob * ls.len * ls.len)) * take(pl.intensity, bins);
    ls.pdf = 1.f;
    ls.delta = true;
  }
  return ls;
}

// ---- per-block compaction by material class (LDS, ballot / prefix sums) ----------------------
// Class of a queued path for shading: 0 = the ray escaped, 1 + shader kind otherwise; inactive
// entries take the last class.
constexpr int kSortClasses = 10;
__device__ __forceinline__ int shade_class(const DeviceScene &sc, const PathQueues &q, uint32_t i) {
  const int prim = as_int(q.hit[i].w);
  if (prim < 0) return 0;
  return 1 + min(sc.shaders[sc.materials[sc.prim_material[prim]].shader].kind, kSortClasses - 3);
}

// Stable counting sort of the block's kWaves x 64 (active, slot) entries by class: per-wave class counts
// by ballot and popcount, block-wide prefix sums over (class, wave), one LDS scatter.  Afterwards
// thread t takes the t-th entry, so each wave shades (mostly) one class and the inactive entries
// gather in the last waves.  Every thread of the block must call it.
template <int kWaves>
__device__ __forceinline__ void block_sort_by_class(const DeviceScene &sc, const PathQueues &q, bool &active, uint32_t &i,
                                                    uint32_t *s_idx, uint32_t (*s_cnt)[kSortClasses]) {
  const int cls = active ? shade_class(sc, q, i) : kSortClasses - 1;
  const int lane = __lane_id(), wave = (int)(threadIdx.x >> 6);
  const uint64_t below = (1ull << lane) - 1ull;
  uint32_t rank = 0;
  for (int c = 0; c < kSortClasses; ++c) {
    const uint64_t m = __ballot(cls == c);
    if (cls == c) rank = (uint32_t)__popcll(m & below);
    if (lane == 0) s_cnt[wave][c] = (uint32_t)__popcll(m);
  }
  __syncthreads();
  uint32_t off = 0;
  for (int c = 0; c < cls; ++c)
#pragma unroll
    for (int w = 0; w < kWaves; ++w) off += s_cnt[w][c];
  for (int w = 0; w < wave; ++w) off += s_cnt[w][cls];
  s_idx[off + rank] = active ? i : 0xFFFFFFFFu;
  __syncthreads();
  i = s_idx[threadIdx.x];
  active = i != 0xFFFFFFFFu;
  __syncthreads();  // the next iteration rewrites s_idx and s_cnt
}

// Block-aggregated appends to two queues: per-wave counts through LDS, one atomic per queue and
// block (instead of one per wave), block-wide prefix over the waves.  Reuses the sort's class
// counters (free once the sort has finished); every thread of the block must call it.
template <int kWaves>
__device__ __forceinline__ void block_append2(uint32_t *ca, bool pa, uint32_t *cb, bool pb, uint32_t (*s_cnt)[kSortClasses],
                                              uint32_t &slot_a, uint32_t &slot_b) {
  static_assert(kSortClasses >= 4, "two counts and two bases per wave row");
  const uint64_t ma = __ballot(pa), mb = __ballot(pb);
  const int lane = __lane_id(), wave = (int)(threadIdx.x >> 6);
  const uint64_t below = (1ull << lane) - 1ull;
  if (lane == 0) {
    s_cnt[wave][0] = (uint32_t)__popcll(ma);
    s_cnt[wave][1] = (uint32_t)__popcll(mb);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t ta = 0, tb = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) { ta += s_cnt[w][0]; tb += s_cnt[w][1]; }
    s_cnt[0][2] = ta ? atomicAdd(ca, ta) : 0u;
    s_cnt[0][3] = tb ? atomicAdd(cb, tb) : 0u;
  }
  __syncthreads();
  uint32_t oa = s_cnt[0][2], ob = s_cnt[0][3];
  for (int w = 0; w < wave; ++w) { oa += s_cnt[w][0]; ob += s_cnt[w][1]; }
  slot_a = oa + (uint32_t)__popcll(ma & below);
  slot_b = ob + (uint32_t)__popcll(mb & below);
  __syncthreads();  // the next iteration rewrites s_cnt
}

__device__ __forceinline__ float mis_weight(bool power, float a, float b) {
  return power ? a * a / (a * a + b * b) : a / (a + b);
}

// ---- shade: emission, NEE, scattering (pt2.cxx:410-443, 479-556, 605-684) --------
// kPt: pt's step instead (renderingalgorithms_pathtracing.hxx:749-794): power heuristic with the
// selection probability in the light pdf, no mollification, and the survival test (at most
// max_depth + 1 nodes, Russian roulette beyond 5) before NEE and scattering.
template <bool kPt>
__global__ void __launch_bounds__(256, TTGPU_SHADE_WAVES) k_shade(DeviceScene sc, PathQueues q, const uint32_t *__restrict__ queue_in,
                                               const uint32_t *__restrict__ count_in, uint32_t *__restrict__ queue_out,
                                               uint32_t *count_out, double *fb, double *fb_sq) {
  __shared__ uint32_t s_idx[256];
  __shared__ uint32_t s_cnt[4][kSortClasses];
  const uint32_t count = *count_in;
  const bool ident = count_in[kIdentOffset] != 0;
  const bool use_nee = sc.sample_mode != TTGPU_SAMPLE_BSDF;
  const bool use_emission = sc.sample_mode != TTGPU_SAMPLE_LIGHTS;
  const bool mis = use_nee && use_emission;
  const uint32_t n_iter = (count + grid_stride() - 1) / grid_stride();
  for (uint32_t it = 0; it < n_iter; ++it) {
    const uint32_t k = it * grid_stride() + gtid();
    bool active = k < count;
    bool push = false, push_shadow = false;
    uint32_t i = 0;
    if (active) i = ident ? k : queue_in[k];
    if (sc.sort_shade) block_sort_by_class<4>(sc, q, active, i, s_idx, s_cnt);
    if (active) {
      const float4 hitv = q.hit[i];
      const float3 dir = xyz(q.dir[i]);
      const float4 org4 = q.org[i];
      const float lambda0 = org4.w;
      float4 thru = q.thru[i];
      float4 rad = q.rad[i];
      const uint32_t bins = q.bins[i];
      uint32_t flags = q.flags[i];
      const float last_pdf = q.last_pdf[i];
      const bool has_last = (flags & kFlagHasLastPdf) != 0;
      const bool last_delta = (flags & kFlagLastPdfDelta) != 0;
      Pcg rng = load_rng(q, i);
      const int prim = as_int(hitv.w);
      if (prim < 0) {
        // AddEnvEmission (pt2.cxx:661-684)
        if (use_emission && sc.num_envs > 0) {
          float penv;
          float4 L = env_eval(sc, -dir, bins, &penv);
          float w = 1.f;
          if (has_last && !last_delta && mis) w = mis_weight(kPt, last_pdf, penv * sc.type_probs[0]);
          rad = add_rgb(rad, spectral_to_rgb(w * (L * thru), bins));
        }
        finalize_path(q, fb, fb_sq, i, rad);
      } else {
        const SurfHit h = make_hit(sc, prim, hitv.y, hitv.z, hitv.x, xyz(org4), dir);
        const DevMaterial mat = sc.materials[h.material];
        // MaybeAddEmission (pt2.cxx:627-658)
        if (use_emission && mat.emitter >= 0) {
          const DevEmitter &em = sc.emitters[mat.emitter];
          if (em.kind == TTGPU_AREA_UNIFORM && dot(h.ng, -dir) > 0.f) {
            float4 L = take(em.radiance, bins);
            float w = 1.f;
            if (has_last && !last_delta && mis) {
              float p_light = sc.area_pick_prob / sc.prim_area[prim] * area_to_solid_angle(hitv.x, dir, h.n);
              w = mis_weight(kPt, last_pdf, p_light);
            }
            rad = add_rgb(rad, spectral_to_rgb(w * (L * thru), bins));
          }
        }
        const DevShader &shd = sc.shaders[mat.shader];
        float rough = kPt ? 0.f : q.roughness[i];
        const float3 wi = -dir;
        const uint32_t node_here = flags & kFlagNodeMask;
        bool survive = true;
        if constexpr (kPt) {
          // SurvivalAtNthScatterNode (rendering_randomwalk_impl.hxx:729-756)
          survive = node_here < (uint32_t)sc.max_depth + 1u;
          if (survive && node_here > 5u) {
            const float p_survive = fminf(0.9f, fmaxf(fmaxf(thru.x, thru.y), fmaxf(thru.z, thru.w)));
            if (rng.uniform() > p_survive) survive = false;
            else thru = thru * (1.f / p_survive);
          }
        }
        // AddDirectLighting (pt2.cxx:479-556), vacuum transmission.
        if (survive && use_nee && (sc.num_area_lights + sc.num_envs + sc.num_points) > 0) {
          const LightSample ls = sample_light<kPt>(sc, h.pos, h.n, bins, rng);
          if (ls.valid) {
            float bsdf_pdf;
            float4 f = eval_bsdf(shd, h, wi, bins, rough, lambda0, ls.dir, &bsdf_pdf);
            const float dfac = fabsf(dot(h.ns, ls.dir));
            float w = 1.f;
            if (!ls.delta && mis) w = mis_weight(kPt, ls.pdf, bsdf_pdf);
            float4 c = (w * dfac) * (thru * f * ls.weight);
            float3 crgb = spectral_to_rgb(c, bins);
            if (crgb.x != 0.f || crgb.y != 0.f || crgb.z != 0.f) {
              const float3 o = offset_origin(h, ls.dir);
              q.sh_org[i] = make_float4(o.x, o.y, o.z, ls.len * 0.9999f);
              q.sh_dir[i] = make_float4(ls.dir.x, ls.dir.y, ls.dir.z, 0.f);
              q.sh_contrib[i] = make_float4(crgb.x, crgb.y, crgb.z, 0.f);
              push_shadow = true;
            }
          }
        }
        // MaybeScatter (pt2.cxx:605-622) and PrepareStateForAfterScattering (:583-591)
        if constexpr (!kPt) rough = fmaxf(my_roughness(shd), rough);
        Scatter s;
        uint32_t node = node_here + 1u;
        bool alive = kPt ? survive : node <= (uint32_t)sc.max_depth;
        if (alive) s = sample_bsdf(shd, h, wi, bins, rough, lambda0, rng);
        if (alive) {
          thru = (fabsf(dot(h.ns, s.dir)) / s.pdf) * (thru * s.value);
          alive = !all_zero(thru) && isfinite(thru.x + thru.y + thru.z + thru.w);
        }
        if (alive) {
          const float3 o = offset_origin(h, s.dir);
          q.org[i] = make_float4(o.x, o.y, o.z, lambda0);
          q.dir[i] = make_float4(s.dir.x, s.dir.y, s.dir.z, 0.f);
          q.thru[i] = thru;
          q.last_pdf[i] = s.pdf;
          q.roughness[i] = rough;
          flags = (flags & ~(kFlagNodeMask | kFlagLastPdfDelta)) | node | kFlagHasLastPdf | (s.delta ? kFlagLastPdfDelta : 0u);
          push = true;
        } else if (push_shadow) {
          flags |= kFlagFinalizeAfterShadow;
        } else {
          finalize_path(q, fb, fb_sq, i, rad);
        }
        q.flags[i] = flags;
        q.rad[i] = rad;
        store_rng(q, i, rng);
      }
    }
    uint32_t slot, sslot;
    block_append2<4>(count_out, push && !q.alive, q.shadow_out, push_shadow, s_cnt, slot, sslot);
    if (q.alive) {
      if (active) q.alive[i] = push ? 1 : 0;
    } else if (push) {
      queue_out[slot] = i;
    }
    if (push_shadow) q.shadow_queue[sslot] = i;
  }
}

// ---- shadow rays: any hit + accumulate + finalize -----------------------------------
__global__ void __launch_bounds__(kTraceBlock, TTGPU_TRACE_WAVES) k_shadow(DeviceScene sc, PathQueues q, double *fb, double *fb_sq, uint32_t *stats) {
  __shared__ int lds_stack[kLdsStack * kTraceBlock];
  const uint32_t count = *q.shadow_out;
  for (uint32_t k = gtid(); k < count; k += grid_stride()) {
    const uint32_t i = q.shadow_queue[k];
    const float4 o = q.sh_org[i];
    Ray r;
    r.org = xyz(o);
    r.dir = xyz(q.sh_dir[i]);
    r.tmax = o.w;
    HitRec h;
    bool occ = traverse<true>(sc.nodes, sc.prims_kz, sc.num_prims, r, lds_stack + threadIdx.x, h);
    float4 rad = q.rad[i];
    if (!occ) rad = add_rgb(rad, xyz(q.sh_contrib[i]));
    if (q.flags[i] & kFlagFinalizeAfterShadow) finalize_path(q, fb, fb_sq, i, rad);
    else q.rad[i] = rad;
  }
  if (gtid() == 0) atomicAdd(stats + kStatShadow, count);
}

// ---- pt: light points connected to the camera (renderingalgorithms_pathtracing.hxx:752-779) ----
// One connection per camera sample g of the pass (its own RNG stream and wavelengths): a light
// point, the pixel it projects to (PerspectiveCamera::Evaluate, camera.hxx:122-148) and, when the
// segment is unoccluded, MIS weight x camera importance (= direction pdf) x light value x
// wavelength weights / pixel count added to that pixel.  With TTGPU_MIS_REFERENCE the pixel index
// truncates toward zero as the reference does.
//
// Every sample hits the light's image, a few hundred to a few thousand pixels, so six FP64 atomics per
// sample on them bound the kernel: 1.88 ms for 4.2 M samples of the 512 x 512 Cornell box (780 pixels), 0.23
// without them.  Each block sums its samples in an LDS table of kConnectSlots pixels and adds each
// slot once at its end: 0.27 ms.  A pixel that finds no slot in kConnectProbes goes to memory as
// before; those are what a small table pays for (512 slots and two probes: 0.82 ms; with 1024 slots
// instead of 2048 images of 1750 and 3100 pixels, 768^2 and 1024^2 x 4 spp: 0.55 and 1.35 ms instead of
// 0.28 and 0.78; larger images gain little, 2048^2 x 4 spp 4.9 ms against 5.3 without a table).  In a
// large scene the traversal bounds the kernel, and one block per CU, which is what LDS admits, has to
// hold all the waves that the registers allow: 1024 threads, whose stacks keep 13 entries in LDS and
// the rest in private memory.  With 512 threads and 24 entries a light over the 1 M triangle terrain
// (960 x 540 x 8 spp) took 0.81 ms, now 0.58 (0.53 without the table).  More than 256 blocks only add
// tables to sum: Cornell box 0.36 ms with 512.
constexpr int kConnectBlock = 1024, kConnectBits = 11, kConnectSlots = 1 << kConnectBits, kConnectProbes = 16, kConnectBlocks = 256;
constexpr int kConnectStack = 13;  // traversal stack entries in LDS

__global__ void __launch_bounds__(kConnectBlock) k_camera_connect(DeviceScene sc, uint64_t first, uint64_t count, uint32_t npix,
                                                                   uint32_t spp_base, uint64_t seed, double *fb, double *fb_sq,
                                                                   uint32_t *stats) {
  static_assert(kConnectBlock % kTraceBlock == 0, "stack columns are laid out per kTraceBlock threads");
  __shared__ int lds_stack[kConnectStack * kConnectBlock];
  __shared__ uint32_t s_pixel[kConnectSlots];  // pixel + 1, 0: free
  __shared__ double s_sum[6][kConnectSlots];
  int *stack = lds_stack + (threadIdx.x / kTraceBlock) * (kConnectStack * kTraceBlock) + threadIdx.x % kTraceBlock;
  for (int k = threadIdx.x; k < kConnectSlots; k += kConnectBlock) {
    s_pixel[k] = 0;
#pragma unroll
    for (int j = 0; j < 6; ++j) s_sum[j][k] = 0.;
  }
  __syncthreads();
  const bool mis = sc.sample_mode == TTGPU_SAMPLE_BOTH;
  const DevCamera &c = sc.cam;
  uint32_t rays = 0;
  // Pixel and sample of g, advanced by the grid's stride without a division per sample.
  const uint32_t step_pixel = grid_stride() % npix, step_sample = grid_stride() / npix;
  uint32_t pixel = (uint32_t)((first + gtid()) % npix);
  uint64_t sample = spp_base + (first + gtid()) / npix;
  for (uint64_t g = gtid(); g < count; g += grid_stride(), pixel += step_pixel, sample += step_sample) {
    if (pixel >= npix) {
      pixel -= npix;
      ++sample;
    }
    Pcg rng;
    rng.seed(seed ^ 0xC2B2AE3D27D4EB4Full, sample * npix + pixel);
    const int main_idx = (int)rng.bounded(kStrata);
    int idx[4] = {main_idx, main_idx + kStrata, main_idx + 2 * kStrata, main_idx + 3 * kStrata};
    const int rot = (int)rng.bounded(4);
    const int t = idx[0]; idx[0] = idx[rot]; idx[rot] = t;
    const uint32_t bins = (uint32_t)idx[0] | ((uint32_t)idx[1] << 8) | ((uint32_t)idx[2] << 16) | ((uint32_t)idx[3] << 24);
    const LightSample ls = sample_light<true>(sc, c.pos, c.dir, bins, rng);
    if (!ls.valid) continue;
    const float z = dot(ls.dir, c.dir);
    if (!(z > 0.f)) continue;
    const float x = dot(ls.dir, c.right) / z, y = dot(ls.dir, c.up) / z;
    const float fx = (x - c.xmin) / c.xper, fy = (y - c.ymin) / c.yper;
    const bool trunc = sc.mis_mode != TTGPU_MIS_CONSISTENT;
    const float ix = trunc ? truncf(fx) : floorf(fx), iy = trunc ? truncf(fy) : floorf(fy);
    if (!(ix >= 0.f && ix < (float)c.width && iy >= 0.f && iy < (float)c.height)) continue;
    const float pdf_cam = camera_pdf(c, x, y);
    const float w = (!ls.delta && mis) ? mis_weight(true, ls.pdf, pdf_cam) : 1.f;
    const float3 crgb = spectral_to_rgb(((float)kStrata * w * pdf_cam / (float)npix) * ls.weight, bins);
    if (crgb.x == 0.f && crgb.y == 0.f && crgb.z == 0.f) continue;
    Ray r;
    r.org = c.pos;
    r.dir = ls.dir;
    r.tmax = ls.len * 0.9999f;
    HitRec hr;
    ++rays;
    if (traverse<true, kConnectStack>(sc.nodes, sc.prims_kz, sc.num_prims, r, stack, hr)) continue;
    const uint32_t p = (uint32_t)((size_t)iy * c.width + (size_t)ix);
    const double v[6] = {(double)crgb.x, (double)crgb.y, (double)crgb.z, (double)crgb.x * crgb.x, (double)crgb.y * crgb.y,
                         (double)crgb.z * crgb.z};
    uint32_t slot = (p * 2654435761u) >> (32 - kConnectBits), owner = 0u;
    for (int probe = 0; probe < kConnectProbes; ++probe) {
      owner = atomicCAS(&s_pixel[slot], 0u, p + 1u);
      if (owner == 0u || owner == p + 1u) break;
      slot = (slot + 1u) & (kConnectSlots - 1);
    }
    if (owner == 0u || owner == p + 1u) {
#pragma unroll
      for (int j = 0; j < 6; ++j) atomicAdd(&s_sum[j][slot], v[j]);
    } else {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        atomicAdd(fb + 3 * (size_t)p + j, v[j]);
        if (fb_sq) atomicAdd(fb_sq + 3 * (size_t)p + j, v[3 + j]);
      }
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kConnectSlots; k += kConnectBlock) {
    if (s_pixel[k] == 0) continue;
    const size_t p = s_pixel[k] - 1u;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      atomicAdd(fb + 3 * p + j, s_sum[j][k]);
      if (fb_sq) atomicAdd(fb_sq + 3 * p + j, s_sum[3 + j][k]);
    }
  }
  wave_stat(stats + kStatShadow, rays);
}

// ---- media: shade with null-path tracking (pt2.cxx:410-443 with media_integrator.cxx) ------
// One Step of the reference's path loop for scenes with participating media: tracking along the
// traced segment (volume boundaries, delta tracking), then emission, NEE and scattering at the
// surface hit or at the real collision in a medium.
// ---- guided integrator (ptg): BSDF/vMF one-sample mixture, power-heuristic MIS, records ------
// Radiance records follow PropagateIlluminationToParents / AddToTrainingData
// (src/renderingalgorithms_pathtracing_guided.cxx:1968-2034): the record of vertex j holds the
// radiance arriving from the direction sampled at j, i.e. the emission and NEE of vertex j+1 plus
// everything found later, carried back with throughput ratios clamped at 10; weight = radiance / pdf.
__device__ __forceinline__ float mean4(float4 v) { return 0.25f * (v.x + v.y + v.z + v.w); }
__device__ __forceinline__ float clamp_ratio(float a, float b) { return b > 0.f ? fminf(a / b, 10.f) : 0.f; }

// Radiance leaving vertex v towards vertex v-1: `direct` is recorded at v-1 as it is, `weighted`
// (emission with its MIS weight, plus NEE) is carried to the vertices before v-1.
__device__ __forceinline__ void propagate_radiance(const PathQueues &q, uint32_t i, int v, float4 direct, float4 weighted,
                                                   float4 thru_prev) {
  if (v <= 0) return;
  const size_t cap = (size_t)q.capacity;
  q.gv_dir_acc[(size_t)(v - 1) * cap + i].w += mean4(direct);
  for (int j = 0; j < v - 1; ++j) {
    const float4 tj = q.gv_thru[(size_t)j * cap + i];
    const float4 r = make_float4(clamp_ratio(thru_prev.x, tj.x), clamp_ratio(thru_prev.y, tj.y), clamp_ratio(thru_prev.z, tj.z),
                                 clamp_ratio(thru_prev.w, tj.w));
    q.gv_dir_acc[(size_t)j * cap + i].w += mean4(r * weighted);
  }
}

__device__ __forceinline__ void emit_records(const PathQueues &q, uint32_t i, int nv) {
  const size_t cap = (size_t)q.capacity;
  for (int j = 0; j < nv; ++j) {
    const float4 pp = q.gv_pos_pdf[(size_t)j * cap + i];
    if (!(pp.w > 0.f)) continue;
    const float4 da = q.gv_dir_acc[(size_t)j * cap + i];
    const uint32_t slot = wave_append(q.counters + kCountRecords, true);
    if (slot < q.rec_capacity) {
      const float w = da.w / pp.w;
      q.rec_pos_w[slot] = make_float4(pp.x, pp.y, pp.z, w);
      q.rec_dir[slot] = make_float4(da.x, da.y, da.z, w);
      if (q.rec_nrm) {
        q.rec_nrm[slot] = q.gv_nrm[(size_t)j * cap + i];
        q.rec_wo[slot] = q.gv_wo[(size_t)j * cap + i];
      }
    } else {
      atomicAdd(q.counters + kStatRecordsDropped, 1u);
    }
  }
}

// kAtmo: some medium is an atmosphere; without one its code and the collision loop go (248 -> 224
// registers, medium sphere 149 -> 146 us per launch).
template <bool kAtmo>
__global__ void __launch_bounds__(kTraceBlock) k_shade_media(DeviceScene sc, PathQueues q, const uint32_t *__restrict__ queue_in,
                                                             const uint32_t *__restrict__ count_in, uint32_t *__restrict__ queue_out,
                                                             uint32_t *count_out, double *fb, double *fb_sq) {
  __shared__ uint32_t s_idx[kTraceBlock];
  __shared__ uint32_t s_cnt[kTraceBlock / 64][kSortClasses];
  const uint32_t count = *count_in;
  const bool ident = count_in[kIdentOffset] != 0;
  const bool use_nee = sc.sample_mode != TTGPU_SAMPLE_BSDF;
  const bool use_emission = sc.sample_mode != TTGPU_SAMPLE_LIGHTS;
  const bool mis = use_nee && use_emission;
  const uint32_t n_iter = (count + grid_stride() - 1) / grid_stride();
  for (uint32_t it = 0; it < n_iter; ++it) {
    const uint32_t k = it * grid_stride() + gtid();
    bool active = k < count;
    bool push = false, push_shadow = false;
    uint32_t i = 0;
    if (active) i = ident ? k : queue_in[k];
    if (sc.sort_shade) block_sort_by_class<kTraceBlock / 64>(sc, q, active, i, s_idx, s_cnt);
    if (active) {
      const float4 hitv = q.hit[i];
      const float3 dir = xyz(q.dir[i]);
      const float4 org4 = q.org[i];
      const float3 org = xyz(org4);
      const float lambda0 = org4.w;
      float4 thru = q.thru[i];
      float4 rad = q.rad[i];
      const uint32_t bins = q.bins[i];
      uint32_t flags = q.flags[i];
      const float last_pdf = q.last_pdf[i];
      const bool mis_last = (flags & kFlagHasLastPdf) && !(flags & kFlagLastPdfDelta) && mis;
      Pcg rng = load_rng(q, i);
      const uint2 tp = q.tracker[i];
      Tracker tr{tp.x, tp.y};
      NullMat wt{q.wt_r[i], q.wt_c[i]};
      const int prim = as_int(hitv.w);
      // nullpath::Tracking(scene, ...) up to just before the surface hit.
      const double tfar = prim >= 0 ? (double)hitv.x : kLargeNumber;
      NullMat nulls = nm_ones(), track = nm_ones();
      double tcoll = 0.;
      float4 vss = f4(0.f);
      int vmed = kVacuum;
      const bool vol = track_scene<kAtmo>(sc, org, dir, tfar * 0.9999, bins, rng, tr, nulls, track, tcoll, vss, vmed);
      NullMat wtn = wt;
      nm_acc(wtn, nulls);
      nm_acc(wt, track);
      if (!vol && prim < 0) {
        // AddEnvEmission (pt2.cxx:661-684)
        if (use_emission && sc.num_envs > 0) {
          float penv;
          const float4 L = env_eval(sc, -dir, bins, &penv);
          const float4 fac = mis_factor(mis_last, last_pdf, penv * sc.type_probs[0], wt, wtn);
          rad = add_rgb(rad, spectral_to_rgb(fac * (L * thru), bins));
        }
        finalize_path(q, fb, fb_sq, i, rad);
      } else {
        SurfHit h;
        D3 vpos{0., 0., 0.};
        float3 here;
        float rough = q.roughness[i];
        int shader = -1;
        if (!vol) {
          h = make_hit(sc, prim, hitv.y, hitv.z, hitv.x, org, dir);
          const DevMaterial mat = sc.materials[h.material];
          shader = mat.shader;
          here = h.pos;
          // MaybeAddEmission (pt2.cxx:627-658)
          if (use_emission && mat.emitter >= 0) {
            const DevEmitter &em = sc.emitters[mat.emitter];
            if (em.kind == TTGPU_AREA_UNIFORM && dot(h.ng, -dir) > 0.f) {
              const float4 L = take(em.radiance, bins);
              const float p_light = sc.area_pick_prob / sc.prim_area[prim] * area_to_solid_angle(hitv.x, dir, h.n);
              const float4 fac = mis_factor(mis_last, last_pdf, p_light, wt, wtn);
              rad = add_rgb(rad, spectral_to_rgb(fac * (L * thru), bins));
            }
          }
        } else {
          vpos = d3_along(d3(org), dir, tcoll);
          here = f3(vpos);
        }
        const float3 wi = -dir;
        // AddDirectLighting (pt2.cxx:479-556); the transmission estimate is made by k_shadow_media.
        if (use_nee && (sc.num_area_lights + sc.num_envs + sc.num_points) > 0) {
          const LightSample ls = sample_light(sc, here, vol ? mk(1.f, 0.f, 0.f) : h.n, bins, rng);
          if (ls.valid) {
            float bsdf_pdf;
            float4 f;
            Tracker ntr = tr;
            float3 o;
            if (!vol) {
              f = eval_bsdf(sc.shaders[shader], h, wi, bins, rough, lambda0, ls.dir, &bsdf_pdf) * fabsf(dot(h.ns, ls.dir));
              maybe_going_through(sc, ntr, ls.dir, h);
              o = offset_origin(h, ls.dir);
            } else {
              f = medium_phase_eval<kAtmo>(sc, vmed, wi, vpos, bins, ls.dir, &bsdf_pdf);
              float4 ss, st;
              medium_coeffs<kAtmo>(sc, vmed, vpos, bins, ss, st);
              f = f * make_float4(ss.x / (st.x + kDblEps), ss.y / (st.y + kDblEps), ss.z / (st.z + kDblEps), ss.w / (st.w + kDblEps));
              o = here;
            }
            const float4 c = thru * f * ls.weight;
            if (!all_zero(c)) {
              q.sh_org[i] = make_float4(o.x, o.y, o.z, ls.len * 0.9999f);
              q.sh_dir[i] = make_float4(ls.dir.x, ls.dir.y, ls.dir.z, ls.delta ? -ls.pdf : ls.pdf);
              q.sh_contrib[i] = c;
              q.sh_aux[i] = make_uint4(ntr.cur, ntr.slots, (uint32_t)as_int(bsdf_pdf), 0u);
              push_shadow = true;
            }
          }
        }
        // MaybeScatter (pt2.cxx:605-622) and PrepareStateForAfterScattering (:583-599)
        Scatter s;
        if (!vol) {
          const DevShader &shd = sc.shaders[shader];
          rough = fmaxf(my_roughness(shd), rough);
          s = sample_bsdf(shd, h, wi, bins, rough, lambda0, rng);
        } else {
          s = medium_phase_sample<kAtmo>(sc, vmed, wi, vpos, bins, rng);
          float4 ss, st;
          medium_coeffs<kAtmo>(sc, vmed, vpos, bins, ss, st);
          s.value = s.value * make_float4(ss.x / (st.x + kDblEps), ss.y / (st.y + kDblEps), ss.z / (st.z + kDblEps), ss.w / (st.w + kDblEps));
        }
        const uint32_t node = (flags & kFlagNodeMask) + 1u;
        bool alive = node <= (uint32_t)sc.max_depth;
        if (alive) {
          const float d = vol ? 1.f : fabsf(dot(h.ns, s.dir));
          thru = (d / s.pdf) * (thru * s.value);
          alive = !all_zero(thru) && isfinite(thru.x + thru.y + thru.z + thru.w);
        }
        if (alive) {
          float3 o;
          if (!vol) {
            o = offset_origin(h, s.dir);
            maybe_going_through(sc, tr, s.dir, h);
          } else {
            o = here;
          }
          q.org[i] = make_float4(o.x, o.y, o.z, lambda0);
          q.dir[i] = make_float4(s.dir.x, s.dir.y, s.dir.z, 0.f);
          q.thru[i] = thru;
          q.last_pdf[i] = s.pdf;
          q.roughness[i] = rough;
          flags = (flags & ~(kFlagNodeMask | kFlagLastPdfDelta)) | node | kFlagHasLastPdf | (s.delta ? kFlagLastPdfDelta : 0u);
          push = true;
        } else if (push_shadow) {
          flags |= kFlagFinalizeAfterShadow;
        } else {
          finalize_path(q, fb, fb_sq, i, rad);
        }
        q.flags[i] = flags;
        q.rad[i] = rad;
        q.tracker[i] = make_uint2(tr.cur, tr.slots);
        q.wt_r[i] = wt.r;
        q.wt_c[i] = wt.c;
        store_rng(q, i, rng);
      }
    }
    uint32_t slot, sslot;
    block_append2<kTraceBlock / 64>(count_out, push && !q.alive, q.shadow_out, push_shadow, s_cnt, slot, sslot);
    if (q.alive) {
      if (active) q.alive[i] = push ? 1 : 0;
    } else if (push) {
      queue_out[slot] = i;
    }
    if (push_shadow) q.shadow_queue[sslot] = i;
  }
}

// ---- media: shadow rays with occlusion + null-path transmission + MIS -----------------------
template <bool kAtmo>
__global__ void __launch_bounds__(kTraceBlock) k_shadow_media(DeviceScene sc, PathQueues q, double *fb, double *fb_sq, uint32_t *stats) {
  __shared__ int lds_stack[kLdsStack * kTraceBlock];
  const uint32_t count = *q.shadow_out;
  const bool mis = sc.sample_mode == TTGPU_SAMPLE_BOTH;
  const bool rec = sc.guide_record != 0 && q.vt != nullptr;
  for (uint32_t k = gtid(); k < count; k += grid_stride()) {
    const uint32_t i = q.shadow_queue[k];
    const float4 o = q.sh_org[i];
    const float4 d4 = q.sh_dir[i];
    Ray r;
    r.org = xyz(o);
    r.dir = xyz(d4);
    r.tmax = o.w;
    HitRec h;
    const bool occ = traverse<true>(sc.nodes, sc.prims_kz, sc.num_prims, r, lds_stack + threadIdx.x, h);
    float4 rad = q.rad[i];
    if (!occ) {
      const uint4 aux = q.sh_aux[i];
      Tracker tr{aux.x, aux.y};
      const float bsdf_pdf = as_float((int)aux.z);
      const uint32_t bins = q.bins[i];
      Pcg rng = load_rng(q, i);
      NullMat nulls = nm_ones(), track = nm_ones();
      transmit_scene<kAtmo>(sc, r.org, r.dir, (double)o.w, bins, rng, tr, nulls, track);
      store_rng(q, i, rng);
      const NullMat wt{q.wt_r[i], q.wt_c[i]};
      nm_acc(nulls, wt);
      nm_acc(track, wt);
      const bool delta = d4.w < 0.f;
      const float4 fac = mis_factor(mis && !delta, fabsf(d4.w), bsdf_pdf, nulls, track);
      rad = add_rgb(rad, spectral_to_rgb(fac * q.sh_contrib[i], bins));
      // Guided integrator: the NEE radiance arriving at the vertex, with its transmission and MIS
      // factor, goes to the radiance records of the vertices before.
      if (rec && aux.w > 0u) {
        const float4 nee = fac * q.sh_nee[i];
        propagate_radiance(q, i, (int)aux.w, nee, nee, q.gv_thru[(size_t)(aux.w - 1u) * (size_t)q.capacity + i]);
      }
    }
    const uint32_t flags = q.flags[i];
    if (flags & kFlagFinalizeAfterShadow) {
      if (rec) emit_records(q, i, (int)((flags & kFlagVertexMask) >> kFlagVertexShift));
      finalize_path(q, fb, fb_sq, i, rad);
    } else {
      q.rad[i] = rad;
    }
  }
  if (gtid() == 0) atomicAdd(stats + kStatShadow, count);
}

// ---- guided integrator in participating media ------------------------------------------------
// The wavefront iteration becomes trace -> k_track_media -> (learned guide: inference at the
// interaction) -> k_shade_media_guided -> k_shadow_media: the interaction a path scatters at (a
// volume collision or its surface hit) must be known before the learned guide's batched inference.
// Distance sampling and transmission are pt2's null-path tracking; the direction at a surface or
// a volume vertex is drawn from the one-sample mixture of BSDF / phase function and guide
// (SampleWithBinaryMixtureDensity, renderingalgorithms_pathtracing_guided.cxx:473-544; at volume
// vertices with the phase function kept with probability 1/2, PROB_BSDF :470, and the guide of the
// vertex's position, :456-466, :1404-1408).  The mixture's density takes the BSDF's place in pt2's
// MIS weights, so the estimator stays pt2's with another direction sampler.  Radiance records
// come from surface and volume vertices alike (volume vertices carry a zero normal).

// nullpath::Tracking(scene, ...) (media_integrator.cxx:330-376) along the ray up to its surface
// hit: the collision distance (or none) and the tracking weights, for k_shade_media_guided.
__global__ void __launch_bounds__(kTraceBlock) k_track_media(DeviceScene sc, PathQueues q, const uint32_t *__restrict__ queue_in,
                                                             const uint32_t *__restrict__ count_in) {
  const uint32_t count = *count_in;
  const bool ident = count_in[kIdentOffset] != 0;
  for (uint32_t k = gtid(); k < count; k += grid_stride()) {
    const uint32_t i = ident ? k : queue_in[k];
    const float4 hitv = q.hit[i];
    const float3 dir = xyz(q.dir[i]);
    const float3 org = xyz(q.org[i]);
    const uint32_t bins = q.bins[i];
    Pcg rng = load_rng(q, i);
    const uint2 tp = q.tracker[i];
    Tracker tr{tp.x, tp.y};
    NullMat wt{q.wt_r[i], q.wt_c[i]};
    const int prim = as_int(hitv.w);
    const double tfar = prim >= 0 ? (double)hitv.x : kLargeNumber;
    NullMat nulls = nm_ones(), track = nm_ones();
    double tcoll = 0.;
    float4 vss;
    int vmed = kVacuum;
    const bool vol = track_scene(sc, org, dir, tfar * 0.9999, bins, rng, tr, nulls, track, tcoll, vss, vmed);
    NullMat wtn = wt;
    nm_acc(wtn, nulls);
    nm_acc(wt, track);
    q.vt[i] = vol ? tcoll : -1.;
    q.wt_r[i] = wt.r;
    q.wt_c[i] = wt.c;
    q.wtn_r[i] = wtn.r;
    q.wtn_c[i] = wtn.c;
    q.tracker[i] = make_uint2(tr.cur, tr.slots);
    store_rng(q, i, rng);
  }
}

// Phase function / guide one-sample mixture at a volume vertex; value includes sigma_s / sigma_t.
constexpr float kGuideProbPhase = 0.5f;
template <class M>
__device__ __forceinline__ Scatter sample_guided_phase(const DeviceScene &sc, int vmed, const M &g, float3 wi, D3 vpos, uint32_t bins,
                                                       Pcg &rng) {
  Scatter s = medium_phase_sample(sc, vmed, wi, vpos, bins, rng);
  if (rng.uniform() < kGuideProbPhase) {
    s.pdf = (1.f - kGuideProbPhase) * guide_pdf(g, s.dir) + kGuideProbPhase * s.pdf;
  } else {
    const float u0 = rng.uniform(), u1 = rng.uniform(), u2 = rng.uniform();
    s.dir = guide_sample(g, u0, u1, u2);
    float pp;
    s.value = medium_phase_eval(sc, vmed, wi, vpos, bins, s.dir, &pp);
    s.pdf = (1.f - kGuideProbPhase) * guide_pdf(g, s.dir) + kGuideProbPhase * pp;
  }
  float4 ss, st;
  medium_coeffs(sc, vmed, vpos, bins, ss, st);
  s.value = s.value * make_float4(ss.x / (st.x + kDblEps), ss.y / (st.y + kDblEps), ss.z / (st.z + kDblEps), ss.w / (st.w + kDblEps));
  return s;
}

template <int kGuide>
__global__ void __launch_bounds__(kTraceBlock) k_shade_media_guided(DeviceScene sc, PathQueues q, const uint32_t *__restrict__ queue_in,
                                                                    const uint32_t *__restrict__ count_in, uint32_t *__restrict__ queue_out,
                                                                    uint32_t *count_out, double *fb, double *fb_sq) {
  __shared__ uint32_t s_idx[kTraceBlock];
  __shared__ uint32_t s_cnt[kTraceBlock / 64][kSortClasses];
  constexpr bool kLearned = kGuide == 1, kQuad = kGuide == 2;
  const uint32_t count = *count_in;
  const bool ident = count_in[kIdentOffset] != 0;
  const bool use_nee = sc.sample_mode != TTGPU_SAMPLE_BSDF;
  const bool use_emission = sc.sample_mode != TTGPU_SAMPLE_LIGHTS;
  const bool mis = use_nee && use_emission;
  const bool rec = sc.guide_record != 0;
  const size_t cap = (size_t)q.capacity;
  const uint32_t n_iter = (count + grid_stride() - 1) / grid_stride();
  for (uint32_t it = 0; it < n_iter; ++it) {
    const uint32_t k = it * grid_stride() + gtid();
    bool active = k < count;
    bool push = false, push_shadow = false;
    uint32_t i = 0;
    if (active) i = ident ? k : queue_in[k];
    if (sc.sort_shade) block_sort_by_class<kTraceBlock / 64>(sc, q, active, i, s_idx, s_cnt);
    if (active) {
      const float4 hitv = q.hit[i];
      const float3 dir = xyz(q.dir[i]);
      const float4 org4 = q.org[i];
      const float3 org = xyz(org4);
      const float lambda0 = org4.w;
      float4 thru = q.thru[i];
      float4 rad = q.rad[i];
      const uint32_t bins = q.bins[i];
      uint32_t flags = q.flags[i];
      const int nv = (int)((flags & kFlagVertexMask) >> kFlagVertexShift);
      const float last_pdf = q.last_pdf[i];
      const bool mis_last = (flags & kFlagHasLastPdf) && !(flags & kFlagLastPdfDelta) && mis;
      Pcg rng = load_rng(q, i);
      const uint2 tp = q.tracker[i];
      Tracker tr{tp.x, tp.y};
      const NullMat wt{q.wt_r[i], q.wt_c[i]}, wtn{q.wtn_r[i], q.wtn_c[i]};
      const int prim = as_int(hitv.w);
      const double tcoll = q.vt[i];
      const bool vol = tcoll >= 0.;
      if (!vol && prim < 0) {
        if (use_emission && sc.num_envs > 0) {
          float penv;
          const float4 L = env_eval(sc, -dir, bins, &penv);
          const float4 fac = mis_factor(mis_last, last_pdf, penv * sc.type_probs[0], wt, wtn);
          rad = add_rgb(rad, spectral_to_rgb(fac * (L * thru), bins));
          if (rec) propagate_radiance(q, i, nv, fac * L, fac * L, thru);
        }
        if (rec) emit_records(q, i, nv);
        finalize_path(q, fb, fb_sq, i, rad);
      } else {
        SurfHit h;
        D3 vpos{0., 0., 0.};
        float3 here;
        float rough = q.roughness[i];
        int shader = -1;
        const int vmed = (int)tr.cur;
        if (!vol) {
          h = make_hit(sc, prim, hitv.y, hitv.z, hitv.x, org, dir);
          const DevMaterial mat = sc.materials[h.material];
          shader = mat.shader;
          here = h.pos;
          if (use_emission && mat.emitter >= 0) {
            const DevEmitter &em = sc.emitters[mat.emitter];
            if (em.kind == TTGPU_AREA_UNIFORM && dot(h.ng, -dir) > 0.f) {
              const float4 L = take(em.radiance, bins);
              const float p_light = sc.area_pick_prob / sc.prim_area[prim] * area_to_solid_angle(hitv.x, dir, h.n);
              const float4 fac = mis_factor(mis_last, last_pdf, p_light, wt, wtn);
              rad = add_rgb(rad, spectral_to_rgb(fac * (L * thru), bins));
              if (rec) propagate_radiance(q, i, nv, fac * L, fac * L, thru);
            }
          }
        } else {
          vpos = d3_along(d3(org), dir, tcoll);
          here = f3(vpos);
        }
        // The guide of this vertex: the learned per-path mixture, or the cell's quadtree or vMF mixture.
        const GuideCell *cellp = nullptr;
        const nn::Mix16 *mixp = nullptr;
        QuadGuide qg{};
        if constexpr (kLearned) mixp = reinterpret_cast<const nn::Mix16 *>(q.gmix) + i;
        else if constexpr (kQuad) qg = quad_guide(sc, guide_lookup(sc, here));
        else cellp = sc.guide_cells + guide_lookup(sc, here);
        auto gpdf = [&](float3 d) -> float {
          if constexpr (kLearned) return guide_pdf(*mixp, d);
          else if constexpr (kQuad) return guide_pdf(qg, d);
          else return guide_pdf(*cellp, d);
        };
        const float3 wi = -dir;
        // NEE; the transmission estimate and the MIS weight (against the mixture's density) are
        // made by k_shadow_media.
        if (use_nee && (sc.num_area_lights + sc.num_envs + sc.num_points) > 0) {
          const LightSample ls = sample_light(sc, here, vol ? mk(1.f, 0.f, 0.f) : h.n, bins, rng);
          if (ls.valid) {
            float mix_pdf;
            float4 f;
            Tracker ntr = tr;
            float3 o;
            if (!vol) {
              const DevShader &shd = sc.shaders[shader];
              float bsdf_pdf;
              f = eval_bsdf(shd, h, wi, bins, rough, lambda0, ls.dir, &bsdf_pdf) * fabsf(dot(h.ns, ls.dir));
              const float alpha = guide_prob_bsdf(shd);
              mix_pdf = (1.f - alpha) * gpdf(ls.dir) + alpha * bsdf_pdf;
              maybe_going_through(sc, ntr, ls.dir, h);
              o = offset_origin(h, ls.dir);
            } else {
              float phase_pdf;
              f = medium_phase_eval(sc, vmed, wi, vpos, bins, ls.dir, &phase_pdf);
              float4 ss, st;
              medium_coeffs(sc, vmed, vpos, bins, ss, st);
              f = f * make_float4(ss.x / (st.x + kDblEps), ss.y / (st.y + kDblEps), ss.z / (st.z + kDblEps), ss.w / (st.w + kDblEps));
              mix_pdf = (1.f - kGuideProbPhase) * gpdf(ls.dir) + kGuideProbPhase * phase_pdf;
              o = here;
            }
            const float4 c = thru * f * ls.weight;
            if (!all_zero(c)) {
              q.sh_org[i] = make_float4(o.x, o.y, o.z, ls.len * 0.9999f);
              q.sh_dir[i] = make_float4(ls.dir.x, ls.dir.y, ls.dir.z, ls.delta ? -ls.pdf : ls.pdf);
              q.sh_contrib[i] = c;
              q.sh_aux[i] = make_uint4(ntr.cur, ntr.slots, (uint32_t)as_int(mix_pdf), (uint32_t)nv);
              if (rec) q.sh_nee[i] = f * ls.weight;
              push_shadow = true;
            }
          }
        }
        Scatter s;
        if (!vol) {
          const DevShader &shd = sc.shaders[shader];
          rough = fmaxf(my_roughness(shd), rough);
          if constexpr (kLearned) s = sample_guided(shd, *mixp, h, wi, bins, rough, lambda0, rng);
          else if constexpr (kQuad) s = sample_guided(shd, qg, h, wi, bins, rough, lambda0, rng);
          else s = sample_guided(shd, *cellp, h, wi, bins, rough, lambda0, rng);
        } else {
          if constexpr (kLearned) s = sample_guided_phase(sc, vmed, *mixp, wi, vpos, bins, rng);
          else if constexpr (kQuad) s = sample_guided_phase(sc, vmed, qg, wi, vpos, bins, rng);
          else s = sample_guided_phase(sc, vmed, *cellp, wi, vpos, bins, rng);
        }
        const uint32_t node = (flags & kFlagNodeMask) + 1u;
        bool alive = node <= (uint32_t)sc.max_depth;
        if (alive) {
          const float d = vol ? 1.f : fabsf(dot(h.ns, s.dir));
          thru = (d / s.pdf) * (thru * s.value);
          alive = !all_zero(thru) && isfinite(thru.x + thru.y + thru.z + thru.w);
        }
        int nv_new = nv;
        if (rec && nv < q.max_vertices) {
          // Vertex nv: where the path scattered, into which direction, with which pdf.
          q.gv_pos_pdf[(size_t)nv * cap + i] = make_float4(here.x, here.y, here.z, (alive && !s.delta) ? s.pdf : -1.f);
          q.gv_dir_acc[(size_t)nv * cap + i] = make_float4(s.dir.x, s.dir.y, s.dir.z, 0.f);
          q.gv_thru[(size_t)nv * cap + i] = alive ? thru : f4(0.f);
          if constexpr (kLearned) {
            const float3 n = vol ? mk(0.f, 0.f, 0.f) : h.ns;
            q.gv_nrm[(size_t)nv * cap + i] = make_float4(n.x, n.y, n.z, 0.f);
            q.gv_wo[(size_t)nv * cap + i] = make_float4(wi.x, wi.y, wi.z, 0.f);
          }
          nv_new = nv + 1;
        }
        flags = (flags & ~kFlagVertexMask) | ((uint32_t)nv_new << kFlagVertexShift);
        if (alive) {
          float3 o;
          if (!vol) {
            o = offset_origin(h, s.dir);
            maybe_going_through(sc, tr, s.dir, h);
          } else {
            o = here;
          }
          q.org[i] = make_float4(o.x, o.y, o.z, lambda0);
          q.dir[i] = make_float4(s.dir.x, s.dir.y, s.dir.z, 0.f);
          q.thru[i] = thru;
          q.last_pdf[i] = s.pdf;
          q.roughness[i] = rough;
          flags = (flags & ~(kFlagNodeMask | kFlagLastPdfDelta)) | node | kFlagHasLastPdf | (s.delta ? kFlagLastPdfDelta : 0u);
          push = true;
        } else if (push_shadow) {
          flags |= kFlagFinalizeAfterShadow;
        } else {
          if (rec) emit_records(q, i, nv_new);
          finalize_path(q, fb, fb_sq, i, rad);
        }
        q.flags[i] = flags;
        q.rad[i] = rad;
        q.tracker[i] = make_uint2(tr.cur, tr.slots);
        store_rng(q, i, rng);
      }
    }
    uint32_t slot, sslot;
    block_append2<kTraceBlock / 64>(count_out, push && !q.alive, q.shadow_out, push_shadow, s_cnt, slot, sslot);
    if (q.alive) {
      if (active) q.alive[i] = push ? 1 : 0;
    } else if (push) {
      queue_out[slot] = i;
    }
    if (push_shadow) q.shadow_queue[sslot] = i;
  }
}

// kGuide: 0 the cell's vMF mixture, 1 the learned per-path mixture, 2 the cell's quadtree.
template <int kGuide>
__global__ void __launch_bounds__(256) k_shade_guided(DeviceScene sc, PathQueues q, const uint32_t *__restrict__ queue_in,
                                                      const uint32_t *__restrict__ count_in, uint32_t *__restrict__ queue_out,
                                                      uint32_t *count_out, double *fb, double *fb_sq) {
  __shared__ uint32_t s_idx[256];
  __shared__ uint32_t s_cnt[4][kSortClasses];
  constexpr bool kLearned = kGuide == 1, kQuad = kGuide == 2;
  const uint32_t count = *count_in;
  const bool ident = count_in[kIdentOffset] != 0;
  const bool use_nee = sc.sample_mode != TTGPU_SAMPLE_BSDF;
  const bool use_emission = sc.sample_mode != TTGPU_SAMPLE_LIGHTS;
  const bool mis = use_nee && use_emission;
  const bool rec = sc.guide_record != 0;
  const size_t cap = (size_t)q.capacity;
  const uint32_t n_iter = (count + grid_stride() - 1) / grid_stride();
  for (uint32_t it = 0; it < n_iter; ++it) {
    const uint32_t k = it * grid_stride() + gtid();
    bool active = k < count;
    bool push = false, push_shadow = false;
    uint32_t i = 0;
    if (active) i = ident ? k : queue_in[k];
    if (sc.sort_shade) block_sort_by_class<4>(sc, q, active, i, s_idx, s_cnt);
    if (active) {
      const float4 hitv = q.hit[i];
      const float3 dir = xyz(q.dir[i]);
      const float4 org4 = q.org[i];
      const float lambda0 = org4.w;
      float4 thru = q.thru[i];
      float4 rad = q.rad[i];
      const uint32_t bins = q.bins[i];
      uint32_t flags = q.flags[i];
      const int nv = (int)((flags & kFlagVertexMask) >> kFlagVertexShift);
      const float last_pdf = q.last_pdf[i];
      const bool mis_last = (flags & kFlagHasLastPdf) && !(flags & kFlagLastPdfDelta) && mis;
      Pcg rng = load_rng(q, i);
      const int prim = as_int(hitv.w);
      if (prim < 0) {
        // AddEnvEmission with the power heuristic
        if (use_emission && sc.num_envs > 0) {
          float penv;
          const float4 L = env_eval(sc, -dir, bins, &penv);
          const float w = mis_last ? power_heuristic(last_pdf, penv * sc.type_probs[0]) : 1.f;
          rad = add_rgb(rad, spectral_to_rgb(w * (L * thru), bins));
          if (rec) propagate_radiance(q, i, nv, L, w * L, thru);
        }
        if (rec) emit_records(q, i, nv);
        finalize_path(q, fb, fb_sq, i, rad);
      } else {
        const SurfHit h = make_hit(sc, prim, hitv.y, hitv.z, hitv.x, xyz(org4), dir);
        const DevMaterial mat = sc.materials[h.material];
        // The guide of this vertex: the kd-tree cell's mixture or quadtree, or the learned
        // per-path mixture.
        const GuideCell *cellp = nullptr;
        const nn::Mix16 *mixp = nullptr;
        QuadGuide qg{};
        if constexpr (kLearned) mixp = reinterpret_cast<const nn::Mix16 *>(q.gmix) + i;
        else if constexpr (kQuad) qg = quad_guide(sc, guide_lookup(sc, h.pos));
        else cellp = sc.guide_cells + guide_lookup(sc, h.pos);
        if (use_emission && mat.emitter >= 0) {
          const DevEmitter &em = sc.emitters[mat.emitter];
          if (em.kind == TTGPU_AREA_UNIFORM && dot(h.ng, -dir) > 0.f) {
            const float4 L = take(em.radiance, bins);
            const float p_light = sc.area_pick_prob / sc.prim_area[prim] * area_to_solid_angle(hitv.x, dir, h.n);
            const float w = mis_last ? power_heuristic(last_pdf, p_light) : 1.f;
            rad = add_rgb(rad, spectral_to_rgb(w * (L * thru), bins));
            if (rec) propagate_radiance(q, i, nv, L, w * L, thru);
          }
        }
        const DevShader &shd = sc.shaders[mat.shader];
        float rough = q.roughness[i];
        const float3 wi = -dir;
        // NEE with the selection probability in the light pdf and the power heuristic against the
        // BSDF/guide mixture.
        if (use_nee && (sc.num_area_lights + sc.num_envs + sc.num_points) > 0) {
          const LightSample ls = sample_light(sc, h.pos, h.n, bins, rng);
          if (ls.valid) {
            float bsdf_pdf;
            const float4 f = eval_bsdf(shd, h, wi, bins, rough, lambda0, ls.dir, &bsdf_pdf);
            const float dfac = fabsf(dot(h.ns, ls.dir));
            // The guided integrator always runs with TTGPU_MIS_CONSISTENT, so ls.pdf includes the
            // light-selection probability.
            float w = 1.f;
            if (!ls.delta && mis) {
              float gp;
              if constexpr (kLearned) gp = guided_pdf(shd, *mixp, ls.dir, bsdf_pdf);
              else if constexpr (kQuad) gp = guided_pdf(shd, qg, ls.dir, bsdf_pdf);
              else gp = guided_pdf(shd, *cellp, ls.dir, bsdf_pdf);
              w = power_heuristic(ls.pdf, gp);
            }
            const float4 nee = (w * dfac) * (f * ls.weight);
            const float3 crgb = spectral_to_rgb(thru * nee, bins);
            if (crgb.x != 0.f || crgb.y != 0.f || crgb.z != 0.f) {
              const float3 o = offset_origin(h, ls.dir);
              q.sh_org[i] = make_float4(o.x, o.y, o.z, ls.len * 0.9999f);
              q.sh_dir[i] = make_float4(ls.dir.x, ls.dir.y, ls.dir.z, as_float(nv));
              q.sh_contrib[i] = make_float4(crgb.x, crgb.y, crgb.z, 0.f);
              if (rec) q.sh_nee[i] = nee;
              push_shadow = true;
            }
          }
        }
        rough = fmaxf(my_roughness(shd), rough);
        Scatter s;
        if constexpr (kLearned) s = sample_guided(shd, *mixp, h, wi, bins, rough, lambda0, rng);
        else if constexpr (kQuad) s = sample_guided(shd, qg, h, wi, bins, rough, lambda0, rng);
        else s = sample_guided(shd, *cellp, h, wi, bins, rough, lambda0, rng);
        const uint32_t node = (flags & kFlagNodeMask) + 1u;
        bool alive = node <= (uint32_t)sc.max_depth;
        if (alive) {
          thru = (fabsf(dot(h.ns, s.dir)) / s.pdf) * (thru * s.value);
          alive = !all_zero(thru) && isfinite(thru.x + thru.y + thru.z + thru.w);
        }
        int nv_new = nv;
        if (rec && nv < q.max_vertices) {
          // Vertex nv: where the path scattered, into which direction, with which pdf.
          q.gv_pos_pdf[(size_t)nv * cap + i] = make_float4(h.pos.x, h.pos.y, h.pos.z, (alive && !s.delta) ? s.pdf : -1.f);
          q.gv_dir_acc[(size_t)nv * cap + i] = make_float4(s.dir.x, s.dir.y, s.dir.z, 0.f);
          q.gv_thru[(size_t)nv * cap + i] = alive ? thru : f4(0.f);
          if constexpr (kLearned) {
            q.gv_nrm[(size_t)nv * cap + i] = make_float4(h.ns.x, h.ns.y, h.ns.z, 0.f);
            q.gv_wo[(size_t)nv * cap + i] = make_float4(wi.x, wi.y, wi.z, 0.f);
          }
          nv_new = nv + 1;
        }
        flags = (flags & ~kFlagVertexMask) | ((uint32_t)nv_new << kFlagVertexShift);
        if (alive) {
          const float3 o = offset_origin(h, s.dir);
          q.org[i] = make_float4(o.x, o.y, o.z, lambda0);
          q.dir[i] = make_float4(s.dir.x, s.dir.y, s.dir.z, 0.f);
          q.thru[i] = thru;
          q.last_pdf[i] = s.pdf;
          q.roughness[i] = rough;
          flags = (flags & ~(kFlagNodeMask | kFlagLastPdfDelta)) | node | kFlagHasLastPdf | (s.delta ? kFlagLastPdfDelta : 0u);
          push = true;
        } else if (push_shadow) {
          flags |= kFlagFinalizeAfterShadow;
        } else {
          if (rec) emit_records(q, i, nv_new);
          finalize_path(q, fb, fb_sq, i, rad);
        }
        q.flags[i] = flags;
        q.rad[i] = rad;
        store_rng(q, i, rng);
      }
    }
    uint32_t slot, sslot;
    block_append2<4>(count_out, push && !q.alive, q.shadow_out, push_shadow, s_cnt, slot, sslot);
    if (q.alive) {
      if (active) q.alive[i] = push ? 1 : 0;
    } else if (push) {
      queue_out[slot] = i;
    }
    if (push_shadow) q.shadow_queue[sslot] = i;
  }
}

// A guided path's shadow ray has been traced: unoccluded NEE goes to the radiance and, when
// recording, to the earlier vertices' records; a path that ended at this vertex emits its records
// and is finalized.
__device__ void shadow_done_guided(const DeviceScene &sc, const PathQueues &q, uint32_t i, bool occluded, double *fb, double *fb_sq) {
  const bool rec = sc.guide_record != 0;
  const size_t cap = (size_t)q.capacity;
  float4 rad = q.rad[i];
  const uint32_t flags = q.flags[i];
  if (!occluded) {
    rad = add_rgb(rad, xyz(q.sh_contrib[i]));
    if (rec) {
      const int v = as_int(q.sh_dir[i].w);
      if (v > 0) {
        const float4 nee = q.sh_nee[i];
        propagate_radiance(q, i, v, nee, nee, q.gv_thru[(size_t)(v - 1) * cap + i]);
      }
    }
  }
  if (flags & kFlagFinalizeAfterShadow) {
    if (rec) emit_records(q, i, (int)((flags & kFlagVertexMask) >> kFlagVertexShift));
    finalize_path(q, fb, fb_sq, i, rad);
  } else {
    q.rad[i] = rad;
  }
}

__global__ void __launch_bounds__(kTraceBlock) k_shadow_guided(DeviceScene sc, PathQueues q, double *fb, double *fb_sq, uint32_t *stats) {
  __shared__ int lds_stack[kLdsStack * kTraceBlock];
  const uint32_t count = *q.shadow_out;
  for (uint32_t k = gtid(); k < count; k += grid_stride()) {
    const uint32_t i = q.shadow_queue[k];
    const float4 o = q.sh_org[i];
    const float4 d4 = q.sh_dir[i];
    Ray r;
    r.org = xyz(o);
    r.dir = xyz(d4);
    r.tmax = o.w;
    HitRec h;
    const bool occ = traverse<true>(sc.nodes, sc.prims_kz, sc.num_prims, r, lds_stack + threadIdx.x, h);
    shadow_done_guided(sc, q, i, occ, fb, fb_sq);
  }
  if (gtid() == 0) atomicAdd(stats + kStatShadow, count);
}

// ---- learned guide: batched inference over the paths about to be shaded -------------------
// One 64-thread workgroup per tile of the queue: encode (hit position, shading normal, outgoing
// direction), MLP on MFMA, 16-lobe mixture per path into q.gmix.
// Sort keys of the queued paths for inference: the Morton code of the hit point (from the ray and
// its hit distance) on a 2^kInferKeyBits grid per axis, so that a sort puts the queries of
// neighbouring points into the same waves; misses and entries past the queue share the last code and
// so the sort's end (it is stable: what is past the queue stays last).  The sort takes eight bits a
// pass: 24 bits cost the three passes of 19 (six bits per axis and one for the misses) and put closer
// points together.  Keys, sort and inference of a 128 x 128, 1024 spp pass: 19.9 ms with 19 bits, 19.2
// with 22, 19.0 with 24; two passes, of 16 bits: 20.6 with five bits per axis, 19.2 - 19.9 with the top
// 16 of 18.
constexpr int kInferKeyBits = 8;
constexpr uint32_t kInferMissKey = (1u << (3 * kInferKeyBits)) - 1u;
__global__ void __launch_bounds__(256) k_infer_keys(PathQueues q, const uint32_t *__restrict__ queue, const uint32_t *__restrict__ count_ptr,
                                                    uint32_t n, nn::NetView net, uint32_t *__restrict__ keys, uint32_t *__restrict__ vals) {
  const uint32_t count = *count_ptr;
  const bool ident = count_ptr[kIdentOffset] != 0;
  for (uint32_t k = gtid(); k < n; k += grid_stride()) {
    uint32_t key = kInferMissKey, i = 0;
    if (k < count) {
      i = ident ? k : queue[k];
      const float4 hv = q.hit[i];
      const double vt = q.vt ? q.vt[i] : -1.;
      if (vt >= 0. || as_int(hv.w) >= 0) {
        const float t = vt >= 0. ? (float)vt : hv.x;
        const float4 o = q.org[i], d = q.dir[i];
        key = nn::morton<kInferKeyBits>(net, make_float3(o.x + t * d.x, o.y + t * d.y, o.z + t * d.z));
      }
    }
    keys[k] = key;
    vals[k] = i;
  }
}

// `sorted`: `queue` is the Morton-sorted queue (never the identity).
__global__ void __launch_bounds__(nn::kTile) k_guide_infer(DeviceScene sc, PathQueues q, const uint32_t *__restrict__ queue,
                                                          const uint32_t *__restrict__ count_ptr, nn::NetView net, int sorted) {
  // Input tile / second hidden layer (x) and first / third hidden layer (h0): 18 KB per one-wave
  // block, so LDS admits eight blocks per CU.  The outputs go from the accumulators to the
  // mixtures without LDS.
  __shared__ __attribute__((aligned(16))) __bf16 x[nn::kTile * nn::kPitch];
  __shared__ __attribute__((aligned(16))) __bf16 h0[nn::kTile * nn::kPitch];
  const uint32_t count = *count_ptr;
  const bool ident = !sorted && count_ptr[kIdentOffset] != 0;
  const int l = threadIdx.x;
  for (uint32_t tile = blockIdx.x; tile * nn::kTile < count; tile += gridDim.x) {
    const uint32_t k = tile * nn::kTile + l;
    uint32_t i = 0;
    bool hit = false;
    // Lanes without a query encode the grid's corner (their outputs are never stored): one
    // encoding per lane, not one per kind of query in the wave.
    float3 pos = mk(net.bb_lo[0], net.bb_lo[1], net.bb_lo[2]), nrm = mk(0.f, 0.f, 0.f), wo = mk(0.f, 0.f, 1.f);
    if (k < count) {
      i = ident ? k : queue[k];
      const float4 hv = q.hit[i];
      const int prim = as_int(hv.w);
      const double vt = q.vt ? q.vt[i] : -1.;
      if (vt >= 0.) {
        // A volume collision (media scenes): the point along the ray, no normal.
        const float3 dir = xyz(q.dir[i]);
        pos = f3(d3_along(d3(xyz(q.org[i])), dir, vt));
        wo = -dir;
        hit = true;
      } else if (prim >= 0) {
        const float3 dir = xyz(q.dir[i]);
        const SurfHit h = make_hit(sc, prim, hv.y, hv.z, hv.x, xyz(q.org[i]), dir);
        pos = h.pos;
        nrm = h.ns;
        wo = -dir;
        hit = true;
      }
    }
    nn::encode_row(net, pos, nrm, wo, x + l * nn::kPitch);
    nn::hidden_layers(net, x, h0, x, nullptr, 0, 0);
    nn::output_mixtures(net, h0, i, hit, reinterpret_cast<nn::Mix16 *>(q.gmix));
    __syncthreads();
  }
}

// ---- ray queries -----------------------------------------------------------------------
// A chunk's rays from page-locked host memory to device memory, 16 B per lane.  Bound by the host
// link; k_trace_rays itself reads 4 B of every 12, and reading the host's copy that way costs more
// than the copy (a million occlusion rays: 2.2 ms, against the figure at QueryRays).
__global__ void __launch_bounds__(256) k_copy_rays(uint4 *to, const uint4 *from, uint32_t n_vec, uint32_t n_val, uint32_t dir_at, uint32_t tmax_at) {
  const uint32_t total = 2 * n_vec + n_val;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
    const uint32_t k = i < n_vec ? i : i < 2 * n_vec ? dir_at + (i - n_vec) : tmax_at + (i - 2 * n_vec);
    to[k] = from[k];
  }
}

__global__ void __launch_bounds__(kTraceBlock) k_trace_rays(DeviceScene sc, int64_t n, const float *org, const float *dir, const float *tmax,
                                                            float *t, int32_t *prim, float *u, float *v, int32_t *occl, int brute) {
  __shared__ int lds_stack[kLdsStack * kTraceBlock];
  for (int64_t i = gtid(); i < n; i += grid_stride()) {
    Ray r;
    r.org = mk(org[3 * i], org[3 * i + 1], org[3 * i + 2]);
    r.dir = mk(dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]);
    r.tmax = tmax[i];
    HitRec h;
    if (brute) {
      // Every primitive, no BVH: the reference the traversal is checked against.
      RayPre p = precompute(r);
      float best = r.tmax;
      int bi = -1;
      float bu = 0.f, bv = 0.f;
      for (int k = 0; k < sc.num_prims; ++k) {
        float tt, uu, vv;
        if (intersect_prim(sc.prims[k], p, r, best, tt, uu, vv)) { best = tt; bi = k; bu = uu; bv = vv; }
      }
      t[i] = bi >= 0 ? best : as_float(0x7f800000);
      prim[i] = bi >= 0 ? as_int(sc.prims[bi].a.w) : -1;
      u[i] = bu;
      v[i] = bv;
    } else if (occl) {
      occl[i] = traverse<true>(sc.nodes, sc.prims_kz, sc.num_prims, r, lds_stack + threadIdx.x, h) ? 1 : 0;
    } else {
      bool any = traverse<false>(sc.nodes, sc.prims_kz, sc.num_prims, r, lds_stack + threadIdx.x, h);
      t[i] = any ? h.t : as_float(0x7f800000);
      prim[i] = any ? as_int(sc.prims[h.prim].a.w) : -1;
      u[i] = any ? h.u : 0.f;
      v[i] = any ? h.v : 0.f;
    }
  }
}

__global__ void k_sample_shader(DevShader s, float3 wi, float3 ng, float3 ns, uint32_t bins, float rough, uint64_t seed, int64_t n,
                                float *out_dir, float *out_val, float *out_pdf) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) {
    Pcg rng;
    rng.seed(seed, (uint64_t)i);
    SurfHit h;
    h.pos = mk(0.f, 0.f, 0.f);
    h.ng = h.n = ng;
    h.ns = ns;
    h.offset = 0.f;
    h.material = 0;
    h.prim = 0;
    Scatter sc = sample_bsdf(s, h, wi, bins, rough, 370.f + 10.f * (bins & 0xFF) + 5.f, rng);
    out_dir[3 * i] = sc.dir.x; out_dir[3 * i + 1] = sc.dir.y; out_dir[3 * i + 2] = sc.dir.z;
    out_val[4 * i] = sc.value.x; out_val[4 * i + 1] = sc.value.y; out_val[4 * i + 2] = sc.value.z; out_val[4 * i + 3] = sc.value.w;
    out_pdf[i] = sc.delta ? -sc.pdf : sc.pdf;
  }
}

__global__ void k_eval_shader(DevShader s, float3 wi, float3 ng, float3 ns, uint32_t bins, float rough, int64_t n, const float *dirs,
                              float *out_val, float *out_pdf) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) {
    SurfHit h;
    h.pos = mk(0.f, 0.f, 0.f);
    h.ng = h.n = ng;
    h.ns = ns;
    h.offset = 0.f;
    h.material = 0;
    h.prim = 0;
    float pdf;
    float4 v = eval_bsdf(s, h, wi, bins, rough, 370.f + 10.f * (bins & 0xFF) + 5.f, mk(dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]), &pdf);
    out_val[4 * i] = v.x; out_val[4 * i + 1] = v.y; out_val[4 * i + 2] = v.z; out_val[4 * i + 3] = v.w;
    out_pdf[i] = pdf;
  }
}

__global__ void k_sample_phase(int kind, float g, float3 wi, uint64_t seed, int64_t n, float *out_dir, float *out_val, float *out_pdf) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) {
    Pcg rng;
    rng.seed(seed, (uint64_t)i);
    float3 d;
    float v;
    phase_sample(kind, g, wi, rng, d, v);
    out_dir[3 * i] = d.x; out_dir[3 * i + 1] = d.y; out_dir[3 * i + 2] = d.z;
    out_val[i] = v;
    out_pdf[i] = v;
  }
}

__global__ void k_sample_phase_mix(PhaseMix m, float3 wi, uint64_t seed, int64_t n, float *out_dir, float *out_val, float *out_pdf) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) {
    Pcg rng;
    rng.seed(seed, (uint64_t)i);
    float3 d;
    float4 v;
    float p;
    phase_mix_sample(m, wi, rng, d, v, p);
    out_dir[3 * i] = d.x; out_dir[3 * i + 1] = d.y; out_dir[3 * i + 2] = d.z;
    out_val[4 * i] = v.x; out_val[4 * i + 1] = v.y; out_val[4 * i + 2] = v.z; out_val[4 * i + 3] = v.w;
    out_pdf[i] = p;
  }
}

// Volume-boundary crossings along each ray from its initial tracker state: the distance of
// every crossing and the current medium after it (nullpath::Tracking's segment walk,
// media_integrator.cxx:330-376, without the collisions).
__global__ void k_media_events(DeviceScene sc, int64_t n, const float *org, const float *dir, const float *tmax,
                               const uint64_t *init, int max_events, double *out_t, int32_t *out_medium, int32_t *out_count) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) {
    Tracker tr{(uint32_t)init[i], (uint32_t)(init[i] >> 32)};
    const float3 o = mk(org[3 * i], org[3 * i + 1], org[3 * i + 2]), d = mk(dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]);
    double tnear = 0.;
    int k = 0;
    while (k < max_events) {
      BoundaryHits bh;
      next_boundaries(sc, o, d, tnear, (double)tmax[i], bh);
      if (!bh.n) break;
      cross_boundaries(sc, tr, bh, o, d);
      out_t[i * max_events + k] = bh.t;
      out_medium[i * max_events + k] = tr.cur == (uint32_t)kVacuum ? -1 : (int32_t)tr.cur;
      tnear = bh.t;
      ++k;
    }
    out_count[i] = k;
  }
}

__global__ void k_pcg32(uint64_t initstate, uint64_t initseq, int64_t n, uint32_t *out) {
  if (gtid() != 0) return;
  Pcg rng;
  rng.seed(initstate, initseq);
  for (int64_t i = 0; i < n; ++i) out[i] = rng.next();
}

__global__ void k_guide_sample(GuideCell c, uint64_t seed, int64_t n, float *out_dir, float *out_pdf) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) {
    Pcg rng;
    rng.seed(seed, (uint64_t)i);
    const float u0 = rng.uniform(), u1 = rng.uniform(), u2 = rng.uniform();
    const float3 d = guide_sample(c, u0, u1, u2);
    out_dir[3 * i] = d.x; out_dir[3 * i + 1] = d.y; out_dir[3 * i + 2] = d.z;
    out_pdf[i] = guide_pdf(c, d);
  }
}
__global__ void k_guide_pdf(GuideCell c, int64_t n, const float *dirs, float *out_pdf) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) out_pdf[i] = guide_pdf(c, mk(dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]));
}

// Quadtree warp of given uniforms (2 per sample): the square point, the direction and its pdf.
__global__ void k_quad_sample(QuadGuide g, int64_t n, const float *u, float *out_uv, float *out_dir, float *out_pdf) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) {
    const float2 p = quad_warp(g, u[2 * i], u[2 * i + 1]);
    const float3 d = quad_square_to_sphere(p.x, p.y);
    out_uv[2 * i] = p.x; out_uv[2 * i + 1] = p.y;
    out_dir[3 * i] = d.x; out_dir[3 * i + 1] = d.y; out_dir[3 * i + 2] = d.z;
    out_pdf[i] = guide_pdf(g, d);
  }
}
__global__ void k_quad_pdf(QuadGuide g, int64_t n, const float *dirs, float *out_pdf) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) out_pdf[i] = guide_pdf(g, mk(dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]));
}

// Density of the handle's uploaded guide at positions / directions (cell lookup + the cell's
// vMF mixture or quadtree), as the guided shade kernel evaluates it.
__global__ void k_guide_pdf_at(DeviceScene sc, int64_t n, const float *pos, const float *dirs, float *out_pdf) {
  for (int64_t i = gtid(); i < n; i += grid_stride()) {
    const float3 p = mk(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]);
    const float3 d = mk(dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]);
    const int cell = guide_lookup(sc, p);
    out_pdf[i] = sc.guide_qcells ? guide_pdf(quad_guide(sc, cell), d) : guide_pdf(sc.guide_cells[cell], d);
  }
}

// ---- bdpt: bidirectional path tracing (renderingalgorithms_pathtracing.hxx:341-700) ----------
// Eye and light subpaths on the random-walk framework, then every strategy of
// BdptWorker::RenderPixel: each camera / scatter vertex of the eye subpath connects to a fresh light
// sample and to the light subpath's vertices 1..; eye vertices on emitters count as light hits;
// connections from the camera are splatted to their pixel.  MIS: the power heuristic over all
// strategies of the full path, strategies with >= 2 eye vertices weighted by 1 / pixel count,
// strategies next to a delta vertex excluded; every density is that of the connection at hand (FP64
// products).  Surfaces in vacuum, pinhole camera.
//
// Three kernels per chunk of samples.  k_bdpt_walk (one thread per sample) walks both subpaths,
// writes their vertices, counts the light hits and lists the connections; k_bdpt_connect takes one
// connection per thread, so that the few samples with many connections do not hold a wave;
// k_bdpt_finish adds the samples to their pixels.  Each vertex carries the products of the densities
// before it and the summed squares of the strategies that connect earlier on its subpath, so a
// connection's MIS weight takes a dozen FP64 operations instead of a product per strategy.  As one
// kernel with private arrays (5.9 KB of scratch per lane, 232 registers, 23 % of the lanes active, 72
// % of the wave cycles waiting) 262,144 samples of the Cornell box took 4.75 ms; these
// take 0.55 + 0.63 + 0.01 ms (0.54 + 0.78 + 0.03 with the connections listed sample by sample, the camera
// vertex and each subpath's last one kept in memory and a thread and six atomics per sample at the end,
// which made frames of short paths slower than the one kernel: 1 M samples of a lit wall 0.77 ms against
// 0.55, now 0.47).
enum { kBvCamera = 0, kBvSurf = 1, kBvArea = 2, kBvEnv = 3, kBvPoint = 4 };

struct BdptVertex {
  SurfHit h;     // kBvSurf / kBvArea: surface; kBvEnv: h.pos = direction the light travels; kBvPoint: h.pos
  float3 wi;     // kBvSurf: direction of the ray that arrived
  float4 beta;   // path weight
  float4 Le;     // kBvArea / kBvEnv radiance, kBvPoint intensity
  float pdf_walk;   // density of this vertex from its own subpath's side
  int type;
  int delta;     // the walk left this vertex through a delta lobe
  // MIS over the strategies that connect within the subpath 0 .. this vertex (index n):
  double prod;   // product of the subpath's densities pdf_walk[0 .. n]
  double sum;    // sum over j <= n - 1 of (w_j prod[j - 1] x the opposite side's densities of j .. n - 2)^2,
                 // j vertices on the subpath's own side, skipping j next to a delta vertex
};

// A vertex in memory: six float4 in the order of BdptVertex's parts.
constexpr int kBdptRows = 6;
enum { kBdptEye = 0, kBdptLight = 1, kBdptDirect = 2 };
__device__ __forceinline__ float4 *bdpt_row(const BdptWork &w, int kind, int k, uint32_t s) {
  return w.verts + ((size_t)(kind * w.max_nodes + k) * w.capacity + s) * kBdptRows;
}
// type in bits 0-2, delta bit 3, n = -ng bit 4, material from bit 5.
__device__ __forceinline__ int bdpt_meta(const BdptVertex &v) {
  const bool flip = (v.type == kBvSurf) && (v.h.n.x != v.h.ng.x || v.h.n.y != v.h.ng.y || v.h.n.z != v.h.ng.z);
  return v.type | (v.delta << 3) | ((flip ? 1 : 0) << 4) | (v.type == kBvSurf ? v.h.material << 5 : 0);
}
__device__ __forceinline__ float4 pack_doubles(double a, double b) {
  return make_float4(as_float(__double2loint(a)), as_float(__double2hiint(a)), as_float(__double2loint(b)), as_float(__double2hiint(b)));
}
__device__ __forceinline__ double unpack_double(float lo, float hi) { return __hiloint2double(as_int(hi), as_int(lo)); }
__device__ __forceinline__ void bdpt_store(const BdptWork &w, int kind, int k, uint32_t s, const BdptVertex &v) {
  float4 *r = bdpt_row(w, kind, k, s);
  r[0] = make_float4(v.h.pos.x, v.h.pos.y, v.h.pos.z, v.h.offset);
  r[1] = make_float4(v.h.ng.x, v.h.ng.y, v.h.ng.z, as_float(bdpt_meta(v)));
  if (kind == kBdptDirect) {
    r[2] = v.Le;
  } else {
    r[2] = make_float4(v.h.ns.x, v.h.ns.y, v.h.ns.z, 0.f);
    r[3] = make_float4(v.wi.x, v.wi.y, v.wi.z, 0.f);
  }
  r[4] = v.beta;
  r[5] = pack_doubles(v.prod, v.sum);
}
// The eye subpath's first vertex is the same for every sample, and not kept in memory.
__device__ __forceinline__ BdptVertex bdpt_camera(const DeviceScene &sc) {
  BdptVertex v{};
  v.type = kBvCamera;
  v.h.pos = sc.cam.pos;
  v.beta = f4((float)kStrata);
  v.pdf_walk = 1.f;
  v.prod = 1.;
  return v;
}
__device__ __forceinline__ void bdpt_unpack_geometry(const float4 *r, BdptVertex &v) {
  const float4 a = r[0], b = r[1];
  const int meta = as_int(b.w);
  v.h.pos = xyz(a);
  v.h.offset = a.w;
  v.h.ng = xyz(b);
  v.type = meta & 7;
  v.delta = (meta >> 3) & 1;
  v.h.n = (meta >> 4) & 1 ? -v.h.ng : v.h.ng;
  v.h.material = meta >> 5;
}
__device__ __forceinline__ void bdpt_load(const BdptWork &w, int kind, int k, uint32_t s, BdptVertex &v) {
  const float4 *r = bdpt_row(w, kind, k, s);
  bdpt_unpack_geometry(r, v);
  const float4 c = r[2], d = r[3], f = r[5];
  if (kind == kBdptDirect) {
    v.Le = c;
    v.h.ns = v.h.ng;
  } else {
    v.h.ns = xyz(c);
    v.wi = xyz(d);
  }
  v.beta = r[4];
  v.prod = unpack_double(f.x, f.y);
  v.sum = unpack_double(f.z, f.w);
}

struct BdptCtx {
  const DeviceScene &sc;
  uint32_t bins;
  float lambda0;
  bool consistent_rr;
  float inv_npix;
};

__device__ __forceinline__ bool bv_surface(const BdptVertex &v) { return v.type == kBvSurf || v.type == kBvArea; }
// PdfConversionFactor (rendering_randomwalk_impl.hxx:495-515)
__device__ __forceinline__ float bv_conv(const BdptVertex &src, const BdptVertex &dst, float3 dir, float len) {
  float f = bv_surface(dst) ? fabsf(dot(dst.h.ng, dir)) : 1.f;
  if (src.type != kBvEnv && dst.type != kBvEnv) f /= len * len;
  return f;
}
// BsdfCorrectionFactor (:651-657) times the cosine at the vertex.
__device__ __forceinline__ float bv_corr(const BdptVertex &v, float3 out, bool importance) {
  const float3 l = importance ? -v.wi : out;
  return fabsf(dot(v.h.ns, l)) / (fabsf(dot(v.h.ng, l)) + 1e-20f) * fabsf(dot(v.h.ng, out));
}
__device__ __forceinline__ float bv_emission_pdf(const BdptCtx &c, const BdptVertex &v, float3 out) {
  if (v.type == kBvArea) return dot(v.h.ng, out) > 0.f ? 1.f / (2.f * kPi) : 0.f;
  if (v.type == kBvPoint) return 1.f / (4.f * kPi);
  if (v.type == kBvEnv) return 1.f / (kPi * 0.25f * c.sc.bb_diag * c.sc.bb_diag);
  return 0.f;
}
// Segment between vertices with anti-self-intersection offsets at surface ends.
__device__ __forceinline__ void bv_segment(const BdptCtx &c, const BdptVertex &a, const BdptVertex &b, float3 &org, float3 &dir,
                                           float &len) {
  const float far = 10.f * c.sc.bb_diag;
  if (b.type == kBvEnv) {
    dir = -b.h.pos;
    len = far;
    org = a.type == kBvSurf ? offset_origin(a.h, dir) : a.h.pos;
    return;
  }
  if (a.type == kBvEnv) {
    dir = a.h.pos;
    len = far;
    org = b.h.pos - dir * len;
    return;
  }
  float3 d = b.h.pos - a.h.pos;
  float l = length(d);
  d = l > 0.f ? d * (1.f / l) : mk(1.f, 0.f, 0.f);
  const float3 pa = a.type == kBvSurf ? offset_origin(a.h, d) : a.h.pos;
  const float3 pb = bv_surface(b) ? offset_origin(b.h, -d) : b.h.pos;
  d = pb - pa;
  len = length(d);
  dir = len > 0.f ? d * (1.f / len) : mk(1.f, 0.f, 0.f);
  org = pa;
}

// SampleEmissiveEnd: light start vertex and its density; pos_delta for point lights.
__device__ bool bv_sample_light(const BdptCtx &c, Pcg &rng, BdptVertex &v, bool &pos_delta) {
  const DeviceScene &sc = c.sc;
  const float u_type = rng.uniform(), u_idx = rng.uniform();
  int kind = 3;
  {
    float r = u_type;
    while (kind > 0 && r >= sc.type_probs[kind]) { r -= sc.type_probs[kind]; --kind; }
  }
  pos_delta = false;
  v.delta = 0;
  if (kind == 1 && sc.num_area_lights > 0) {
    const uint32_t li = min((uint32_t)(u_idx * sc.num_area_lights), (uint32_t)sc.num_area_lights - 1u);
    const int lp = sc.area_lights[li];
    const PrimRecord pr = sc.prims[lp];
    const float r0 = rng.uniform(), r1 = rng.uniform();
    if (as_int(pr.b.w) == 0) {
      const float3 v0 = xyz(pr.a), v1 = xyz(pr.b), v2 = xyz(pr.c);
      const float sq = sqrtf(r0);
      const float b0 = 1.f - sq, b1 = (1.f - r1) * sq, b2 = r1 * sq;
      v.h.pos = v0 * b0 + v1 * b1 + v2 * b2;
      v.h.ng = normalize(cross(v1 - v0, v2 - v0));
      const float g7 = 7.f * kFltEps * 0.5f / (1.f - 7.f * kFltEps * 0.5f);
      const float3 e = mk(fabsf(v0.x * b0) + fabsf(v1.x * b1) + fabsf(v2.x * b2), fabsf(v0.y * b0) + fabsf(v1.y * b1) + fabsf(v2.y * b2),
                          fabsf(v0.z * b0) + fabsf(v1.z * b1) + fabsf(v2.z * b2)) * g7;
      v.h.offset = e.x * fabsf(v.h.ng.x) + e.y * fabsf(v.h.ng.y) + e.z * fabsf(v.h.ng.z);
    } else {
      v.h.ng = to_uniform_sphere(r0, r1);
      v.h.pos = xyz(pr.a) + v.h.ng * pr.b.x;
      const float g5 = 5.f * kFltEps * 0.5f / (1.f - 5.f * kFltEps * 0.5f);
      v.h.offset = (fabsf(v.h.pos.x) * fabsf(v.h.ng.x) + fabsf(v.h.pos.y) * fabsf(v.h.ng.y) + fabsf(v.h.pos.z) * fabsf(v.h.ng.z)) * g5;
    }
    v.h.n = v.h.ng;
    v.h.ns = v.h.ng;
    v.h.prim = lp;
    v.h.material = sc.prim_material[lp];
    v.type = kBvArea;
    const DevEmitter &em = sc.emitters[sc.materials[v.h.material].emitter];
    v.Le = em.kind == TTGPU_AREA_UNIFORM ? take(em.radiance, c.bins) : f4(0.f);
    v.pdf_walk = sc.area_pick_prob / sc.prim_area[lp];
    return true;
  }
  if (kind == 0 && sc.num_envs > 0) {
    float3 dout;
    float p;
    bool delta;
    env_sample(sc, c.bins, rng, dout, v.Le, p, delta);
    v.type = kBvEnv;
    v.h.pos = dout;
    v.pdf_walk = sc.type_probs[0] * p;
    pos_delta = delta;
    return true;
  }
  if (kind == 2 && sc.num_points > 0) {
    const uint32_t li = min((uint32_t)(u_idx * sc.num_points), (uint32_t)sc.num_points - 1u);
    const DevPointLight &pl = sc.points[li];
    v.type = kBvPoint;
    v.h.pos = pl.pos;
    v.Le = take(pl.intensity, c.bins);
    v.pdf_walk = sc.type_probs[2] / sc.num_points;
    pos_delta = true;
    return true;
  }
  return false;
}

__device__ __forceinline__ float bv_scatter_pdf(const BdptCtx &c, const BdptVertex &v, float3 in, float3 out, bool importance) {
  float pdf = 0.f;
  eval_bsdf(c.sc.shaders[c.sc.materials[v.h.material].shader], v.h, in, c.bins, 0.f, c.lambda0, out, &pdf, importance);
  return pdf;
}

__device__ __forceinline__ double sq(double x) { return x * x; }

// BdptForwardTrace (:598-646) from `cur`, the subpath's first vertex (index 0, already stored), with
// the sampled direction `dir`; stores the vertices and returns their number.  Eye subpaths add their
// light hits (HandleLightHit, :526-556) to `acc`.
template <bool kLight>
__device__ int bv_walk(const BdptCtx &c, const BdptWork &w, uint32_t s, BdptVertex cur, float3 org, float3 dir, float pdf, float4 factor,
                       bool light_delta, Pcg &rng, int *lds_stack, uint32_t &rays, float4 &acc) {
  const DeviceScene &sc = c.sc;
  constexpr int kKind = kLight ? kBdptLight : kBdptEye;
  BdptVertex prev;
  int n = 1;
  float carry = 1.f;
  bool pdf_delta = false;
  const double inv = c.inv_npix;
  for (;;) {
    if (all_zero(factor) || !(pdf > 0.f) || !isfinite(factor.x + factor.y + factor.z + factor.w)) return n;
    Ray r;
    r.org = org;
    r.dir = dir;
    r.tmax = 3.0e38f;
    HitRec hr;
    ++rays;
    const bool hit = traverse<false>(sc.nodes, sc.prims_kz, sc.num_prims, r, lds_stack, hr);
    if (!hit && (kLight || sc.num_envs == 0)) return n;  // light subpaths end at the environment
    if (pdf_delta) {
      cur.delta = 1;
      bdpt_row(w, kKind, n - 1, s)[1].w = as_float(bdpt_meta(cur));
    }
    factor = carry * factor;
    carry = 1.f;
    bool survive = n + 1 < w.max_nodes;
    if (survive && n + 1 > 5) {
      const float ps = fminf(0.9f, fmaxf(fmaxf(factor.x, factor.y), fmaxf(factor.z, factor.w)));
      if (rng.uniform() > ps) survive = false;
      else if (c.consistent_rr) carry = 1.f / ps;
      else factor = factor * (1.f / ps);
    }
    BdptVertex v;
    v.beta = cur.beta * factor;
    v.delta = 0;
    float penv = 0.f;
    if (!hit) {
      v.type = kBvEnv;
      v.h.pos = -dir;
      v.Le = env_eval(sc, -dir, c.bins, &penv);
      v.pdf_walk = pdf;
    } else {
      v.type = kBvSurf;
      v.h = make_hit(sc, hr.prim, hr.u, hr.v, hr.t, org, dir);
      v.wi = dir;
      v.pdf_walk = pdf * bv_conv(cur, v, dir, hr.t);
    }
    // The opposite side's density of vertex n - 2, now that the scatter at n - 1 is known, and the
    // sums of the strategies that connect earlier.
    if (n >= 2) {
      const float rp = pdf_delta ? pdf : bv_scatter_pdf(c, cur, dir, -cur.wi, kLight);
      float3 o, d;
      float len;
      bv_segment(c, cur, prev, o, d, len);
      const double other = rp * bv_conv(cur, prev, d, len);
      v.sum = cur.sum * sq(other);
      if (!prev.delta && !cur.delta) v.sum += sq((!kLight && n - 1 >= 2 ? inv : 1.) * prev.prod);
    } else {
      v.sum = kLight && !light_delta && !cur.delta ? 1. : 0.;
    }
    v.prod = cur.prod * v.pdf_walk;
    if (v.type == kBvSurf && n + 1 < w.max_nodes) bdpt_store(w, kKind, n, s, v);  // the last vertex connects to nothing
    if constexpr (!kLight) {
      float4 Le = f4(0.f);
      float p_start = 0.f, p_emit = 0.f;
      BdptVertex as_light = v;
      if (v.type == kBvEnv) {
        Le = v.Le;
        p_start = penv * sc.type_probs[0];
        p_emit = bv_emission_pdf(c, v, v.h.pos);
      } else if (sc.materials[v.h.material].emitter >= 0) {
        const DevEmitter &em = sc.emitters[sc.materials[v.h.material].emitter];
        const bool facing = dot(v.h.ng, -v.wi) > 0.f;
        if (em.kind == TTGPU_AREA_UNIFORM && facing) Le = take(em.radiance, c.bins);
        p_start = sc.area_pick_prob / sc.prim_area[v.h.prim];
        as_light.type = kBvArea;
        p_emit = facing ? 1.f / (2.f * kPi) : 0.f;
      }
      if (!all_zero(Le)) {
        float3 o2, d2;
        float l2;
        bv_segment(c, as_light, cur, o2, d2, l2);
        const double pl_prev = (double)p_emit * bv_conv(as_light, cur, d2, l2);
        const double p_hit = sq((n + 1 >= 2 ? inv : 1.) * v.prod);  // all n + 1 vertices from the eye
        double den = p_hit + v.sum * sq(pl_prev * p_start);
        if (!cur.delta) den += sq((n >= 2 ? inv : 1.) * cur.prod * p_start);
        if (den > 0.) acc = acc + (float)(p_hit / den) * (v.beta * Le);
      }
    }
    ++n;
    if (!survive || v.type == kBvEnv) return v.type == kBvEnv ? n - 1 : n;
    const DevShader &shd = sc.shaders[sc.materials[v.h.material].shader];
    const Scatter sct = sample_bsdf(shd, v.h, -v.wi, c.bins, 0.f, c.lambda0, rng, kLight);
    factor = (bv_corr(v, sct.dir, kLight) / sct.pdf) * sct.value;
    pdf = sct.pdf;
    pdf_delta = sct.delta;
    dir = sct.dir;
    org = offset_origin(v.h, sct.dir);
    prev = cur;
    cur = v;
  }
}

// Wavelengths and random numbers of a camera sample (as init_camera_path).
__device__ __forceinline__ BdptCtx bdpt_context(const DeviceScene &sc, Pcg &rng, uint32_t npix) {
  const int main_idx = (int)rng.bounded(kStrata);
  int idx[4] = {main_idx, main_idx + kStrata, main_idx + 2 * kStrata, main_idx + 3 * kStrata};
  const int rot = (int)rng.bounded(4);
  const int t = idx[0]; idx[0] = idx[rot]; idx[rot] = t;
  const float lambda0 = 370.f + 10.f * idx[0] + 10.f * rng.uniform();
  rng.uniform(); rng.uniform(); rng.uniform();
  const uint32_t bins = (uint32_t)idx[0] | ((uint32_t)idx[1] << 8) | ((uint32_t)idx[2] << 16) | ((uint32_t)idx[3] << 24);
  return BdptCtx{sc, bins, lambda0, sc.mis_mode == TTGPU_MIS_CONSISTENT, 1.f / (float)npix};
}

// Sample `first + s` of the pass for every s < count (at most w.capacity).
__global__ void __launch_bounds__(kTraceBlock) k_bdpt_walk(DeviceScene sc, BdptWork w, uint64_t first, uint32_t count, uint32_t npix,
                                                            uint32_t spp_base, uint64_t seed, uint32_t *stats) {
  __shared__ int lds_stack[kLdsStack * kTraceBlock];
  const uint32_t s = gtid();
  uint32_t rays = 0, num = 0;
  int ne = 0, nl = 0;
  uint32_t directs = 0;  // bit e: eye vertex e has a light sample to connect to
  if (s < count) {
    const uint64_t g = first + s;
    const uint32_t pixel = (uint32_t)(g % npix);
    Pcg rng;
    rng.seed(seed, (spp_base + g / npix) * npix + pixel);
    const BdptCtx c = bdpt_context(sc, rng, npix);
    float4 acc = f4(0.f);
    // eye subpath
    {
      const BdptVertex v = bdpt_camera(sc);
      const int px = pixel % sc.cam.width, py = pixel / sc.cam.width;
      const float r0 = rng.uniform(), r1 = rng.uniform();
      float3 dir;
      float pdf_cam;
      camera_ray(sc.cam, px, py, r0, r1, dir, &pdf_cam);
      ne = 1;
      if (w.max_nodes > 1)
        ne = bv_walk<false>(c, w, s, v, sc.cam.pos, dir, pdf_cam, f4(1.f), false, rng, lds_stack + threadIdx.x, rays, acc);
    }
    // light subpath
    bool light_delta = false;
    BdptVertex v{};
    if (bv_sample_light(c, rng, v, light_delta)) {
      v.beta = f4(1.f / v.pdf_walk);
      v.prod = v.pdf_walk;
      v.sum = 0.;
      bdpt_store(w, kBdptLight, 0, s, v);
      nl = 1;
      const float r0 = rng.uniform(), r1 = rng.uniform();
      float3 org, dir;
      float pdf;
      float4 factor;
      if (v.type == kBvArea) {
        const float3 l = to_uniform_hemisphere(r0, r1);
        const Frame fr = make_frame(v.h.ng);
        dir = fr.to_world(l);
        pdf = 1.f / (2.f * kPi);
        factor = (fabsf(dot(v.h.ng, dir)) * 2.f * kPi) * v.Le;
        org = offset_origin(v.h, dir);
      } else if (v.type == kBvPoint) {
        dir = to_uniform_sphere(r0, r1);
        pdf = 1.f / (4.f * kPi);
        factor = (4.f * kPi) * v.Le;
        org = v.h.pos;
      } else {
        // EnvLightPointSamplingBeyondScene (light.cxx:201-219): a disc across the scene's box.
        dir = v.h.pos;
        const float rr = sqrtf(r0), ph = 2.f * kPi * r1;
        float sn, cs;
        fast_sincos(ph, &sn, &cs);
        const Frame fr = make_frame(dir);
        org = sc.bb_center - dir * (10.f * sc.bb_diag) + fr.to_world(mk(rr * cs, rr * sn, 0.f)) * (0.5f * sc.bb_diag);
        pdf = bv_emission_pdf(c, v, dir);
        factor = (1.f / pdf) * v.Le;
      }
      if (w.max_nodes > 1)
        nl = bv_walk<true>(c, w, s, v, org, dir, pdf, factor, light_delta, rng, lds_stack + threadIdx.x, rays, acc);
    }
    // A fresh light sample per eye vertex, and the number of connections.
    for (int e = 0; e < ne && e + 1 < w.max_nodes; ++e) {
      BdptVertex d{};
      bool dl_delta;
      if (bv_sample_light(c, rng, d, dl_delta)) {
        d.beta = f4(1.f / d.pdf_walk);
        d.prod = d.pdf_walk;
        d.sum = 0.;
        d.delta = dl_delta ? 1 : 0;
        bdpt_store(w, kBdptDirect, e, s, d);
        directs |= 1u << e;
        ++num;
      }
      num += (uint32_t)max(0, min(nl, w.max_nodes - e - 1) - 1);
    }
    w.info[s] = make_uint2(c.bins, (uint32_t)as_int(c.lambda0));
    const float3 rgb = spectral_to_rgb(acc, c.bins);
    w.acc[3 * (size_t)s + 0] = rgb.x;
    w.acc[3 * (size_t)s + 1] = rgb.y;
    w.acc[3 * (size_t)s + 2] = rgb.z;
  }
  // The wave's connections, listed with one atomic and by strategy, so that the lanes of a connection wave
  // load neighbouring samples' vertices and mostly agree in what they evaluate.
  uint32_t total = num, longest = (uint32_t)ne;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    total += __shfl_xor(total, o);
    longest = max(longest, (uint32_t)__shfl_xor(longest, o));
  }
  if (total) {
    const int lane = (int)(threadIdx.x & 63);
    uint32_t at = 0;
    if (lane == 0) at = atomicAdd(w.count, total);
    at = __shfl(at, 0);
    const uint64_t below = (1ull << lane) - 1ull;
    for (int e = 0; e < (int)longest && e + 1 < w.max_nodes; ++e)
      for (int l = 0; l < w.max_nodes - e - 1; ++l) {
        const bool mine = l == 0 ? ((directs >> e) & 1u) != 0 : e < ne && l < nl;
        const uint64_t lanes = __ballot(mine);
        if (mine) w.pairs[at + (uint32_t)__popcll(lanes & below)] = s | ((uint32_t)e << 20) | ((uint32_t)l << 25);
        at += (uint32_t)__popcll(lanes);
      }
  }
  wave_stat(stats + kStatClosest, rays);
}

// Connection of an eye vertex with a light vertex (index l >= 1) or with its light sample (l = 0).
__global__ void __launch_bounds__(kTraceBlock) k_bdpt_connect(DeviceScene sc, BdptWork w, uint32_t npix, double *fb, uint32_t *stats) {
  __shared__ int lds_stack[kLdsStack * kTraceBlock];
  const uint32_t count = *w.count;
  const double inv = 1.f / (float)npix;
  uint32_t rays = 0;
  for (uint32_t k = gtid(); k < count; k += grid_stride()) {
    const uint32_t id = w.pairs[k], s = id & 0xfffffu;
    const int e = (int)((id >> 20) & 31u), l = (int)(id >> 25);
    const uint2 info = w.info[s];
    const BdptCtx c{sc, info.x, as_float((int)info.y), false, 1.f / (float)npix};
    BdptVertex a, b;
    if (e == 0) a = bdpt_camera(sc);
    else bdpt_load(w, kBdptEye, e, s, a);
    if (l == 0) bdpt_load(w, kBdptDirect, e, s, b);
    else bdpt_load(w, kBdptLight, l, s, b);
    float3 org, dir;
    float len;
    bv_segment(c, a, b, org, dir, len);
    float4 fa;
    float pa_fwd = 0.f, pa_rev = 0.f;
    int pixel = -1;
    if (a.type == kBvCamera) {
      const DevCamera &cam = sc.cam;
      const float z = dot(dir, cam.dir);
      if (!(z > 0.f)) continue;
      const float x = dot(dir, cam.right) / z, y = dot(dir, cam.up) / z;
      const float fx = (x - cam.xmin) / cam.xper, fy = (y - cam.ymin) / cam.yper;
      const bool trunc = sc.mis_mode != TTGPU_MIS_CONSISTENT;
      const float ix = trunc ? truncf(fx) : floorf(fx), iy = trunc ? truncf(fy) : floorf(fy);
      if (!(ix >= 0.f && ix < (float)cam.width && iy >= 0.f && iy < (float)cam.height)) continue;
      pixel = (int)iy * cam.width + (int)ix;
      pa_fwd = camera_pdf(cam, x, y);
      fa = f4(pa_fwd);
    } else {
      const DevShader &shd = sc.shaders[sc.materials[a.h.material].shader];
      fa = bv_corr(a, dir, false) * eval_bsdf(shd, a.h, -a.wi, c.bins, 0.f, c.lambda0, dir, &pa_fwd);
    }
    float4 fl;
    float pb_fwd = 0.f, pb_rev = 0.f;
    if (b.type == kBvSurf) {
      const DevShader &shd = sc.shaders[sc.materials[b.h.material].shader];
      fl = bv_corr(b, -dir, true) * eval_bsdf(shd, b.h, -b.wi, c.bins, 0.f, c.lambda0, -dir, &pb_fwd, true);
    } else {
      pb_fwd = bv_emission_pdf(c, b, -dir);
      fl = b.type == kBvArea ? (dot(b.h.ng, -dir) > 0.f ? fabsf(dot(b.h.ng, dir)) : 0.f) * b.Le : b.Le;
    }
    const float4 f = fa * fl;
    if (all_zero(f)) continue;
    const float G = b.type == kBvEnv ? 1.f : 1.f / (len * len);
    Ray r;
    r.org = org;
    r.dir = dir;
    r.tmax = len * 0.9999f;
    HitRec hr;
    ++rays;
    if (traverse<true>(sc.nodes, sc.prims_kz, sc.num_prims, r, lds_stack + threadIdx.x, hr)) continue;
    // Strategies of the full path by their number of eye vertices j: up to e - 1 (a.sum), e, this one
    // (e + 1), e + 2, and more (b.sum).
    const double pe_b = (double)pa_fwd * bv_conv(a, b, dir, len), pl_a = (double)pb_fwd * bv_conv(b, a, -dir, len);
    const double mine = sq((e >= 1 ? inv : 1.) * a.prod * b.prod);
    double den = mine;
    if (e >= 1) {
      BdptVertex p = bdpt_camera(sc);
      if (e >= 2) {
        const float4 *row = bdpt_row(w, kBdptEye, e - 1, s);
        bdpt_unpack_geometry(row, p);
        p.prod = unpack_double(row[5].x, row[5].y);
        // a.sum is zero for e < 2: no strategy connects before the first scatter vertex.
        pa_rev = bv_scatter_pdf(c, a, dir, -a.wi, false);
        float3 o2, d2;
        float l2;
        bv_segment(c, a, p, o2, d2, l2);
        den += a.sum * sq((double)pa_rev * bv_conv(a, p, d2, l2) * pl_a * b.prod);
      }
      if (!p.delta) den += sq((e >= 2 ? inv : 1.) * p.prod * pl_a * b.prod);
    }
    if (l >= 1) {
      BdptVertex p;
      const float4 *row = bdpt_row(w, kBdptLight, l - 1, s);
      bdpt_unpack_geometry(row, p);
      const float4 m = row[5];
      if (!p.delta) den += sq(inv * a.prod * pe_b * unpack_double(m.x, m.y));
      if (b.sum > 0.) {
        pb_rev = bv_scatter_pdf(c, b, -dir, -b.wi, true);
        float3 o2, d2;
        float l2;
        bv_segment(c, b, p, o2, d2, l2);
        den += b.sum * sq(inv * a.prod * pe_b * (double)pb_rev * bv_conv(b, p, d2, l2));
      }
    } else if (!b.delta) {
      den += sq(inv * a.prod * pe_b);
    }
    const float wgt = den > 0. ? (float)(mine / den) : 0.f;
    const float4 contrib = (wgt * G) * (a.beta * b.beta * f);
    if (e == 0) {
      const float3 rgb = spectral_to_rgb(c.inv_npix * contrib, c.bins);
      atomicAdd(fb + 3 * (size_t)pixel + 0, (double)rgb.x);
      atomicAdd(fb + 3 * (size_t)pixel + 1, (double)rgb.y);
      atomicAdd(fb + 3 * (size_t)pixel + 2, (double)rgb.z);
    } else {
      const float3 rgb = spectral_to_rgb(contrib, c.bins);
      atomicAdd(w.acc + 3 * (size_t)s + 0, (double)rgb.x);
      atomicAdd(w.acc + 3 * (size_t)s + 1, (double)rgb.y);
      atomicAdd(w.acc + 3 * (size_t)s + 2, (double)rgb.z);
    }
  }
  wave_stat(stats + kStatClosest, rays);
}

// Adds the samples to their pixels: with kPerPixel one thread per pixel of the chunk, without atomics,
// else one thread per sample.
template <bool kPerPixel>
__global__ void __launch_bounds__(256) k_bdpt_finish(BdptWork w, uint64_t first, uint32_t count, uint32_t npix, double *fb, double *fb_sq) {
  const uint32_t k = gtid();
  if (k == 0) *w.count = 0;
  if (k >= min(count, kPerPixel ? npix : count)) return;
  const size_t pixel = (size_t)((first + k) % npix);
  double sum[3] = {0., 0., 0.}, sum_sq[3] = {0., 0., 0.};
  for (uint32_t s = k; s < count; s += kPerPixel ? npix : count) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double v = (double)(float)w.acc[3 * (size_t)s + c];
      sum[c] += v;
      sum_sq[c] += v * v;
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (kPerPixel) {
      fb[3 * pixel + c] += sum[c];
      if (fb_sq) fb_sq[3 * pixel + c] += sum_sq[c];
    } else {
      atomicAdd(fb + 3 * pixel + c, sum[c]);
      if (fb_sq) atomicAdd(fb_sq + 3 * pixel + c, sum_sq[c]);
    }
  }
}

// ---- host-side launchers ------------------------------------------------------------------
hipError_t UploadSpectralTables(const float *to_rgb, const float *smits) {
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_spec_to_rgb), to_rgb, sizeof(float) * 3 * kNBins);
  if (e != hipSuccess) return e;
  return hipMemcpyToSymbol(HIP_SYMBOL(c_smits), smits, sizeof(float) * 7 * kNBins);
}

static int Blocks(uint64_t n, int block, int cap) {
  uint64_t b = (n + block - 1) / block;
  if (b < 1) b = 1;
  return (int)(b > (uint64_t)cap ? cap : b);
}

void LaunchResetCounter(uint32_t *counters, int which, hipStream_t st) {
  hipLaunchKernelGGL(k_reset_counter, dim3(1), dim3(64), 0, st, counters, which);
}
void LaunchFill(double *p, double *p2, size_t n, double v, hipStream_t st) {
  hipLaunchKernelGGL(k_fill_f64, dim3(Blocks(n, 256, 4096)), dim3(256), 0, st, p, p2, n, v);
}
void LaunchRaygen(const DeviceScene &sc, const PathQueues &q, uint32_t count, uint32_t npix, uint32_t spp_base, uint64_t seed,
                  hipStream_t st) {
  hipLaunchKernelGGL(k_raygen, dim3(Blocks(count, 256, 65535)), dim3(256), 0, st, sc, q, count, npix, spp_base, seed);
}
size_t SelectTempBytes(uint32_t capacity) {
  return sizeof(SlotTemp) + 3 * (size_t)((capacity + kSlotBlock - 1) / kSlotBlock) * sizeof(uint32_t);
}

void LaunchRegen(const DeviceScene &sc, const PathQueues &q, const RegenArgs &a, hipStream_t st) {
  if (q.alive) {
    const uint32_t nb = (a.slots + kSlotBlock - 1) / kSlotBlock, per_block = kSlotBlock / 64;
    SlotTemp *tmp = static_cast<SlotTemp *>(a.select_temp);
    hipLaunchKernelGGL(k_slot_select, dim3((nb + per_block - 1) / per_block), dim3(kSlotBlock), 0, st, q, a.slots, nb, tmp, a.count_out,
                       a.limit, a.npix, a.spp_base, a.with_shadow ? 1 : 0, a.host, a.seq);
    hipLaunchKernelGGL(k_slot_scatter, dim3(nb), dim3(kSlotBlock), 0, st, sc, q, a.slots, nb, tmp, a.npix, a.seed, a.queue_out);
    return;
  }
  hipLaunchKernelGGL(k_regen, dim3(Blocks(a.slots, 256, 8192)), dim3(256), 0, st, sc, q, a.queue_out, a.count_out, a.limit, a.npix,
                     a.spp_base, a.seed);
  hipLaunchKernelGGL(k_regen_commit, dim3(1), dim3(64), 0, st, q, a.count_out, a.limit, a.with_shadow ? 1 : 0, a.host, a.seq);
}
void LaunchReport(const PathQueues &q, PassReport *host, hipStream_t st) {
  hipLaunchKernelGGL(k_report, dim3(1), dim3(64), 0, st, q, host);
}
// Blocks of a trace launch: four times what is resident at five waves per SIMD, so that short runs
// (about 100-200 rays of a 4 M-path wavefront) even out at the launch's end; or one wave per 64
// rays when there are fewer.  1080p benchmark with 2560 / 4096 / 5120 / 7680 / 10240 / 16384 blocks:
// 16.8 / 17.7 / 16.5 / 16.1 / 15.9 / 16.0 ms per pass.
constexpr int kTraceGrid = 10240;

void LaunchTrace(const DeviceScene &sc, const PathQueues &q, const uint32_t *queue, const uint32_t *count, uint32_t max_count,
                 double *fb, double *fb_sq, bool with_shadow, hipStream_t st) {
  // With shadow rays, up to max_count of each kind.
  const dim3 grid(Blocks((with_shadow ? 2ull : 1ull) * max_count, kTraceBlock, kTraceGrid)), block(kTraceBlock);
  const bool guided = sc.guide_cells || sc.guide_qcells || q.gmix;
  if (with_shadow && guided) hipLaunchKernelGGL(k_trace<2>, grid, block, 0, st, sc, q, queue, count, q.counters, fb, fb_sq);
  else if (with_shadow) hipLaunchKernelGGL(k_trace<1>, grid, block, 0, st, sc, q, queue, count, q.counters, fb, fb_sq);
  else hipLaunchKernelGGL(k_trace<0>, grid, block, 0, st, sc, q, queue, count, q.counters, fb, fb_sq);
}
void LaunchTrackMedia(const DeviceScene &sc, const PathQueues &q, const uint32_t *queue, const uint32_t *count, uint32_t max_count,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_track_media, dim3(Blocks(max_count, kTraceBlock, 16384)), dim3(kTraceBlock), 0, st, sc, q, queue, count);
}
void LaunchShade(const DeviceScene &sc, const PathQueues &q, const uint32_t *queue_in, const uint32_t *count_in, uint32_t *queue_out,
                 uint32_t *count_out, uint32_t max_count, double *fb, double *fb_sq, hipStream_t st) {
  if (q.vt) {  // guided integrator in a media scene (k_track_media has run)
    const dim3 grid(Blocks(max_count, kTraceBlock, 16384)), block(kTraceBlock);
    if (sc.guide_cells) hipLaunchKernelGGL(k_shade_media_guided<0>, grid, block, 0, st, sc, q, queue_in, count_in, queue_out, count_out, fb, fb_sq);
    else if (sc.guide_qcells) hipLaunchKernelGGL(k_shade_media_guided<2>, grid, block, 0, st, sc, q, queue_in, count_in, queue_out, count_out, fb, fb_sq);
    else hipLaunchKernelGGL(k_shade_media_guided<1>, grid, block, 0, st, sc, q, queue_in, count_in, queue_out, count_out, fb, fb_sq);
    return;
  }
  if (sc.algo_pt)
    hipLaunchKernelGGL(k_shade<true>, dim3(Blocks(max_count, 256, 8192)), dim3(256), 0, st, sc, q, queue_in, count_in, queue_out,
                       count_out, fb, fb_sq);
  else if (sc.guide_cells)
    hipLaunchKernelGGL(k_shade_guided<0>, dim3(Blocks(max_count, 256, 8192)), dim3(256), 0, st, sc, q, queue_in, count_in,
                       queue_out, count_out, fb, fb_sq);
  else if (sc.guide_qcells)
    hipLaunchKernelGGL(k_shade_guided<2>, dim3(Blocks(max_count, 256, 8192)), dim3(256), 0, st, sc, q, queue_in, count_in,
                       queue_out, count_out, fb, fb_sq);
  else if (q.gmix)
    hipLaunchKernelGGL(k_shade_guided<1>, dim3(Blocks(max_count, 256, 8192)), dim3(256), 0, st, sc, q, queue_in, count_in,
                       queue_out, count_out, fb, fb_sq);
  else if (sc.has_media)
    hipLaunchKernelGGL(sc.has_atmosphere ? k_shade_media<true> : k_shade_media<false>, dim3(Blocks(max_count, kTraceBlock, 16384)), dim3(kTraceBlock), 0, st, sc, q, queue_in, count_in,
                       queue_out, count_out, fb, fb_sq);
  else
    hipLaunchKernelGGL(k_shade<false>, dim3(Blocks(max_count, 256, 8192)), dim3(256), 0, st, sc, q, queue_in, count_in, queue_out, count_out,
                       fb, fb_sq);
}
size_t BdptVertexBytes(int max_nodes) { return (size_t)3 * max_nodes * kBdptRows * sizeof(float4); }
void LaunchBdpt(const DeviceScene &sc, const BdptWork &w, uint64_t first, uint32_t count, uint32_t npix, uint32_t spp_base, uint64_t seed,
                double *fb, double *fb_sq, uint32_t *stats, hipStream_t st) {
  if (count == 0) return;
  hipLaunchKernelGGL(k_bdpt_walk, dim3((count + kTraceBlock - 1) / kTraceBlock), dim3(kTraceBlock), 0, st, sc, w, first, count, npix, spp_base,
                     seed, stats);
  hipLaunchKernelGGL(k_bdpt_connect, dim3(Blocks((uint64_t)count * 8, kTraceBlock, 16384)), dim3(kTraceBlock), 0, st, sc, w, npix, fb, stats);
  // A pixel's samples one after the other (0.5 us each) against atomics on rows that others add to as well
  // (0.1 us per thousand samples): equal near 5000 pixels, whatever the chunk.  2^20 samples on 512 x
  // 512 pixels 11 / 107 us, 128 x 128: 35 / 110, 64 x 64: 131 / 117, 16 x 16: 1853 / 271.
  const bool per_pixel = npix >= (1u << 13);
  const uint32_t threads = per_pixel ? std::min(count, npix) : count;
  hipLaunchKernelGGL(per_pixel ? k_bdpt_finish<true> : k_bdpt_finish<false>, dim3((threads + 255) / 256), dim3(256), 0, st, w, first, count,
                     npix, fb, fb_sq);
}
void LaunchCameraConnect(const DeviceScene &sc, uint64_t first, uint64_t count, uint32_t npix, uint32_t spp_base, uint64_t seed,
                         double *fb, double *fb_sq, uint32_t *stats, hipStream_t st) {
  if (count == 0) return;
  hipLaunchKernelGGL(k_camera_connect, dim3(Blocks(count, kConnectBlock, kConnectBlocks)), dim3(kConnectBlock), 0, st, sc, first, count,
                     npix, spp_base, seed, fb, fb_sq, stats);
}
bool ShadowInTrace(const DeviceScene &sc, const PathQueues &q) { return sc.shadow_in_trace && !q.vt && !sc.has_media; }
void LaunchShadow(const DeviceScene &sc, const PathQueues &q, uint32_t max_count, double *fb, double *fb_sq, hipStream_t st) {
  const dim3 grid(Blocks(max_count, kTraceBlock, 16384)), block(kTraceBlock);
  if (sc.has_media)
    hipLaunchKernelGGL(sc.has_atmosphere ? k_shadow_media<true> : k_shadow_media<false>, grid, block, 0, st, sc, q, fb, fb_sq, q.counters);
  else if (sc.guide_cells || sc.guide_qcells || q.gmix)
    hipLaunchKernelGGL(k_shadow_guided, grid, block, 0, st, sc, q, fb, fb_sq, q.counters);
  else
    hipLaunchKernelGGL(k_shadow, grid, block, 0, st, sc, q, fb, fb_sq, q.counters);
}
void LaunchTraceRays(const DeviceScene &sc, int64_t n, const float *org, const float *dir, const float *tmax, float *t, int32_t *prim,
                     float *u, float *v, int32_t *occl, int brute, hipStream_t st) {
  hipLaunchKernelGGL(k_trace_rays, dim3(Blocks(n, kTraceBlock, 16384)), dim3(kTraceBlock), 0, st, sc, n, org, dir, tmax, t, prim, u, v,
                     occl, brute);
}
void LaunchCopyRays(void *to, const void *from, size_t n, size_t stride, hipStream_t st) {
  const uint32_t n_vec = (uint32_t)((12 * n + 15) / 16), n_val = (uint32_t)((4 * n + 15) / 16);
  hipLaunchKernelGGL(k_copy_rays, dim3(Blocks(2 * (size_t)n_vec + n_val, 256, 1024)), dim3(256), 0, st, static_cast<uint4 *>(to),
                     static_cast<const uint4 *>(from), n_vec, n_val, (uint32_t)(12 * stride / 16), (uint32_t)(24 * stride / 16));
}
void LaunchSampleShader(const DevShader &s, float3 wi, float3 ng, float3 ns, uint32_t bins, float rough, uint64_t seed, int64_t n,
                        float *d, float *v, float *p, hipStream_t st) {
  hipLaunchKernelGGL(k_sample_shader, dim3(Blocks(n, 256, 8192)), dim3(256), 0, st, s, wi, ng, ns, bins, rough, seed, n, d, v, p);
}
void LaunchEvalShader(const DevShader &s, float3 wi, float3 ng, float3 ns, uint32_t bins, float rough, int64_t n, const float *dirs,
                      float *v, float *p, hipStream_t st) {
  hipLaunchKernelGGL(k_eval_shader, dim3(Blocks(n, 256, 8192)), dim3(256), 0, st, s, wi, ng, ns, bins, rough, n, dirs, v, p);
}
size_t InferSortTempBytes(uint32_t capacity) {
  size_t bytes = 0;
  (void)hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint32_t *)nullptr, (uint32_t *)nullptr, (const uint32_t *)nullptr,
                                           (uint32_t *)nullptr, (int)capacity, 0, 3 * kInferKeyBits);
  return bytes;
}

void LaunchGuideInfer(const DeviceScene &sc, const PathQueues &q, const uint32_t *queue, const uint32_t *count, uint32_t max_count,
                      const nn::NetView &net, const InferSort *sort, hipStream_t st) {
  const dim3 grid(Blocks(max_count, nn::kTile, 16384)), block(nn::kTile);
  if (!sort) {
    hipLaunchKernelGGL(k_guide_infer, grid, block, 0, st, sc, q, queue, count, net, 0);
    return;
  }
  // The first max_count entries (the pass's slots bound the queue) sorted by hit point.
  hipLaunchKernelGGL(k_infer_keys, dim3(Blocks(max_count, 256, 8192)), dim3(256), 0, st, q, queue, count, max_count, net, sort->keys,
                     sort->vals);
  size_t bytes = sort->temp_bytes;
  const hipError_t e = hipcub::DeviceRadixSort::SortPairs(sort->temp, bytes, sort->keys, sort->keys + sort->capacity, sort->vals,
                                                          sort->vals + sort->capacity, (int)max_count, 0, 3 * kInferKeyBits, st);
  if (e != hipSuccess) throw std::runtime_error(std::string("inference queue sort: ") + hipGetErrorString(e));
  hipLaunchKernelGGL(k_guide_infer, grid, block, 0, st, sc, q, sort->vals + sort->capacity, count, net, 1);
}
void LaunchGuideSample(const GuideCell &c, uint64_t seed, int64_t n, float *d, float *p, hipStream_t st) {
  hipLaunchKernelGGL(k_guide_sample, dim3(Blocks(n, 256, 8192)), dim3(256), 0, st, c, seed, n, d, p);
}
void LaunchQuadSample(const QuadNode *nodes, int root, float w_root, int64_t n, const float *u, float *uv, float *d, float *p,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_quad_sample, dim3(Blocks(n, 256, 4096)), dim3(256), 0, st, QuadGuide{nodes, root, w_root}, n, u, uv, d, p);
}
void LaunchQuadPdf(const QuadNode *nodes, int root, float w_root, int64_t n, const float *dirs, float *p, hipStream_t st) {
  hipLaunchKernelGGL(k_quad_pdf, dim3(Blocks(n, 256, 4096)), dim3(256), 0, st, QuadGuide{nodes, root, w_root}, n, dirs, p);
}
void LaunchGuidePdfAt(const DeviceScene &sc, int64_t n, const float *pos, const float *dirs, float *p, hipStream_t st) {
  hipLaunchKernelGGL(k_guide_pdf_at, dim3(Blocks(n, 256, 4096)), dim3(256), 0, st, sc, n, pos, dirs, p);
}
void LaunchGuidePdf(const GuideCell &c, int64_t n, const float *dirs, float *p, hipStream_t st) {
  hipLaunchKernelGGL(k_guide_pdf, dim3(Blocks(n, 256, 8192)), dim3(256), 0, st, c, n, dirs, p);
}
void LaunchSamplePhase(int kind, float g, float3 wi, uint64_t seed, int64_t n, float *d, float *v, float *p, hipStream_t st) {
  hipLaunchKernelGGL(k_sample_phase, dim3(Blocks(n, 256, 8192)), dim3(256), 0, st, kind, g, wi, seed, n, d, v, p);
}

void LaunchSamplePhaseMix(const PhaseMix &m, float3 wi, uint64_t seed, int64_t n, float *d, float *v, float *p, hipStream_t st) {
  hipLaunchKernelGGL(k_sample_phase_mix, dim3(Blocks(n, 256, 8192)), dim3(256), 0, st, m, wi, seed, n, d, v, p);
}
void LaunchMediaEvents(const DeviceScene &sc, int64_t n, const float *org, const float *dir, const float *tmax, const uint64_t *init,
                       int max_events, double *t, int32_t *medium, int32_t *count, hipStream_t st) {
  hipLaunchKernelGGL(k_media_events, dim3(Blocks(n, 64, 4096)), dim3(64), 0, st, sc, n, org, dir, tmax, init, max_events, t, medium,
                     count);
}
void LaunchPcg32(uint64_t initstate, uint64_t initseq, int64_t n, uint32_t *out, hipStream_t st) {
  hipLaunchKernelGGL(k_pcg32, dim3(1), dim3(64), 0, st, initstate, initseq, n, out);
}

bool TakeStackOverflow(hipStream_t st) {
  unsigned int v = 0;
  if (hipMemcpyFromSymbolAsync(&v, HIP_SYMBOL(g_stack_overflow), sizeof(v), 0, hipMemcpyDeviceToHost, st) != hipSuccess) return false;
  if (hipStreamSynchronize(st) != hipSuccess) return false;
  if (v) {
    const unsigned int zero = 0;
    (void)hipMemcpyToSymbolAsync(HIP_SYMBOL(g_stack_overflow), &zero, sizeof(zero), 0, hipMemcpyHostToDevice, st);
    (void)hipStreamSynchronize(st);
  }
  return v != 0;
}

}  // namespace ttgpu
