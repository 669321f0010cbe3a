// Host-callable launchers of the wavefront kernels (defined in kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "device_scene.hpp"
#include "nn.hpp"
#include "pass_progress.hpp"

namespace ttgpu {

hipError_t UploadSpectralTables(const float *to_rgb, const float *smits);
void LaunchResetCounter(uint32_t *counters, int which, hipStream_t st);
void LaunchFill(double *p, double *p2, size_t n, double v, hipStream_t st);  // two arrays of n values
// First `count` camera paths of a pass into slots [0, count) of queue A; resets the pass counters.
void LaunchRaygen(const DeviceScene &sc, const PathQueues &q, uint32_t count, uint32_t npix, uint32_t spp_base, uint64_t seed,
                  hipStream_t st);
// Path regeneration of an iteration: freed slots take the pass's next camera paths (at most `limit`
// issued in total) and the next queue is built in queue_out, its length (and identity flag) in
// count_out; the iteration's progress goes to `host` with sequence number `seq`.
struct RegenArgs {
  uint32_t *queue_out, *count_out;
  uint32_t slots;           // slots the pass uses: [0, slots)
  uint64_t limit;
  uint32_t npix, spp_base;
  uint64_t seed;
  bool with_shadow;         // the queued shadow rays are work of the next trace launch
  PassProgress *host;       // device address of the page-locked record
  unsigned long long seq;
  void *select_temp;        // SelectTempBytes(capacity) bytes (slot-ordered queues)
};
void LaunchRegen(const DeviceScene &sc, const PathQueues &q, const RegenArgs &a, hipStream_t st);
// Counters and the stack-overflow flag (then cleared) to the page-locked report.
void LaunchReport(const PathQueues &q, PassReport *host, hipStream_t st);
size_t SelectTempBytes(uint32_t capacity);
// with_shadow: the launch also takes the shadow rays of the previous shade launch
// (ShadowInTrace), and LaunchShadow is not called.
void LaunchTrace(const DeviceScene &sc, const PathQueues &q, const uint32_t *queue, const uint32_t *count, uint32_t max_count,
                 double *fb, double *fb_sq, bool with_shadow, hipStream_t st);
bool ShadowInTrace(const DeviceScene &sc, const PathQueues &q);
void LaunchTrackMedia(const DeviceScene &sc, const PathQueues &q, const uint32_t *queue, const uint32_t *count, uint32_t max_count,
                      hipStream_t st);
void LaunchShade(const DeviceScene &sc, const PathQueues &q, const uint32_t *queue_in, const uint32_t *count_in, uint32_t *queue_out,
                 uint32_t *count_out, uint32_t max_count, double *fb, double *fb_sq, hipStream_t st);
constexpr int kBdptMaxVertices = 17;  // BDPT subpath vertices per thread: max_ray_depth <= 16
// Workspace of a chunk of at most `capacity` (<= 2^20) BDPT samples.
struct BdptWork {
  float4 *verts;     // eye, light and light-sample vertices: capacity x BdptVertexBytes(max_nodes)
  uint32_t *pairs;   // connections: sample | eye vertex << 20 | light vertex << 25 (0: light sample)
  uint32_t *count;   // number of connections; zero between chunks
  uint2 *info;       // per sample: wavelength bins, lambda of the hero wavelength
  double *acc;       // per sample: rgb
  int max_nodes;     // vertices per subpath
  uint32_t capacity;
};
size_t BdptVertexBytes(int max_nodes);
// Connections of a sample at most: eye vertex e < max_nodes - 1 with its light sample and the light
// vertices 1 .. max_nodes - e - 2.
constexpr size_t BdptMaxPairs(int max_nodes) { return max_nodes > 1 ? (size_t)max_nodes * (max_nodes - 1) / 2 : 1; }
// Samples [first, first + count) of the pass, count <= capacity.
void LaunchBdpt(const DeviceScene &sc, const BdptWork &w, uint64_t first, uint32_t count, uint32_t npix, uint32_t spp_base, uint64_t seed,
                double *fb, double *fb_sq, uint32_t *stats, hipStream_t st);
void LaunchCameraConnect(const DeviceScene &sc, uint64_t first, uint64_t count, uint32_t npix, uint32_t spp_base, uint64_t seed,
                         double *fb, double *fb_sq, uint32_t *stats, hipStream_t st);
void LaunchShadow(const DeviceScene &sc, const PathQueues &q, uint32_t max_count, double *fb, double *fb_sq, hipStream_t st);
void LaunchTraceRays(const DeviceScene &sc, int64_t n, const float *org, const float *dir, const float *tmax, float *t, int32_t *prim,
                     float *u, float *v, int32_t *occl, int brute, hipStream_t st);
// Ray arrays of n <= stride rays from page-locked memory: origins at 0, directions at 12 x stride,
// tmax at 24 x stride bytes, in both; stride is a multiple of 16.
void LaunchCopyRays(void *to, const void *from, size_t n, size_t stride, hipStream_t st);
void LaunchSampleShader(const DevShader &s, float3 wi, float3 ng, float3 ns, uint32_t bins, float rough, uint64_t seed, int64_t n,
                        float *d, float *v, float *p, hipStream_t st);
void LaunchEvalShader(const DevShader &s, float3 wi, float3 ng, float3 ns, uint32_t bins, float rough, int64_t n, const float *dirs,
                      float *v, float *p, hipStream_t st);
// Buffers of the inference queue sort: keys and values twice `capacity` entries each, and the
// sort's storage (InferSortTempBytes(capacity) bytes).
struct InferSort {
  uint32_t *keys, *vals;
  void *temp;
  size_t temp_bytes;
  uint32_t capacity;
};
size_t InferSortTempBytes(uint32_t capacity);
// Learned-guide inference over the queue; with `sort`, over the queue's first max_count entries
// sorted by hit point (max_count >= the queue's length).
void LaunchGuideInfer(const DeviceScene &sc, const PathQueues &q, const uint32_t *queue, const uint32_t *count, uint32_t max_count,
                      const nn::NetView &net, const InferSort *sort, hipStream_t st);
void LaunchGuideSample(const GuideCell &c, uint64_t seed, int64_t n, float *d, float *p, hipStream_t st);
void LaunchQuadSample(const QuadNode *nodes, int root, float w_root, int64_t n, const float *u, float *uv, float *d, float *p,
                      hipStream_t st);
void LaunchQuadPdf(const QuadNode *nodes, int root, float w_root, int64_t n, const float *dirs, float *p, hipStream_t st);
void LaunchGuidePdfAt(const DeviceScene &sc, int64_t n, const float *pos, const float *dirs, float *p, hipStream_t st);
void LaunchGuidePdf(const GuideCell &c, int64_t n, const float *dirs, float *p, hipStream_t st);
void LaunchSamplePhase(int kind, float g, float3 wi, uint64_t seed, int64_t n, float *d, float *v, float *p, hipStream_t st);
struct PhaseMix;
void LaunchSamplePhaseMix(const PhaseMix &m, float3 wi, uint64_t seed, int64_t n, float *d, float *v, float *p, hipStream_t st);
void LaunchMediaEvents(const DeviceScene &sc, int64_t n, const float *org, const float *dir, const float *tmax, const uint64_t *init,
                       int max_events, double *t, int32_t *medium, int32_t *count, hipStream_t st);
// True (and the flag cleared) when a traversal since the last call found its stack full.
bool TakeStackOverflow(hipStream_t st);
void LaunchPcg32(uint64_t initstate, uint64_t initseq, int64_t n, uint32_t *out, hipStream_t st);

}  // namespace ttgpu
