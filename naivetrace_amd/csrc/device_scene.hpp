// Device-side layout of the scene and of the path-state queues.
//
// Everything here lives in HBM as structure-of-arrays.  The scene is the
// flattened ToyTrace `Scene` (src/scene.hxx:134-315) after the host BVH build:
// primitives are stored in BVH leaf order so the traversal touches them
// contiguously; every per-primitive array below is indexed by that order.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/ttgpu.h"

namespace ttgpu {

constexpr int kNBins = 36;
constexpr int kNW = 4;              // wavelengths per path
constexpr int kStrata = kNBins / kNW;
constexpr int kMaxEnvLights = 8;
constexpr int kMaxMedia = 32;
constexpr int kVacuum = 0xFF;       // medium id of vacuum in the packed tracker
constexpr int kEmptySlot = 0xFE;

// BVH2 node, 64 bytes: both child boxes are stored in the parent so one fetch
// decides both children (Aila & Laine 2009 layout).
struct alignas(16) BvhNode {
  float4 lxy;   // left  lo.x hi.x lo.y hi.y
  float4 rxy;   // right lo.x hi.x lo.y hi.y
  float4 lrz;   // left lo.z hi.z, right lo.z hi.z
  int4 ch;      // left, right: >= 0 inner node, < 0 leaf ~first_prim; z/w: prim counts of leaves
};

// Traversal node of the surface BVH, 64 bytes (two per 128-byte cache line): four children whose boxes
// have 8-bit planes on a per-node grid, laid out for few instructions per visit.  A node's inner children are consecutive nodes and take its first slots, so that child
// slot c is node child_base + c; the primitives of its leaves are consecutive too, so that the
// leaves a ray enters are one bit mask.
//   origin : xyz = grid origin, w = the grid steps' exponents (signed bytes x, y, z)
//   qxy    : lo.x, hi.x, lo.y, hi.y rows, byte c = child c; qlz, qhz: the z rows.  Planes are
//            origin + q * 2^e in exact arithmetic, outside the child's box by a margin that covers
//            the slab test's rounding (PackTraversal)
//   leaf   : per slot 0 for an inner child, else bit 31 and the leaf's primitives as bits of the
//            node's primitives (bit k: prim_base + k; none for an empty slot)
struct alignas(64) TravNode {
  float4 origin;
  uint4 qxy;
  uint32_t qlz, qhz;
  int child_base, prim_base;
  uint4 leaf;
};

constexpr int kStackEntries = 96;                   // traversal stack entries per lane
// A BVH4 node pushes at most three children, so a tree of depth D needs 3 (D + 1) entries.
constexpr int kMaxBvh4Depth = kStackEntries / 3 - 1;

// Primitive record in leaf order, 48 bytes.
//   triangle: a = (v0, orig_id bits), b = (v1, kind=0), c = (v2, 0)
//   sphere  : a = (centre, orig_id bits), b = (radius, 0, 0, kind=1), c = 0
struct alignas(16) PrimRecord {
  float4 a, b, c;
};

struct DevShader {
  int kind;
  float alpha, alpha_min, ior_ratio, ior_lambda_coeff, specular;
  float reflectance[kNBins];
};

struct DevMedium {
  int kind, priority, phase_kind;
  float phase_g;
  float sigma_s[kNBins];
  float sigma_t[kNBins];
  double planet_center[3];
  double planet_radius, rayleigh_inv_h, mie_inv_h, lower_cutoff;
  float mie_g;
  float rayleigh_sigma_s[kNBins], mie_sigma_s[kNBins], mie_sigma_a[kNBins];
  // tabulated atmosphere: rows of 3 x 36 (extinction, molecular and aerosol scattering) per
  // altitude table_h0 + i / table_inv_dh, and the extinction majorant per altitude
  int table_n;
  double table_h0, table_inv_dh;
  const float *table;
  const float *table_majorant;
};


struct DevMaterial {
  int shader, medium, outer_medium, emitter;
};

struct DevEmitter {
  int kind;
  float radiance[kNBins];   // already divided by 2 pi for uniform emitters
};

struct DevEnvLight {
  int kind;
  float3 frame_x, frame_y, frame_z;   // sun: cone frame (z = centre of dir_out); map: up frame
  float cos_open, pdf;               // sun
  float spectrum[kNBins];            // sun (power * pdf * solar), dome, directional
  float3 dir;                        // dome: up; directional: dir_out
  int tex_w, tex_h;
  // map: texels and alias tables (Walker/Vose) over rows and, per row, over columns.  Alias entry:
  // {keep threshold, alias index (int bits), probability of the entry, probability of its alias}.
  const float4 *texel;               // h * w: R, G, B, probability of the column within its row
  const float4 *alias_rows;          // h
  const float4 *alias_cols;          // h * w (row-major)
};

struct DevPointLight {
  float3 pos;
  float intensity[kNBins];           // spectrum / (4 pi)
};

struct DevCamera {
  int kind;
  float3 pos, right, up, dir;
  float xmin, ymin, xper, yper, fish_delta;
  int width, height;
};

// Guiding kd-tree node: a child >= 0 is a branch, < 0 the leaf (cell) ~child.
struct GuideNode {
  float split;
  int axis;
  int left, right;
};

// Baked 8-lobe vMF mixture of one cell: lobe = (mean direction, concentration),
// wn = weight x k / (2 pi (1 - exp(-2k))), cdf = cumulative lobe weights.
constexpr int kGuideLobes = 8;
struct GuideCell {
  float4 lobe[kGuideLobes];
  float wn[kGuideLobes];
  float cdf[kGuideLobes];
};

// Quadtree directional distribution of one cell over the equal-area square of the sphere.  Only
// branches are stored, 32 bytes each: w = sampling weights of the children (0 bottom-left, 1
// bottom-right, 2 top-left, 3 top-right), child = branch index of a child, -1 for a leaf child.
constexpr int kQuadMaxDepth = 8;
struct QuadNode {
  float4 w;
  int4 child;
};
struct QuadCell {
  int root;      // branch index of the root; -1: the root is a leaf (uniform over the sphere)
  float w_root;  // weight of the root (the sum of its children's weights)
};

struct DeviceScene {
  const TravNode *nodes;           // surface BVH
  const PrimRecord *prims;         // leaf order
  // Three copies of prims for traversal, in the order of the nodes' primitive ranges: copy k holds
  // each triangle's vertex coordinates in the order ((k+1) mod 3, (k+2) mod 3, k), the frame of the
  // watertight test for rays whose largest direction component is k (spheres are stored
  // unchanged).  a.w holds the primitive's index in the leaf-order arrays.
  const PrimRecord *prims_kz;
  const int *prim_material;        // leaf order
  const float4 *prim_normals;      // leaf order, 3 per triangle (vertex normals), or null
  const float *prim_area;          // leaf order
  int num_prims;
  int num_triangles;
  // volume boundaries (separate BVH)
  const BvhNode *vol_nodes;
  const PrimRecord *vol_prims;
  const int *vol_material;
  int num_vol_prims;
  // tables
  const DevShader *shaders;
  const DevMedium *media;
  const DevMaterial *materials;
  const DevEmitter *emitters;
  const DevEnvLight *envs;
  const DevPointLight *points;
  const int *area_lights;          // leaf-order prim index of each area light
  int num_area_lights, num_envs, num_points, num_media;
  float type_probs[4];             // env, area, point, volume
  float area_pick_prob;            // probability to pick one given area light (incl. type)
  float bb_diag;
  float3 bb_center;                // centre of the scene's bounding box
  int empty_space_medium;          // kVacuum or medium id
  int has_media;
  int has_atmosphere;              // 1: some medium is an atmosphere (its coefficients vary along a ray)
  uint64_t cam_tracker;            // packed medium tracker at the camera
  DevCamera cam;
  int sample_mode, mis_mode, max_depth;
  int algo_pt;                     // 1: pt semantics (power heuristic, Russian roulette, camera connections)
  int shadow_in_trace;             // 1: surface passes trace shadow rays in the next closest-hit launch
  int sort_shade;                  // 1: the surface shade kernel sorts each block's paths by shader class
  // guiding (guided integrator only)
  const GuideNode *guide_nodes;
  const GuideCell *guide_cells;     // vMF mixtures, or null
  const QuadCell *guide_qcells;     // quadtree distributions, or null
  const QuadNode *guide_qnodes;
  int guide_root;                  // root handle (< 0: the tree is a single cell ~root)
  int guide_record;                // 1: training pass, write radiance records
};

// Path state, structure of arrays over the wavefront capacity.
struct PathQueues {
  float4 *org;          // xyz
  float4 *dir;          // xyz
  float4 *hit;          // t, u, v, prim (int bits); prim < 0: miss
  float4 *thru;         // throughput per wavelength
  float4 *rad;          // accumulated rgb, w: unused
  uint32_t *bins;       // 4 x 8-bit bin indices
  uint32_t *pixel;
  uint2 *rng_state;
  uint2 *rng_inc;
  uint32_t *flags;      // bits 0-7 node count, 8 has_last_pdf, 9 last_pdf_delta, 10 finalize_after_shadow
  float *last_pdf;
  float *roughness;
  uint2 *tracker;       // packed medium tracker: current | 4 slots
  // shadow rays
  float4 *sh_org;       // xyz, tmax
  float4 *sh_dir;       // xyz; media scenes: w = light pdf, negative for a delta light
  float4 *sh_contrib;   // rgb if unoccluded (media scenes: per-wavelength value before transmission and MIS)
  // queues
  uint32_t *queue_a, *queue_b, *shadow_queue;
  uint32_t *counters;   // [0] queue_a count, [1] queue_b count, [2] shadow count, [3..] stats
  // Lengths of the shadow queue: of the rays the previous shade launch queued (which the trace
  // launch takes) and of those this iteration's shade launch queues.  Slot-ordered queues
  // alternate between two counters, so that none is cleared between two launches.
  uint32_t *shadow_in, *shadow_out;
  // path regeneration: slots of the paths finished in the current iteration, and the pass's
  // progress ([0] camera paths issued so far, [1] paths queued for the next iteration)
  uint32_t *free_slots;
  unsigned long long *progress;
  // slot-ordered queues: 1 for every slot whose path continues next iteration, and for every slot
  // freed for regeneration (null: the shade kernels append continuing paths to the next queue and
  // finished paths to free_slots instead)
  uint8_t *alive, *freed;
  // guided integrator: per-vertex state, depth-major ([vertex * capacity + path]), and records
  float4 *gv_pos_pdf;   // scatter position, mixture pdf of the sampled direction (<= 0: no record)
  float4 *gv_dir_acc;   // sampled direction, accumulated incident radiance (mean over wavelengths)
  float4 *gv_thru;      // path throughput after the scatter at the vertex
  float4 *sh_nee;       // shadow ray: NEE radiance towards the previous vertex (per wavelength)
  float4 *rec_pos_w;    // records: position, weight = radiance / pdf
  float4 *rec_dir;      // records: direction, weight
  // learned guide only: per-vertex shading normal and outgoing direction, the same in the records,
  // and the per-path 16-lobe mixture from batched inference (24 float4 per path)
  float4 *gv_nrm, *gv_wo, *rec_nrm, *rec_wo;
  float4 *gmix;
  uint32_t rec_capacity;
  int max_vertices;
  // media (only when the scene has media, else null)
  float4 *wt_r, *wt_c;  // path-space tracking weights r (x) c of the null-path formulation
  uint4 *sh_aux;        // shadow ray: medium tracker (x, y), BSDF/phase pdf bits (z), guided: vertex count (w)
  // guided integrator in media (tracking runs in its own kernel, before the guide's inference):
  // distance of the volume collision along the ray (< 0: none, the ray's surface hit or escape
  // follows), and the tracking weights with the null collisions (the emission MIS's other factor)
  double *vt;
  float4 *wtn_r, *wtn_c;
  int capacity;
};

enum FlagBits : uint32_t {
  kFlagNodeMask = 0xFFu,
  kFlagHasLastPdf = 1u << 8,
  kFlagLastPdfDelta = 1u << 9,
  kFlagFinalizeAfterShadow = 1u << 10,
  kFlagVertexShift = 16,            // guided integrator: number of stored vertices in bits 16-23
  kFlagVertexMask = 0xFFu << 16,
};

enum Counter {
  kCountA = 0, kCountB = 1, kCountShadow = 2, kCountRecords = 3, kStatClosest = 4, kStatShadow = 5, kStatPaths = 6,
  kStatRecordsDropped = 7, kCountFree = 9, kIdentA = 10, kIdentB = 11, kCountShadow2 = 12, kSlotTicket = 13,
  kNumCounters = 16
};
// What the slot selection of an iteration hands to the regeneration: how many freed slots take the
// next camera paths of the pass, and the pixel and sample of the first of them.
struct SlotPlan {
  unsigned long long sample0;
  uint32_t pixel0, refill;
};
// End of a pass, written by the device into page-locked host memory.
struct PassReport {
  uint32_t counters[kNumCounters];
  uint32_t stack_overflow;
};
// Queues A and B carry a flag beside their length (counters[kIdentA], counters[kIdentB]): 1 when the
// queue holds every slot of the wavefront, so that entry k may be taken as slot k.
constexpr int kIdentOffset = kIdentA - kCountA;
static_assert(kIdentB - kCountB == kIdentOffset, "identity flags follow the queue lengths");

}  // namespace ttgpu
