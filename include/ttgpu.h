/*
 * ttgpu.h - C ABI of the MI355X wavefront path tracer.
 *
 * This is the drop-in boundary for ToyTrace's `pt2` (forward path tracing with
 * next-event estimation and spectral null-path tracking) and `ptg` (guided)
 * integrators. In the reference those sit behind `class RenderingAlgo`
 * (src/renderingalgorithms_interface.hxx:13-30), created by
 * `RenderAlgorithmFactory` (src/renderingalgorithms.cxx:27-42) from a `Scene`
 * (src/scene.hxx:134-315) and `RenderingParameters` (src/scene.hxx:24-43).
 *
 * Across this ABI the scene is a flat, caller-owned description: float
 * vertices, u32 triangle indices, a material id per primitive and small tables
 * of shaders, media, emitters and lights with 36-bin spectra (370-730 nm,
 * src/spectral.hxx:270-274).  Nothing but plain C types crosses the boundary.
 * Every entry point returns a status code (TTGPU_OK == 0); the message of the
 * last failure on a handle is available from ttgpu_last_error().  No C++
 * exception escapes.
 *
 * Thread-safety: ttgpu_request_interrupt() and ttgpu_request_stop() may be
 * called from any thread at any time, also before ttgpu_run() (mirrors
 * RequestInterrupt/RequestFullStop, src/renderingalgorithms_pathtracing2.cxx:216-227).
 * All other calls on one handle must come from one thread at a time.
 */
#ifndef TTGPU_H
#define TTGPU_H

#include <stdint.h>
#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

#define TTGPU_NBINS 36          /* spectral bins, src/spectral.hxx:274 */
#define TTGPU_ABI_VERSION 1

/* ---- status codes ---------------------------------------------------- */
enum {
  TTGPU_OK = 0,
  TTGPU_ERR_INVALID_ARGUMENT = 1,  /* std::invalid_argument in the reference */
  TTGPU_ERR_RUNTIME = 2,           /* std::runtime_error in the reference */
  TTGPU_ERR_DEVICE = 3,            /* HIP error */
  TTGPU_ERR_INTERRUPTED = 4,       /* a pass was cut short by interrupt/stop */
  TTGPU_ERR_OUT_OF_MEMORY = 5
};

/* ---- shaders (src/shader.cxx:251-1081) ------------------------------- */
enum ttgpu_shader_kind {
  TTGPU_SHADER_DIFFUSE = 0,             /* DiffuseShader, shader.cxx:251-318 */
  TTGPU_SHADER_MIRROR = 1,              /* SpecularReflectiveShader, :322-366 */
  TTGPU_SHADER_DIELECTRIC = 2,          /* SpecularTransmissiveDielectricShader, :378-630 */
  TTGPU_SHADER_BECKMANN_METAL = 3,      /* MicrofacetShader (Beckmann, V-cavity VNDF), :634-707 */
  TTGPU_SHADER_GGX_METAL = 4,           /* new: GGX NDF, Smith G2, visible-normal sampling */
  TTGPU_SHADER_INVISIBLE = 5,           /* InvisibleShader, :948-972 */
  TTGPU_SHADER_GLOSSY_DIELECTRIC = 6,   /* GlossyTransmissiveDielectricShader, :710-787 */
  TTGPU_SHADER_DENSE_DIELECTRIC = 7     /* SpecularDenseDielectricShader, :977-1081 */
};

typedef struct ttgpu_shader {
  int32_t kind;            /* ttgpu_shader_kind */
  float alpha;             /* roughness (Beckmann/GGX/glossy dielectric) */
  float alpha_min;         /* glossy dielectric lower roughness (== alpha without texture) */
  float ior_ratio;         /* inside ior / outside ior */
  float ior_lambda_coeff;  /* dispersion d(ior)/d(lambda nm); 0 = none (abbe_number in YAML) */
  float specular;          /* dense dielectric specular reflectivity */
  float reflectance[TTGPU_NBINS]; /* albedo / glossy reflectance spectrum */
} ttgpu_shader;

/* ---- phase functions (src/phasefunctions.cxx) -------------------------- */
enum ttgpu_phase_kind {
  TTGPU_PHASE_UNIFORM = 0,          /* phasefunctions.cxx:23-37 */
  TTGPU_PHASE_HENYEY_GREENSTEIN = 1,/* :85-138 */
  TTGPU_PHASE_RAYLEIGH = 2          /* :41-80 */
};

/* ---- media (src/shader.cxx:1162-1316, src/atmosphere.cxx) ------------ */
enum ttgpu_medium_kind {
  TTGPU_MEDIUM_VACUUM = 0,
  TTGPU_MEDIUM_HOMOGENEOUS = 1,
  TTGPU_MEDIUM_ATMOSPHERE = 2,      /* exponential Rayleigh + Mie shells, FP64 geometry */
  TTGPU_MEDIUM_ATMOSPHERE_TABULATED = 3 /* coefficient tables over altitude (TabulatedConstituents) */
};

typedef struct ttgpu_medium {
  int32_t kind;            /* ttgpu_medium_kind */
  int32_t priority;        /* MediumTracker priority, src/rendering_util.hxx:63-90 */
  int32_t phase_kind;      /* homogeneous: ttgpu_phase_kind */
  float phase_g;           /* HG asymmetry */
  float sigma_s[TTGPU_NBINS]; /* 1/length unit of the scene */
  float sigma_a[TTGPU_NBINS];
  /* Atmosphere (kind == TTGPU_MEDIUM_ATMOSPHERE), src/atmosphere.hxx:95-123,
   * src/atmosphere.cxx:132-200.  Lengths in scene units; coefficients are
   * sea-level values per scene unit.  Rayleigh scatters only; Mie scatters
   * and absorbs and uses an HG phase with mie_g. */
  double planet_center[3];
  double planet_radius;
  double atmosphere_height;     /* outer shell radius = planet_radius + height */
  double rayleigh_scale_height;
  double mie_scale_height;
  float mie_g;
  float rayleigh_sigma_s[TTGPU_NBINS];
  float mie_sigma_s[TTGPU_NBINS];
  float mie_sigma_a[TTGPU_NBINS];
  /* Tabulated atmosphere (kind == TTGPU_MEDIUM_ATMOSPHERE_TABULATED), TabulatedConstituents
   * (src/atmosphere.cxx:219-353): spectra at altitudes table_h0 + i * table_dh, i < table_size,
   * each table_size x 36 values per scene unit; coefficients are interpolated linearly in
   * altitude, zero above the table, the lowest entry below it.  Geometry (planet_center,
   * planet_radius) and mie_g (HG of the aerosols) as for the exponential atmosphere. */
  int32_t table_size;
  double table_h0, table_dh;
  const float *table_sigma_t;            /* extinction */
  const float *table_sigma_s_molecules;  /* Rayleigh scattering */
  const float *table_sigma_s_aerosols;   /* HG scattering */
} ttgpu_medium;

/* ---- materials (src/scene.hxx:46-72) ----------------------------------- */
typedef struct ttgpu_material {
  int32_t shader;          /* index into shaders, -1 = none (volume boundary only) */
  int32_t medium;          /* medium inside (against the geometric normal), -1 = none */
  int32_t outer_medium;    /* medium outside, -1 = none */
  int32_t emitter;         /* index into area_emitters, -1 = none */
} ttgpu_material;

/* ---- area emitters (src/light.hxx:72-141) ------------------------------ */
enum ttgpu_area_kind {
  TTGPU_AREA_UNIFORM = 0,   /* UniformAreaLight: L = spectrum / (2 pi), one-sided */
  TTGPU_AREA_PARALLEL = 1   /* ParallelAreaLight (delta in direction) */
};

typedef struct ttgpu_area_emitter {
  int32_t kind;
  float spectrum[TTGPU_NBINS];
} ttgpu_area_emitter;

/* ---- environment / infinite lights (src/light.hxx:148-288, light.cxx:88-189) */
enum ttgpu_env_kind {
  TTGPU_ENV_SUN = 0,         /* Sun: cone of opening_angle_deg, built-in solar spectrum x total_power */
  TTGPU_ENV_DOME = 1,        /* DistantDomeLight: uniform upper hemisphere around dir */
  TTGPU_ENV_DIRECTIONAL = 2, /* DistantDirectionalLight: delta direction */
  TTGPU_ENV_MAP = 3          /* EnvMapLight: float RGB lat-long texture, row/col CDF sampling */
};

typedef struct ttgpu_env_light {
  int32_t kind;
  double dir[3];            /* SUN/DIRECTIONAL: direction from the scene towards the light
                               (YAML "direction"; light travels along -dir);
                               DOME: up direction (light arrives from the hemisphere around dir);
                               MAP: polar axis of the lat-long map */
  double opening_angle_deg; /* SUN */
  double total_power;       /* SUN */
  float spectrum[TTGPU_NBINS]; /* DOME / DIRECTIONAL */
  int32_t tex_width, tex_height; /* MAP: row-major RGB float texture; row y holds the directions
                                    looked at (from the scene towards the map) whose angle to +dir
                                    lies in [pi*y/h, pi*(y+1)/h]: row 0 is seen looking along dir */
  const float *texture_rgb;
} ttgpu_env_light;

typedef struct ttgpu_point_light {
  double pos[3];
  float spectrum[TTGPU_NBINS]; /* total power; radiant intensity = spectrum / (4 pi) */
} ttgpu_point_light;

/* ---- camera (src/camera.hxx) ------------------------------------------ */
enum ttgpu_camera_kind {
  TTGPU_CAMERA_PINHOLE = 0,   /* PerspectiveCamera, camera.hxx:62-156 */
  TTGPU_CAMERA_FISHEYE = 1    /* FisheyeHemisphereCamera, camera.hxx:159-232 */
};

typedef struct ttgpu_camera {
  int32_t kind;
  double pos[3];
  double dir[3];
  double up[3];
  double fov_deg;             /* pinhole: full horizontal angle */
} ttgpu_camera;

/* ---- scene ------------------------------------------------------------- */
typedef struct ttgpu_scene {
  int64_t num_vertices;
  const float *vertices;        /* 3 x num_vertices */
  const float *normals;         /* 3 x num_vertices or NULL (flat shading) */
  int64_t num_triangles;        /* num_triangles + num_spheres < 2^28 */
  const uint32_t *indices;      /* 3 x num_triangles */
  const int32_t *tri_material;  /* num_triangles */
  int64_t num_spheres;
  const float *spheres;         /* 4 x num_spheres: centre xyz, radius */
  const int32_t *sphere_material;
  int32_t num_shaders;
  const ttgpu_shader *shaders;
  int32_t num_media;
  const ttgpu_medium *media;
  int32_t empty_space_medium;   /* index of the medium filling space, -1 = vacuum */
  int32_t num_materials;
  const ttgpu_material *materials;
  int32_t num_area_emitters;
  const ttgpu_area_emitter *area_emitters;
  int32_t num_env_lights;
  const ttgpu_env_light *env_lights;
  int32_t num_point_lights;
  const ttgpu_point_light *point_lights;
  ttgpu_camera camera;
} ttgpu_scene;

/* ---- parameters (src/scene.hxx:24-43) ---------------------------------- */
/* PT2: spectral null-path tracing with NEE (pt2); PTG: guided (ptg); PT: the
 * forward path tracer of the random-walk framework (pt, the reference's default
 * --algo): power-heuristic MIS, Russian roulette beyond 5 nodes, light points
 * connected to the camera and splatted to the pixel they project to; surface
 * scenes only.  BDPT: bidirectional path tracing (bdpt, BdptWorker,
 * src/renderingalgorithms_pathtracing.hxx:341-700): surface scenes, pinhole
 * camera, uniform area, point and environment lights (no directional),
 * max_ray_depth <= 16; mis_mode REFERENCE keeps the reference's Russian-roulette
 * placement and pixel truncation, CONSISTENT is unbiased. */
enum ttgpu_algo { TTGPU_ALGO_PT2 = 0, TTGPU_ALGO_PTG = 1, TTGPU_ALGO_PT = 2, TTGPU_ALGO_BDPT = 3 };
enum ttgpu_sample_mode {     /* --pt-sample-mode */
  TTGPU_SAMPLE_BOTH = 0, TTGPU_SAMPLE_BSDF = 1, TTGPU_SAMPLE_LIGHTS = 2
};
enum ttgpu_mis_mode {
  /* pt2's NEE MIS weight uses the light pdf without the light-selection
   * probability (src/renderingalgorithms_pathtracing2.cxx:489-501) while the
   * emission weight includes it (:641-644).  REFERENCE keeps that; CONSISTENT
   * multiplies the selection probability into the NEE side as well. */
  TTGPU_MIS_REFERENCE = 0, TTGPU_MIS_CONSISTENT = 1
};
/* VMF_TREE: kd-tree cells with 8-lobe vMF mixtures; QUADTREE: kd-tree cells with
 * quadtree directional distributions and UCB node weights, the reference's
 * active model (src/path_guiding.hxx:343-344); LEARNED: hash grid + MLP. */
enum ttgpu_guide_kind {
  TTGPU_GUIDE_NONE = 0, TTGPU_GUIDE_VMF_TREE = 1, TTGPU_GUIDE_LEARNED = 2, TTGPU_GUIDE_QUADTREE = 3
};

typedef struct ttgpu_params {
  int32_t algo;                 /* ttgpu_algo */
  int32_t width, height;
  int32_t max_ray_depth;        /* --rd, RayTermination max_node_count */
  int32_t max_samples_per_pixel;/* --spp; <= 0: unbounded */
  int32_t sample_mode;          /* ttgpu_sample_mode */
  int32_t mis_mode;             /* ttgpu_mis_mode */
  int32_t num_wavelengths;      /* wavelengths per path; 4 on the GPU */
  uint64_t seed;                /* PCG32 initial state; stream = global sample index */
  int64_t wavefront_paths;      /* paths in flight per wavefront; 0 = automatic.  TTGPU_ALGO_BDPT: samples
                                   in flight, from 2^13 to 2^20 (2.8 KB each at depth 8, 5.5 KB at 16) or
                                   as many as 1.4 GB hold */
  int32_t linear_output;        /* --linear-out for GenerateImage */
  int32_t num_threads;          /* CPU threads (oracle / host side) */
  /* guiding (ptg) */
  int32_t guide_kind;           /* ttgpu_guide_kind (TTGPU_ALGO_PTG: QUADTREE when NONE) */
  int32_t guide_max_spp;        /* --guide-max-spp: training sweeps of 2, 4, .. up to this many spp (512) */
  float guide_mix_bsdf;         /* ignored: the probability of keeping the BSDF sample is the
                                   shader's (0.5; glossy dielectric with alpha > 0.05: 0.1),
                                   src/shader.cxx:224-227, 937-941 */
  int32_t guide_subdiv_factor;  /* --guide-subdiv-factor: min records per kd-tree leaf (100) */
  int32_t reserved[7];
} ttgpu_params;

typedef struct ttgpu_stats {
  uint64_t paths_traced;        /* camera paths completed */
  uint64_t rays_closest;        /* closest-hit queries */
  uint64_t rays_shadow;         /* occlusion queries */
  uint64_t total_spp;           /* samples per pixel rendered so far */
  double render_ms;             /* device time of the last ttgpu_run/ttgpu_render_spp */
  double bvh_build_ms;          /* host BVH build */
  double upload_ms;
  uint64_t bvh_nodes;
  uint64_t scene_bytes;         /* device bytes of BVH + primitives */
  uint64_t state_bytes;         /* device bytes of path state queues */
  int32_t passes;
  int32_t wavefront_paths;
} ttgpu_stats;

typedef struct ttgpu_handle ttgpu_handle;
typedef void (*ttgpu_pass_callback)(void *user, int32_t is_complete_pass);

/* Lifecycle.  Replaces PathTracingAlgo2's ctor + InitializeScene
 * (src/renderingalgorithms_pathtracing2.cxx:242-263).  Copies everything it
 * needs out of `scene` (the caller may free it afterwards), builds the BVH on
 * the host and uploads scene and path-state queues to the current HIP device. */
int ttgpu_create(const ttgpu_scene *scene, const ttgpu_params *params, ttgpu_handle **out);
void ttgpu_destroy(ttgpu_handle *h);
const char *ttgpu_last_error(const ttgpu_handle *h);
/* Message of the last ttgpu_create failure (no handle exists then). */
const char *ttgpu_create_error(void);

/* PathTracingAlgo2::Run (src/renderingalgorithms_pathtracing2.cxx:269-295):
 * passes with doubling spp (1,2,4,..,1024 per pass, capped so the total does
 * not exceed max_samples_per_pixel; src/renderingalgorithms_simplebase.hxx:34-62)
 * until the budget is used or a stop is requested.  max_passes <= 0: no cap.
 * The callback (if set) fires after each pass with is_complete_pass = 1, or 0
 * when the pass was interrupted. */
int ttgpu_run(ttgpu_handle *h, int32_t max_passes);
/* One pass of exactly `spp` samples per pixel (the benchmark step). */
int ttgpu_render_spp(ttgpu_handle *h, int32_t spp);
int ttgpu_request_interrupt(ttgpu_handle *h);
int ttgpu_request_stop(ttgpu_handle *h);
int ttgpu_set_pass_callback(ttgpu_handle *h, ttgpu_pass_callback cb, void *user);
/* Clear framebuffer and sample counters (not the RNG stream position). */
int ttgpu_reset_framebuffer(ttgpu_handle *h);

/* Framebuffer: linear RGB sums (double, width*height*3, row-major, row 0 =
 * first image row of the camera) and the samples accumulated per pixel
 * (spp: array of width*height counts, may be NULL).
 * rgb_sq (optional, may be NULL): per-pixel sums of squared per-path RGB
 * estimates, for variance estimates. */
int ttgpu_read_framebuffer(ttgpu_handle *h, double *rgb, double *rgb_sq, uint64_t *spp);
/* GenerateImage (src/renderingalgorithms_pathtracing2.cxx:298-309 with
 * src/renderbuffer.hxx:99-125): 8-bit RGB, rows flipped, clamped, sRGB unless
 * params.linear_output. */
int ttgpu_generate_image(ttgpu_handle *h, uint8_t *rgb8);
int ttgpu_stats_get(ttgpu_handle *h, ttgpu_stats *out);

/* Timing of the most recent run measured with HIP events on the stream the
 * kernels run on: per-kernel-class total milliseconds and launch counts.
 * names: "trace", "shade", "shadow", "raygen", "media", "guide". */
int ttgpu_kernel_time(ttgpu_handle *h, const char *kernel_class, double *total_ms, int64_t *launches);
int ttgpu_enable_kernel_timing(ttgpu_handle *h, int32_t enable);

/* ---- scene queries (replace EmbreeAccelerator, src/embreeaccelerator.cxx:87-304) */
/* Closest hit for `count` rays; t = +inf and prim = -1 when nothing is hit.
 * prim indexes triangles first, then spheres (num_triangles + sphere index). */
int ttgpu_trace_closest(ttgpu_handle *h, int64_t count, const float *org, const float *dir,
                        const float *tmax, float *t, int32_t *prim, float *u, float *v);
int ttgpu_trace_occluded(ttgpu_handle *h, int64_t count, const float *org, const float *dir,
                         const float *tmax, int32_t *occluded);
/* Medium changes along rays through volume boundaries (test entry point for the medium
 * tracker, MediumTracker + SegmentIterator, src/rendering_util.hxx:18-207, and the ordered
 * boundary query IntersectionsWithVolumes, src/scene.cxx).  `scene` is the description the
 * handle was created from.  For each ray: the medium at its origin (out_initial; -1 = vacuum;
 * MediumTracker::initializePosition, src/rendering_util.cxx:13-37), then for each of up to
 * max_events boundary crossings in (0, tmax) the distance (out_t, FP64) and the current medium
 * after it (out_medium), max_events per ray; out_count = crossings found. */
int ttgpu_media_events(ttgpu_handle *h, const ttgpu_scene *scene, int64_t count, const float *org,
                       const float *dir, const float *tmax, int32_t max_events, int32_t *out_initial,
                       double *out_t, int32_t *out_medium, int32_t *out_count);
/* Same as ttgpu_trace_closest but testing every primitive without the BVH
 * (test entry point: the traversal's own reference on the device). */
int ttgpu_trace_closest_bruteforce(ttgpu_handle *h, int64_t count, const float *org, const float *dir,
                                   const float *tmax, float *t, int32_t *prim, float *u, float *v);
/* Allocation-free variant of ttgpu_trace_closest, with the same arguments and results.  It has
 * no counterpart in the reference: it is for callers that cannot allocate device memory (code
 * under HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).  The rays and
 * hits are staged in one static device array per GPU that holds TTGPU_NOALLOC_MAX_RAYS rays
 * (11.5 MB, kept until the process ends); the call makes no hipMalloc or hipFree.  A larger
 * count is rejected with TTGPU_ERR_INVALID_ARGUMENT.  Every call on one GPU uses the same array,
 * so calls that overlap on one GPU (several threads or handles) race: the caller serialises
 * them.  The handle's device must be the current device. */
#define TTGPU_NOALLOC_MAX_RAYS 262144
int ttgpu_trace_closest_noalloc(ttgpu_handle *h, int64_t count, const float *org, const float *dir,
                                const float *tmax, float *t, int32_t *prim, float *u, float *v);

/* ---- sampler entry points for the statistical tests ------------------------
 * Run the GPU BSDF sampler of `shader` at a surface with geometric normal ng
 * and shading normal ns (both already oriented towards wi), for `count`
 * independent samples.  Mirrors Shader::SampleBSDF / EvaluateBSDF
 * (src/shader.hxx:58-59).  bins: the 4 wavelength bins of the path.
 * out_dir: 3*count, out_value: 4*count, out_pdf: count (negative = delta,
 * src/sampler.hxx:552-590).  roughness: ShaderQuery::minimum_roughness. */
int ttgpu_sample_shader(const ttgpu_shader *shader, const float wi[3], const float ng[3],
                        const float ns[3], const int32_t bins[4], float roughness,
                        uint64_t seed, int64_t count,
                        float *out_dir, float *out_value, float *out_pdf);
int ttgpu_eval_shader(const ttgpu_shader *shader, const float wi[3], const float ng[3],
                      const float ns[3], const int32_t bins[4], float roughness,
                      int64_t count, const float *dirs, float *out_value, float *out_pdf);
/* Phase function sampling (src/phasefunctions.cxx): wi = reverse incident dir. */
int ttgpu_sample_phase(int32_t phase_kind, float g, const float wi[3], uint64_t seed,
                       int64_t count, float *out_dir, float *out_value, float *out_pdf);
/* Mixture of two phase functions, PhaseFunctions::SimpleCombined (src/phasefunctions.cxx:
 * 206-270), the atmosphere's Rayleigh + Henyey-Greenstein phase (src/atmosphere.cxx:107-125).
 * weights: 4 per constituent (one per wavelength of the path), normalised per wavelength;
 * every weight >= 0 and every wavelength's total > 0.  out_value: 4 per sample. */
int ttgpu_sample_phase_mixture(const int32_t kinds[2], const float g[2], const float weights[8],
                               const float wi[3], uint64_t seed, int64_t count, float *out_dir,
                               float *out_value, float *out_pdf);
/* The device's PCG32 (XSH-RR, 64-bit LCG; the generator behind src/sampler.cxx:371-393):
 * the first `count` 32-bit outputs after seeding with (initstate, initseq). */
int ttgpu_pcg32(uint64_t initstate, uint64_t initseq, int64_t count, uint32_t *out);

/* ---- guiding (TTGPU_ALGO_PTG) ------------------------------------------------
 * ttgpu_run on a guided handle first trains: one 1-spp pass, then sweeps of
 * 2, 4, .. up to guide_max_spp 1-spp passes, each pass recording radiance and
 * refitting the recorder, each sweep splitting kd-tree cells and baking the
 * mixtures the renderer samples (PathTracingAlgo2::Run of the guided
 * integrator, src/renderingalgorithms_pathtracing_guided.cxx:1110-1211).  Then
 * it renders with the final guide on the usual doubling schedule.  The
 * framebuffer is cleared before each sweep and before the final render.
 * Recorder state: kd-tree cells, training rounds (1-spp passes), records of the
 * last training pass and records dropped for lack of buffer space. */
int ttgpu_guide_info(ttgpu_handle *h, int32_t *cells, int32_t *rounds, int64_t *records_last_pass,
                     int64_t *records_dropped);
/* Density of the current guide (vMF-tree or quadtree handles) at positions pos
 * (3 per query) for directions dirs (3 per query, unit length): the cell's
 * distribution the renderer samples (RadianceDistributionSampled::Pdf,
 * src/path_guiding.hxx:248-254; vmf_fitting::Pdf).  on_device = 0: the
 * recorder's host copy; 1: the copy uploaded for the GPU kernels. */
int ttgpu_guide_pdf(ttgpu_handle *h, int64_t count, const float *pos, const float *dirs, int32_t on_device,
                    float *out_pdf);

/* 8-lobe von Mises-Fisher mixture (vmf_fitting::VonMisesFischerMixture<8>,
 * src/distribution_mixture_models.hxx:17-29). */
typedef struct ttgpu_vmf8 {
  float mu[8][3];
  float kappa[8];
  float w[8];
} ttgpu_vmf8;
/* Building blocks of the recorder, for tests (host code of the library):
 * InitializeForUnitSphere<8> (distribution_mixture_models.cxx:167-183);
 * incremental::Fit over n weighted directions with the recorder's parameters for
 * a cell of max_num_samples records (prior strength max(1, 0.01 max_num_samples),
 * M-step every 10x that; path_guiding.cxx:62-77, distribution_mixture_models.cxx:247-343),
 * continuing from *m; kdtree::Builder (path_guiding_tree.hxx:300-438): leaf index
 * of every point. */
int ttgpu_guide_init_vmf(ttgpu_vmf8 *out);
int ttgpu_guide_fit_vmf(ttgpu_vmf8 *m, const float *dirs, const float *weights, int64_t n, int64_t max_num_samples);
int ttgpu_guide_build_kdtree(const double *pts, int64_t n, int32_t min_points, int32_t max_depth,
                             int32_t *leaf_of_point, int32_t *num_leafs);
/* The same incremental::Fit run by the device fit of the training passes (one cell, one
 * wavefront, M-steps at the same sample counts; distribution_mixture_models.cxx:247-343), on
 * the given samples in their order.  Test access to the device EM. */
int ttgpu_guide_fit_vmf_gpu(ttgpu_vmf8 *m, const float *dirs, const float *weights, int64_t n, int64_t max_num_samples);
/* The leaf statistics the device fit keeps of a cell's records (count, mean and covariance of the
 * positions, merged per chunk of 64; Accumulators::OnlineCovariance of path_guiding.cxx), over the
 * given points.  Test access. */
int ttgpu_guide_leaf_stats_gpu(const float *pts, int64_t n, int64_t *count, double mean[3], double cov[9]);
/* GPU sampling and pdf of a mixture, as the guided kernels use them
 * (vmf_fitting::Sample / Pdf, distribution_mixture_models.cxx:88-150). */
int ttgpu_guide_sample_vmf(const ttgpu_vmf8 *m, uint64_t seed, int64_t count, float *out_dir, float *out_pdf);
int ttgpu_guide_pdf_vmf(const ttgpu_vmf8 *m, int64_t count, const float *dirs, float *out_pdf);

/* ---- quadtree directional distribution (guide_kind TTGPU_GUIDE_QUADTREE) -------
 * A tree over the unit square, to which the sphere maps by v = (z + 1) / 2,
 * u = (atan2(y, x) / pi + 1) / 2 (equal area: densities differ by 1 / (4 pi);
 * src/path_guiding.cxx:112-129).  Trees are given in pre-order with the root at
 * index 0: children[4 n + c] is child c of node n (0 bottom-left, 1 bottom-right,
 * 2 top-left, 3 top-right), all four -1 for a leaf; at most 8 levels.
 * Builder (src/path_guiding_quadtree.hxx:317-352, .cxx:32-88): nodes whose
 * weight exceeds fraction x the total weight are split.  TreeAdaptor
 * (src/path_guiding_quadtree.hxx:209-315): threshold fraction x root weight;
 * out_old_index / out_fraction = NewToOld mapping.  `capacity` bounds the
 * output node count (*num_nodes reports the size even when it does not fit). */
int ttgpu_quadtree_build(const float *uv, const float *weights, int64_t n, float fraction, int32_t capacity,
                         int32_t *children, float *node_weights, int32_t *num_nodes);
int ttgpu_quadtree_adapt(const int32_t *children, const float *weights, int32_t num_nodes, float fraction,
                         int32_t capacity, int32_t *out_children, float *out_weights, int32_t *out_old_index,
                         float *out_fraction, int32_t *out_num_nodes);
/* GPU warping of given uniforms u (2 per sample) through a tree with node
 * sampling weights `probs` (quadtree::Sample, src/path_guiding_quadtree.cxx:168-244),
 * and the density over the sphere (quadtree::Pdf x 1/(4 pi), .cxx:247-259;
 * RadianceDistributionSampled::Pdf, src/path_guiding.hxx:248-254), as the
 * guided kernels use them. */
int ttgpu_quadtree_sample(const int32_t *children, const float *probs, int32_t num_nodes, int64_t count,
                          const float *u, float *out_uv, float *out_dir, float *out_pdf);
int ttgpu_quadtree_pdf(const int32_t *children, const float *probs, int32_t num_nodes, int64_t count,
                       const float *dirs, float *out_pdf);
/* One cell's learned and sampled quadtree distributions (host code of the
 * library; RadianceDistributionLearned / RadianceDistributionSampled,
 * src/path_guiding.hxx:200-340, src/path_guiding.cxx:156-294):
 * initial_fit = InitialFit over all samples (builder fraction 0.1);
 * bake = Bake (sampled <- learned); incremental_fit = IncrementalFit of the
 * samples with original == 0 at the given round (UCB exploration term
 * sqrt(log(round) / (count + 1)) x root flux); update_and_bake =
 * IterationUpdateAndBake (adaptor fraction 0.05, statistics reset).
 * which = 0 learned tree, 1 sampled tree.  filter_direction =
 * ComputeStochasticFilteredDirection of the sampled tree (src/path_guiding.cxx:132-153). */
typedef struct ttgpu_qmodel ttgpu_qmodel;
ttgpu_qmodel *ttgpu_qmodel_create(void);
void ttgpu_qmodel_free(ttgpu_qmodel *m);
int ttgpu_qmodel_initial_fit(ttgpu_qmodel *m, const float *dirs, const float *weights, int64_t n);
int ttgpu_qmodel_bake(ttgpu_qmodel *m);
int ttgpu_qmodel_incremental_fit(ttgpu_qmodel *m, const float *dirs, const float *weights, const uint8_t *original,
                                 int64_t n, int32_t round);
/* The same IncrementalFit run by the device fit of the training passes (per-node sums merged into
 * the running statistics, the weights recomputed and propagated on the device), on the given
 * samples.  Test access to the device quadtree fit. */
int ttgpu_qmodel_incremental_fit_gpu(ttgpu_qmodel *m, const float *dirs, const float *weights, const uint8_t *original,
                                     int64_t n, int32_t round);
int ttgpu_qmodel_update_and_bake(ttgpu_qmodel *m);
int ttgpu_qmodel_num_nodes(const ttgpu_qmodel *m, int32_t which, int32_t *out);
int ttgpu_qmodel_get_learned(const ttgpu_qmodel *m, int32_t *children, int64_t *counts, double *means, double *m2);
int ttgpu_qmodel_get_sampled(const ttgpu_qmodel *m, int32_t *children, double *means, double *stddev, float *probs,
                             float *prior);
int ttgpu_qmodel_filter_direction(const ttgpu_qmodel *m, const float dir[3], double u0, double u1, float out[3]);

/* ---- learned guide (guide_kind TTGPU_GUIDE_LEARNED) ---------------------------
 * A multiresolution hash-grid encoding of the position (levels x 2 features,
 * 2^log2_table entries per level, resolutions base_res .. max_res geometric),
 * the shading normal and the outgoing direction (38 inputs) feed an MLP
 * 38 -> 64 -> 64 -> 64 -> 80 (ReLU) whose outputs are a 16-lobe vMF mixture:
 * per lobe (logit, m.xyz, s) -> weight softmax(logit), mean m/|m|,
 * concentration min(softplus(s) + 0.05, 100).  bf16 MFMA with fp32
 * accumulation; trained online with Adam on the renderer's radiance records
 * by minimising -(radiance / pdf) log q(direction).  No counterpart in the
 * reference (new guiding method).
 * Positions map to [0,1]^3 through lo' = bb_lo - 1e-3 ext, scale 1 / (1.002 ext).
 * Parameter vector (fp32): grid [levels][2^log2_table][2] | W1T[64][64] | W2T[64][64] |
 * W3T[64][64] | W4T[96][64] | b1[64] | b2[64] | b3[64] | b4[96]; WkT[out][in],
 * input columns 38..63 and output rows 80..95 stay zero. */
typedef struct ttgpu_nn_config {
  int32_t levels;        /* 16 */
  int32_t log2_table;    /* 19 */
  float base_res;        /* 16 */
  float max_res;         /* 1024 */
  int32_t batch;         /* records per Adam step (65536) */
  float lr;              /* Adam learning rate (1e-2) */
  float bb_lo[3], bb_hi[3];
  uint64_t seed;
} ttgpu_nn_config;
int64_t ttgpu_nn_param_count(const ttgpu_nn_config *cfg);
/* Initial parameters as the renderer draws them from cfg->seed. */
int ttgpu_nn_init_params(const ttgpu_nn_config *cfg, float *params);
/* Raw outputs (n x 96, entries 80..95 zero) for n records: pos, nrm, wo are n x 3. */
int ttgpu_nn_forward(const ttgpu_nn_config *cfg, const float *params, int64_t n, const float *pos, const float *nrm,
                     const float *wo, float *out);
/* Gradient of the mean over the n records of -weight log q(wi) with respect to every parameter,
 * and the mean loss.  n <= cfg->batch. */
int ttgpu_nn_gradient(const ttgpu_nn_config *cfg, const float *params, int64_t n, const float *pos, const float *nrm,
                      const float *wo, const float *wi, const float *weight, float *grad, float *loss);
/* `passes` training passes over the records (as the renderer trains after each pass);
 * params in/out; loss_per_pass (optional) receives each pass's mean loss. */
int ttgpu_nn_train(const ttgpu_nn_config *cfg, float *params, int64_t n, const float *pos, const float *nrm, const float *wo,
                   const float *wi, const float *weight, int32_t passes, float *loss_per_pass);

/* ---- HDR image files ------------------------------------------------------
 * Linear counterparts of GenerateImage's 8-bit sRGB output (src/renderbuffer.hxx:99-125):
 * PFM (little-endian float RGB, bottom row first) or OpenEXR (single-part scanline file,
 * uncompressed 32-bit float B, G, R channels).  No counterpart in the reference, which writes
 * PNG only. */
enum ttgpu_image_format { TTGPU_IMAGE_PFM = 0, TTGPU_IMAGE_EXR = 1 };
/* `rgb`: width x height x 3 floats, top row first. */
int ttgpu_write_rgb_image(const float *rgb, int32_t width, int32_t height, const char *path, int32_t format);
/* The framebuffer's mean radiance per pixel (linear RGB sums / samples per pixel; pixels
 * without samples are 0). */
int ttgpu_write_image(ttgpu_handle *h, const char *path, int32_t format);

/* ---- scene files ----------------------------------------------------------
 * Scene::ParseNFF / ParseNFFString (src/parsenff.cxx:992-1028): ToyTrace's NFF dialect
 * (scopes, transforms, yaml{ }yaml blocks, shaders, media, lights, `include`) with the OBJ
 * and COLLADA meshes named by `m` (assimp::Read, src/parse_common.cxx:225-249).  The file
 * object owns every array of the scene description it hands out.  Errors (status
 * TTGPU_ERR_INVALID_ARGUMENT for malformed input or unsupported directives, TTGPU_ERR_RUNTIME
 * for unreadable files, as the reference's exceptions) are described by ttgpu_create_error(). */
typedef struct ttgpu_scene_file ttgpu_scene_file;
/* A file named *.yaml / *.yml is read as a YAML scene (below), any other as NFF. */
int ttgpu_scene_file_load(const char *path, ttgpu_scene_file **out);
/* NFF text; relative file names resolve against the directory of `path_hint` (may be NULL). */
int ttgpu_scene_file_parse(const char *nff_text, const char *path_hint, ttgpu_scene_file **out);
/* Scene::ParseYAML (src/parse_yaml_scene.cxx:622-628): ToyTrace's YAML scene format -- scopes
 * with transforms, shaders, media, arealights, lights, materials (named or inlined parts),
 * models (mesh files with material maps, spheres), nested scopes and the view.  Unknown or
 * unused keys, unnamed top-level items and named inline items are errors, as in the reference.
 * The camera's resolution is the reference's default 640 x 480 (the render parameters set the
 * real one).  Textures and modulated-density media are rejected. */
int ttgpu_scene_file_parse_yaml(const char *yaml_text, const char *path_hint, ttgpu_scene_file **out);
const ttgpu_scene *ttgpu_scene_file_scene(const ttgpu_scene_file *f);
/* The resolution of the file's camera (0 x 0 without a camera). */
int ttgpu_scene_file_resolution(const ttgpu_scene_file *f, int32_t *width, int32_t *height);
void ttgpu_scene_file_free(ttgpu_scene_file *f);

/* Device / build information string ("gfx950, 256 CUs, ..."). */
const char *ttgpu_device_info(void);
int ttgpu_abi_version(void);

#ifdef __cplusplus
}
#endif
#endif /* TTGPU_H */
