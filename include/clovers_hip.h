/*
 * clovers_hip.h -- C ABI of the MI355X wavefront spectral path tracer.
 *
 * This is the drop-in boundary for the reference renderer's hot path.  The
 * reference (Walther/clovers, Rust) renders with exactly one call,
 *
 *     draw_cpu::draw(&GlobalOptions, &RenderOptions, &Scene, Sampler) -> Vec<Xyz<E>>
 *         clovers-cli/src/draw_cpu.rs:26-98, called at clovers-cli/src/render.rs:149
 *
 * after building a `Scene` (clovers/src/scenes.rs:9-18) from a scene file
 * (clovers-cli/src/scenefile.rs:34-117).  Here the scene arrives as a flat,
 * plain-old-data descriptor (clv_scene_desc) that mirrors the reference's
 * object/material model one-to-one, and clv_render() returns the same pixel
 * buffer draw() returns: linear XYZ with white point E, row 0 = top of the
 * image, index = x + row*W, averaged over samples (draw_cpu.rs:51,66,145).
 *
 * Conventions: C99, POD structs only, no exceptions cross the boundary, every
 * entry point returns a clv_status and never aborts.  A context is not
 * re-entrant (calls on one clv_ctx are serialised by the caller); separate
 * contexts may be used from separate host threads.  All device memory is
 * owned by the context.  All pointers passed in are host pointers; the library
 * copies what it keeps.
 */
#ifndef CLOVERS_HIP_H
#define CLOVERS_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define CLV_ABI_VERSION 7u

typedef enum {
  CLV_OK = 0,
  CLV_EINVAL = 1,        /* malformed argument or scene */
  CLV_ENOMEM = 2,        /* host or device allocation failed */
  CLV_EDEVICE = 3,       /* no HIP device / HIP runtime error */
  CLV_EUNSUPPORTED = 4,  /* valid in the reference's schema, not supported here */
  CLV_EINTERNAL = 5
} clv_status;

/* ---------------------------------------------------------------- scene --- */

/* Object kinds: clovers/src/objects.rs:59-87 (the in-scope subset).  A Boxy is
 * one object made of six quads (objects/boxy.rs:43-83). */
typedef enum {
  CLV_OBJ_SPHERE = 0,   /* p = center.xyz, radius                         (objects/sphere.rs:43-54) */
  CLV_OBJ_QUAD = 1,     /* p = q.xyz, u.xyz, v.xyz                        (objects/quad.rs:248-270) */
  CLV_OBJ_TRIANGLE = 2, /* p = a.xyz, b.xyz, c.xyz (absolute corners)     (objects/triangle.rs:106-117) */
  CLV_OBJ_BOXY = 3,     /* p = corner_0.xyz, corner_1.xyz                  (objects/boxy.rs:43-83) */
  CLV_OBJ_TRIANGLE_QUV = 4, /* p = q.xyz, u.xyz, v.xyz (scene-file Triangle)  (objects/triangle.rs:61-101) */
  CLV_OBJ_MOVING_SPHERE = 5, /* p = center_0.xyz, center_1.xyz, radius; time_0 = 0, time_1 = 1
                               (objects/moving_sphere.rs, objects.rs:104-109).  Never a light-sampling
                               target: its sampler is unimplemented in the reference (a panic), so
                               priority = 1 is CLV_EINVAL */
  /* ConstantMedium (objects/constant_medium.rs:65-126, objects.rs:99-103) with a Sphere or a Boxy
   * boundary; material = a CLV_MAT_ISOTROPIC phase function carrying the medium's texture.  A
   * boundary's own RotateY/Translate wrappers go on the medium object (the same hit: distances are
   * measured along the same ray).  Never a light-sampling target (random() is unimplemented in
   * the reference), so priority = 1 is CLV_EINVAL.  The free-flight uniform that the reference
   * draws from the path's generator during traversal is drawn from a hash of the path's stream
   * state and the medium's object index instead, so that it does not depend on traversal order. */
  CLV_OBJ_CONSTANT_MEDIUM_SPHERE = 6, /* p = center.xyz, radius, density */
  CLV_OBJ_CONSTANT_MEDIUM_BOXY = 7    /* p = corner_0.xyz, corner_1.xyz, density */
} clv_object_kind;

/* One top-level hitable of the reference's flattened list (scenefile.rs:63-103):
 * STL/PLY/ObjectList lists are flattened into one object per element. */
typedef struct {
  uint32_t kind;      /* clv_object_kind */
  uint32_t material;  /* index into clv_scene_desc.materials */
  uint32_t priority;  /* 1: also a multiple-importance-sampling target (scenefile.rs:89-100) */
  uint32_t xform;     /* index into clv_scene_desc.xforms, or CLV_NO_XFORM */
  float p[9];
  uint32_t _pad[3];
} clv_object;         /* 64 bytes */

#define CLV_NO_XFORM 0xFFFFFFFFu

/* Instance wrappers: Translate (objects/translate.rs:41-103) and RotateY
 * (objects/rotate.rs:40-182).  ops[0] is the OUTERMOST wrapper, e.g. the
 * reference idiom Translate{RotateY{Boxy}} is {TRANSLATE, ROTATE_Y}. */
typedef enum { CLV_XF_TRANSLATE = 0, CLV_XF_ROTATE_Y = 1 } clv_xform_op_kind;
#define CLV_MAX_XFORM_OPS 4
typedef struct {
  uint32_t kind;      /* clv_xform_op_kind */
  float v[3];         /* TRANSLATE: offset.xyz; ROTATE_Y: angle in degrees in v[0] */
} clv_xform_op;
typedef struct {
  uint32_t n_ops;
  uint32_t _pad[3];
  clv_xform_op ops[CLV_MAX_XFORM_OPS];
} clv_xform;

/* Material kinds: clovers/src/materials.rs:141-156 (in-scope subset). */
typedef enum {
  CLV_MAT_LAMBERTIAN = 0,     /* materials/lambertian.rs  albedo texture */
  CLV_MAT_METAL = 1,          /* materials/metal.rs       albedo texture, fuzz */
  CLV_MAT_DIELECTRIC = 2,     /* materials/dielectric.rs  refractive_index, color (Xyz<E>) */
  CLV_MAT_DISPERSIVE = 3,     /* materials/dispersive.rs  cauchy_a, cauchy_b (um^2) */
  CLV_MAT_DIFFUSE_LIGHT = 4,  /* materials/diffuse_light.rs  emit texture */
  CLV_MAT_CONE_LIGHT = 5,     /* materials/cone_light.rs  emit texture, spread (degrees) */
  CLV_MAT_ISOTROPIC = 6       /* materials/isotropic.rs   albedo texture (not a surface checker); only
                                 as the phase function of a constant medium */
} clv_material_kind;

/* Texture kinds: clovers/src/textures.rs:22-109 (in-scope subset). */
typedef enum {
  CLV_TEX_SOLID = 0,          /* SolidColor: color = Xyz<E> (textures/solid_color.rs) */
  CLV_TEX_ILLUMINANT_D65 = 1, /* CIE D65 table x intensity (build.rs:66-112) */
  CLV_TEX_ILLUMINANT_D50 = 2, /* CIE D50 table x intensity */
  CLV_TEX_SPATIAL_CHECKER = 3, /* even = color, odd = odd_color, density; by world position
                                  (textures/spatial_checker.rs) */
  CLV_TEX_SURFACE_CHECKER = 4  /* even = color, odd = odd_color, density; by surface (u, v)
                                  (textures/surface_checker.rs) */
} clv_texture_kind;

typedef struct {
  uint32_t kind;          /* clv_material_kind */
  uint32_t texture;       /* clv_texture_kind of albedo (Lambertian/Metal) or emit (DiffuseLight/ConeLight) */
  float color[3];         /* SolidColor / checker even cells / Dielectric color, already converted to Xyz<E> */
  float intensity;        /* illuminant intensity (default 1.0) */
  float fuzz;             /* Metal; NOT clamped (the scene-file path does not clamp, metal.rs:60) */
  float refractive_index; /* Dielectric (default 1.5) */
  float cauchy_a;         /* Dispersive (default 1.5046) */
  float cauchy_b;         /* Dispersive (default 0.00420) */
  uint32_t thin_film;     /* 1: ThinFilm layer present (materials.rs:63-103, thin_film.rs) */
  float film_index;       /* ThinFilm refractive_index (default 1.5) */
  float film_thickness;   /* ThinFilm thickness in nm (default 500) */
  float density;          /* checker textures: cells per unit (spatial default 1, surface default 10) */
  float odd_color[3];     /* checker textures: odd cells, Xyz<E> */
  float spread;           /* ConeLight: half-angle of the emitting cone in degrees */
} clv_material;           /* 72 bytes */

/* CameraInit + scene times (camera.rs:40-54, scenefile.rs:21-29). */
typedef struct {
  float look_from[3];
  float look_at[3];
  float up[3];
  float vertical_fov;     /* degrees */
  float aperture;
  float focus_distance;
  float time_0, time_1;
} clv_camera_init;

typedef enum { CLV_BVH_LAM = 0, CLV_BVH_SAH = 1 } clv_bvh_algorithm; /* bvh.rs:32-40 */

typedef struct {
  uint32_t abi_version;           /* must be CLV_ABI_VERSION */
  uint32_t n_objects;
  const clv_object *objects;      /* in scene-file order (affects only BVH shape) */
  uint32_t n_materials;
  const clv_material *materials;
  uint32_t n_xforms;
  const clv_xform *xforms;
  clv_camera_init camera;
  float background[3];            /* Xyz<E> of the scene background (scenefile.rs:43-44) */
  uint32_t mis_bvh_algorithm;     /* clv_bvh_algorithm of both trees, as the reference builds them
                                     (scenefile.rs:106-108): the multiple-importance-sampling tree, whose
                                     shape sets light-selection probabilities, and the scene tree built on
                                     the host (a LAM or binned-SAH binary tree collapsed to 4-wide nodes;
                                     its shape only decides which of two equally distant hits is reported).
                                     The device builder (clv_scene_upload_ex) clusters regardless. */
} clv_scene_desc;

/* --------------------------------------------------------------- render --- */

typedef enum {
  CLV_GUIDE_OFF = 0,      /* plain method: the reference's light/BSDF mixture (trace.rs:80-120) */
  CLV_GUIDE_ON = 1        /* learned vMF-mixture proposal, one-sample MIS with the plain mixture */
} clv_guiding;

/* RenderOptions (clovers-cli/src/render.rs:17-49) plus the seed that replaces
 * the reference's OS-seeded per-row generators (draw_cpu.rs:56,62). */
typedef struct {
  uint32_t width, height;
  uint32_t samples;        /* spp */
  uint32_t max_depth;      /* trace() returns 0 once depth > max_depth (trace.rs:35) */
  uint64_t seed;           /* per-path PCG streams are keyed by (seed, pixel, sample) */
  uint32_t sample_offset;  /* first sample index (progressive rendering / sharding by sample) */
  uint32_t guiding;        /* clv_guiding */
  uint32_t fp64_accum;     /* 1: accumulate per-pixel sums in f64 */
  uint32_t flags;          /* CLV_FLAG_* */
} clv_render_opts;

#define CLV_FLAG_TIME_KERNELS 1u  /* time every traversal launch with HIP events (clv_counters.extend_ms) */
#define CLV_FLAG_COUNT 2u         /* counting traversal: node visits / primitive tests (slower) */
#define CLV_FLAG_GUIDE_FROZEN 4u  /* guided jobs sample with the network but never train it (ablation, or a
                                     network trained earlier with CLV_FLAG_GUIDE_KEEP): no training slices */
#define CLV_FLAG_GUIDE_KEEP 8u    /* guided jobs start from the context's current network instead of a fresh one */

/* RenderMode (clovers-cli/src/render.rs:52-62). */
typedef enum {
  CLV_MODE_PATH_TRACING = 0,          /* clv_render / clv_render_batch */
  CLV_MODE_NORMAL_MAP = 1,            /* first-hit normal as a colour (draw_cpu.rs:148-166, normals.rs:9-33) */
  CLV_MODE_BVH_TEST_COUNT = 2,        /* BVH nodes visited by the pixel's ray, as a colour ramp */
  CLV_MODE_PRIMITIVE_TEST_COUNT = 3   /* primitives tested by the pixel's ray, as a colour ramp
                                         (draw_cpu.rs:168-207, debug_visualizations.rs:9-61) */
} clv_render_mode;

/* Counters of the last clv_render / clv_primary_hits on a context. */
typedef struct {
  uint64_t samples;          /* camera paths traced */
  uint64_t rays;             /* extension rays traced (all bounces) */
  uint64_t node_visits;      /* wide-BVH nodes fetched (CLV_FLAG_COUNT only, else 0) */
  uint64_t prim_tests;       /* primitives tested (CLV_FLAG_COUNT only, else 0) */
  double render_ms;          /* device time of the render, HIP events on the context's stream */
  double extend_ms;          /* summed device time of the traversal launches (CLV_FLAG_TIME_KERNELS) */
  double build_ms;           /* host time of the last clv_scene_upload (spectra + BVHs) */
  uint32_t extend_launches;  /* traversal launches of the render; one per pass that runs whole paths */
  uint32_t passes;           /* passes (each covers a block of samples of every pixel) */
  uint32_t bvh_nodes;        /* wide nodes of the scene BVH */
  uint32_t bvh_width;        /* children per node */
  uint32_t node_bytes;       /* bytes per wide node */
  uint32_t prim_bytes;       /* bytes of primitive records / number of primitives */
  uint32_t n_prims;          /* primitives after flattening (a Boxy is 6) */
  uint32_t bvh_depth;        /* depth of the wide BVH */
  uint64_t guide_queries;    /* guided renders: network evaluations (one per guided diffuse vertex) */
  uint64_t guide_records;    /* guided renders: training records used (summed over steps) */
  double guide_infer_ms;     /* device time of the network evaluations (CLV_FLAG_TIME_KERNELS) */
  double guide_train_ms;     /* device time of the training rounds (CLV_FLAG_TIME_KERNELS) */
  uint32_t guide_rounds;     /* training rounds run */
  uint32_t _pad;
} clv_counters;

typedef struct clv_ctx clv_ctx;

/* Create a context on HIP device `hip_device` (binds the device and a stream). */
clv_status clv_create(int hip_device, clv_ctx **out);
/* Free every device allocation of the context. NULL is accepted. */
void clv_destroy(clv_ctx *ctx);
/* Human-readable detail of the last failure on ctx (valid until the next call). */
const char *clv_last_error(const clv_ctx *ctx);

/* Build (host: spectra, instance chains, BVH) and upload a scene.
 * Replaces SceneFile::initialize's BVH builds (scenefile.rs:104-109).
 * The scene stays resident in HBM until clv_scene_free or clv_destroy. */
clv_status clv_scene_upload(clv_ctx *ctx, const clv_scene_desc *desc, uint32_t *scene_id);

/* clv_scene_upload with a choice of scene-BVH builder.  CLV_BUILD_HOST is the
 * host binned-SAH build of clv_scene_upload.  CLV_BUILD_DEVICE packs the
 * primitive records on the host and builds the tree on the GPU (Morton sort,
 * PLOC clustering, breadth-first collapse into 4-wide nodes): the same node
 * and record layout, a different tree.  Renders agree with the host build's
 * up to ties between equally distant hits.  A device-built tree deeper than
 * the traversal stack allows is CLV_EUNSUPPORTED.  No reference counterpart:
 * the reference builds on the host only (bvh/build/surface_area_heuristic.rs:18-156). */
typedef enum { CLV_BUILD_HOST = 0, CLV_BUILD_DEVICE = 1 } clv_scene_builder;
clv_status clv_scene_upload_ex(clv_ctx *ctx, const clv_scene_desc *desc, uint32_t builder, uint32_t *scene_id);
clv_status clv_scene_free(clv_ctx *ctx, uint32_t scene_id);

/* Host-only scene check, no device needed: runs the full host build (spectra,
 * flattening, scene BVH, light tree) and reports its shape.  The counterpart of
 * the reference's `validate` subcommand (clovers-cli/src/validate.rs:14-30),
 * which initialises a scene and reports success or the failure. */
typedef struct {
  uint32_t n_objects;
  uint32_t n_prims;        /* after flattening (a Boxy is 6 quads) */
  uint32_t n_lights;       /* multiple-importance-sampling targets */
  uint32_t bvh_nodes;      /* 4-wide nodes */
  uint32_t bvh_depth;
  uint32_t light_nodes;    /* binary light-tree nodes */
  uint64_t device_bytes;   /* HBM the scene occupies once uploaded */
  double build_ms;
  char error[256];         /* empty on success */
} clv_scene_info;
clv_status clv_scene_validate(const clv_scene_desc *desc, clv_scene_info *info);

/* Scene files, no device needed.  Parses the reference's scene-file JSON --
 * SceneFile::initialize (clovers-cli/src/scenefile.rs:34-117 with
 * json_scene.rs:12-27) and object_to_hitable (clovers/src/objects.rs:92-157),
 * including STL / PLY meshes (objects/stl.rs:38-96, objects/ply.rs:37-103)
 * -- into a descriptor owned by the returned handle, ready for
 * clv_scene_upload / clv_scene_validate.  json: the file's text,
 * NUL-terminated.  mesh_root: directory that relative mesh paths are read
 * from (NULL: the working directory, as the reference).  bvh_algorithm: the
 * clv_bvh_algorithm of the light-sampling tree.  Kinds the reference's
 * schema has but this library does not render are CLV_EUNSUPPORTED; inputs
 * on which the reference panics are CLV_EINVAL.  err (nullable) receives the
 * reason. */
typedef struct clv_scene_file clv_scene_file;
clv_status clv_scene_file_parse(const char *json, const char *mesh_root, uint32_t bvh_algorithm,
                                clv_scene_file **out, char *err, uint32_t err_len);
/* The parsed descriptor; valid until clv_scene_file_free. */
const clv_scene_desc *clv_scene_file_desc(const clv_scene_file *file);
void clv_scene_file_free(clv_scene_file *file);

/* Image files of a clv_render pixel buffer (W*H*3 floats, Xyz<E>, row 0 =
 * top), no device needed.  clv_write_png == write::png (clovers-cli/src/
 * write.rs:18-84): sRGB 8-bit (Bradford E -> D65, sRGB transfer function,
 * clamped), with a tEXt "Comment" (comment, nullable) and "Software".
 * clv_write_exr == write::exr (write.rs:86-125): float R/G/B = X/Y/Z with the
 * XYZ chromaticities attribute, uncompressed scanlines. */
clv_status clv_write_png(const float *xyz, uint32_t width, uint32_t height, const char *path, const char *comment);
clv_status clv_write_exr(const float *xyz, uint32_t width, uint32_t height, const char *path);

/* == draw_cpu::draw for RenderMode::PathTracing (draw_cpu.rs:26-146).
 * xyz_out: caller-allocated W*H*3 floats (row 0 = top, index = x + row*W),
 * the per-pixel mean over opts->samples.  xyz_sq_out (nullable): per-pixel
 * mean of the squared per-sample contribution, for Monte Carlo error bars.
 * Blocking. */
clv_status clv_render(clv_ctx *ctx, uint32_t scene_id, const clv_render_opts *opts,
                      float *xyz_out, float *xyz_sq_out);

/* The debug render modes (CLV_MODE_NORMAL_MAP, _BVH_TEST_COUNT,
 * _PRIMITIVE_TEST_COUNT): one ray per pixel through the pixel's corner with
 * no lens offset, colours as the reference's (linear sRGB -> Xyz<E>), same
 * output layout as clv_render.  Counts are this library's: 4-wide BVH nodes
 * fetched and primitives tested (the reference counts its binary tree), with
 * the reference's ramp: grey n/255 up to 255, yellow to 511, orange to 1023,
 * red beyond.  opts: width, height, seed, sample_offset (the stream index). */
clv_status clv_render_debug(clv_ctx *ctx, uint32_t scene_id, const clv_render_opts *opts, uint32_t mode,
                            float *xyz_out);

/* One job of a batched render: one view of one uploaded scene.  No reference
 * counterpart -- the reference renders one scene per process run
 * (clovers-cli/src/render.rs:137-176); this is how a caller renders several
 * views or scenes in one go.  Jobs of different scenes, sizes, sample counts
 * and depths share the wavefront passes of one launch sequence. */
typedef struct {
  uint32_t scene_id;
  uint32_t use_camera;       /* 1: `camera` replaces the scene's camera for this job */
  clv_camera_init camera;
  uint32_t _pad;
  clv_render_opts opts;      /* per job: size, spp, depth, seed, sample_offset, fp64_accum, guiding;
                                flags are OR-ed over the batch */
  float *xyz_out;            /* W*H*3 floats, as clv_render */
  float *xyz_sq_out;         /* nullable, as clv_render */
} clv_job;                   /* 128 bytes */

/* Render every job (at most 8192, at most 2^28 pixels in all).  Each job's
 * output equals what clv_render gives for it alone: paths are keyed by
 * (job seed, pixel, sample), so batching does not change any path.  Blocking.
 * clv_counters then covers the whole batch (BVH fields: the job with the most
 * samples). */
clv_status clv_render_batch(clv_ctx *ctx, const clv_job *jobs, uint32_t n_jobs);

/* Launch shapes of a context.  No reference counterpart (the reference has no
 * device launches); set by clv_autotune or by hand. */
typedef enum {
  CLV_TRACE_SIMPLE = 0,     /* one ray per thread, 256-thread blocks, stack top in LDS */
  CLV_TRACE_PERSISTENT = 1, /* persistent waves refilling lanes from a work counter */
  CLV_TRACE_WW = 2,         /* one ray per thread, node steps and leaf steps in separate loops */
  CLV_TRACE_LDS_CACHED = 3  /* 768-thread blocks, top of the BVH and leading records cached in LDS; renders without
                               guided jobs run every path from the camera to its end in one launch per pass, from
                               LDS if the scene of all jobs fits in lds_bytes whole, else from memory; guided
                               renders read the scene from memory where LDS holds less than half of it */
} clv_trace_kernel;
typedef struct {
  uint32_t target_paths;    /* samples per wavefront pass (queue and path-state capacity).  The default, 2^22,
                               stands for the automatic size; any other value is kept to (2^22 - 1 asks for passes
                               of the default size and no larger ones).  Automatic: a pass that runs whole paths in
                               one launch (CLV_TRACE_LDS_CACHED, no guided job, no CLV_FLAG_TIME_KERNELS or _COUNT)
                               holds up to 2^27, at 12 bytes per sample beside up to 140 MB of traversal stacks;
                               wavefront passes behind the last training round are joined up to 2^25 (9.2 GB).  Where
                               memory is short, both keep to 2^22; a later call that finds none gets theirs */
  uint32_t trace_kernel;    /* clv_trace_kernel */
  uint32_t lds_bytes;       /* dynamic LDS per block of CLV_TRACE_LDS_CACHED (<= 64512) */
  uint32_t shade_grid_cap;  /* largest grid of the shading kernel, in 256-thread blocks (the library also caps it
                               at the blocks of the launched instance that fit on the device at once) */
  uint32_t guide_train_spp; /* guided jobs: samples per pixel of each training pass (default 4) */
  float guide_alpha;        /* at a diffuse vertex, share of the cosine half of the mixture drawn from the
                               learned lobes (default 0.5) */
  float guide_lr;           /* Adam learning rate (default 0.005) */
  uint32_t guide_records;   /* training records used per round (default 2^21, in steps of 16384) */
  float guide_wclip;        /* training weight F/p capped at this multiple of its mean (default 1e6) */
  uint32_t guide_rounds;    /* training rounds after passes of a guided render (default 1); later samples use
                               the trained network in large passes without training */
  uint32_t use_graph;       /* 1 (default): a render repeated with identical arguments is captured as a hipGraph
                               on its second call and replayed from then on; never for CLV_FLAG_TIME_KERNELS
                               or a batch with a guided job */
  uint32_t guide_credit;    /* radiance a training record is credited with: 1 (default) only what arrives
                               through a specular chain or further bounces (direct light is the light-tree
                               half's to sample); 0 everything that reaches the path after the vertex */
  uint32_t guide_warmup;    /* 0 (default): the training rounds' samples are the guided job's first samples;
                               1: they are extra warm-up samples the image never sees (stream indices from
                               2^31 on), so every image sample uses the trained network */
  uint32_t tail_depth;      /* 0 (default): every bounce of a pass is a traversal and a shading launch over the
                               live paths; d > 0: from bounce d on, one launch traces and shades each remaining
                               path to its end (the same results; fewer launches when few paths are left);
                               without effect where whole paths run in one launch (trace_kernel) */
  uint32_t guide_photons;   /* light-traced training records per round (default 2^20, at most 2^24; 0 = none):
                               paths from the emitters aimed at the light-sampling targets, recorded at their
                               first diffuse hit after a specular chain */
  uint32_t guide_pre_rounds;/* with guide_photons: training rounds on light-traced records alone before a guided
                               render's first pass, so its first samples already use the network (default 8) */
  float guide_gate_density; /* with guide_photons: a 64^3 grid over each guided job's scene box counts where the
                               light-traced records land; a diffuse vertex uses the learned lobes only in a cell
                               whose 3x3x3 neighbourhood holds, per cell, at least this multiple of the job's
                               records spread evenly over one 64x64 plane of the grid (or in every cell if the
                               job received none); elsewhere it samples the plain mixture and the network is
                               not evaluated.  Default 0.5; 0 = lobes everywhere */
} clv_tuning;
clv_status clv_tuning_get(const clv_ctx *ctx, clv_tuning *out);
clv_status clv_tuning_set(clv_ctx *ctx, const clv_tuning *t);
/* Autotuner: renders a shortened copy of the batch (the same jobs with fewer
 * samples, about `trial_samples` in all; 0 = 64M) under each candidate launch
 * shape -- the automatic pass size (2^22) and 2^23..2^26 paths (sizes that give
 * other passes than it) x {LDS-cached traversal with a 64 KB or 16 KB cache,
 * plain traversal}, then the best of them with tail_depth 2, 3 and 4 unless a
 * job is guided or whole paths run in one launch -- keeps the fastest on the
 * context and returns it.  Outputs of the trials are discarded. */
clv_status clv_autotune(clv_ctx *ctx, const clv_job *jobs, uint32_t n_jobs, uint64_t trial_samples,
                        clv_tuning *best_out);

/* The plan of passes of `tuning`'s size for `jobs` (target_paths,
 * guide_train_spp, guide_rounds), computed on the host, no device or uploaded
 * scene needed (scene ids are not looked up).  clv_render_batch follows it,
 * except that at the default target_paths it runs larger passes (see there).  Items are
 * in pass order; up to `cap` are written, *n_items and *n_passes receive the
 * full counts. */
typedef struct {
  uint32_t pass;         /* pass index */
  uint32_t job;          /* index into jobs */
  uint32_t samples;      /* samples per pixel of the job in this pass */
  uint32_t sample_base;  /* absolute index of the slice's first sample */
  uint32_t pass_paths;   /* paths of the whole pass */
  uint32_t train;        /* 1: a training round of the guiding network follows the pass */
  uint32_t warmup;       /* 1: warm-up samples (clv_tuning.guide_warmup): not in the image */
} clv_pass_item;
clv_status clv_plan_passes(const clv_job *jobs, uint32_t n_jobs, const clv_tuning *tuning, clv_pass_item *items,
                           uint32_t cap, uint32_t *n_items, uint32_t *n_passes);

/* Guiding network probes (no reference counterpart: the learned proposal is
 * this library's own).  The network maps (position normalised to the scene
 * box, oriented normal, (lambda - 380) / 400) to 8 vMF lobes; its fp32
 * parameter vector has CLV_GUIDE_NPARAM entries (W1 b1 W2 b2 W3 b3 W4 b4,
 * W row-major [out][in]: 64x64, 64x64, 64x64, 48x64 with output rows 40..47
 * unused).  A guided render starts from a fresh network seeded by the job's
 * seed unless CLV_FLAG_GUIDE_KEEP is set. */
#define CLV_GUIDE_NPARAM 15600u
#define CLV_GUIDE_OUT 40u
/* fresh parameters from `seed` */
clv_status clv_guide_reset(clv_ctx *ctx, uint64_t seed);
clv_status clv_guide_params(clv_ctx *ctx, float *params_out, uint32_t n);
clv_status clv_guide_set_params(clv_ctx *ctx, const float *params, uint32_t n);
/* forward pass on the device: inputs n x 7 (p xyz, normal xyz, lambda);
 * raw_out n x 40 network outputs; lobes_out n x 40 (per lobe mu xyz, kappa,
 * mixture weight).  Either output may be NULL. */
clv_status clv_guide_eval(clv_ctx *ctx, const float *inputs, uint32_t n, float *raw_out, float *lobes_out);
/* gradient of the training loss on the device, without an update: samples
 * n x 11 (p xyz, normal xyz, lambda, direction xyz, weight F/p > 0); loss =
 * mean over samples of -(w / mean w) log q(direction); grad_out receives
 * CLV_GUIDE_NPARAM floats. */
clv_status clv_guide_grad(clv_ctx *ctx, const float *samples, uint32_t n, float *grad_out);

/* Primary-ray closest hits for sample `opts->sample_offset` of every pixel,
 * same camera and ray seeds as clv_render (the parity probe of the hit path).
 * prim_id_out: W*H ids, object_index*8 + face (face = 0..5 for a Boxy side,
 * else 0), 0xFFFFFFFF on a miss.  t_out: W*H hit distances (nullable). */
clv_status clv_primary_hits(clv_ctx *ctx, uint32_t scene_id, const clv_render_opts *opts,
                            uint32_t *prim_id_out, float *t_out);

/* clv_primary_hits for callers that cannot allocate (code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc).  No
 * counterpart in the reference.  Same results and argument meaning as
 * clv_primary_hits, except that prim_id_out and t_out (nullable) are DEVICE
 * memory of the context's device, W*H entries each.  The call allocates
 * nothing: its working memory is one fixed device array per GPU
 * (CLV_NOALLOC_SCRATCH_BYTES, held until the process ends) and the scene
 * must already be uploaded.  At most CLV_NOALLOC_MAX_PIXELS pixels per call
 * (CLV_EINVAL beyond).  Every call on a GPU shares that GPU's array, so calls
 * that overlap on one GPU (several contexts, several host threads) race.
 * Blocking, like clv_primary_hits. */
#define CLV_NOALLOC_SCRATCH_BYTES 20972288u
#define CLV_NOALLOC_MAX_PIXELS (1u << 27)
clv_status clv_primary_hits_noalloc(clv_ctx *ctx, uint32_t scene_id, const clv_render_opts *opts,
                                    uint32_t *prim_id_out, float *t_out);

/* Counters of the last render on ctx. */
clv_status clv_counters_get(const clv_ctx *ctx, clv_counters *out);

/* Library ABI version (CLV_ABI_VERSION the library was built with). */
uint32_t clv_abi_version(void);

/* Host-side spectral helpers, no device needed.
 * clv_spectral_power: clovers::spectrum::spectral_power (clovers/src/spectrum.rs:46-56),
 *   Meng et al. 2015 upsampling of an Xyz<E> colour at an integer wavelength in nm.
 * clv_wavelength_into_xyz: clovers::wavelength::wavelength_into_xyz
 *   (clovers/src/wavelength.rs:62-83) for lambda in [380, 780); CLV_EINVAL outside. */
float clv_spectral_power(const float xyz[3], uint32_t lambda);
clv_status clv_wavelength_into_xyz(uint32_t lambda, float xyz_out[3]);

#ifdef __cplusplus
}
#endif
#endif /* CLOVERS_HIP_H */
