/* kernels.h -- device-side views of the scene and path state, and the kernel
 * launchers (implemented in kernels.hip). */
#ifndef CLV_KERNELS_H
#define CLV_KERNELS_H
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/clovers_hip.h"
#include "clv_layout.h"
#include "guide.h"

namespace clv {

/* slots of the per-render counter array */
#define CNT_QA 0u       /* ray queue A size */
#define CNT_QB 1u       /* ray queue B size */
#define CNT_SHADE 2u    /* MC_COUNT shading queue sizes start here */
#define CNT_FETCH 7u    /* work counter of the persistent traversal */
#define CNT_TOTAL 8u

/* path meta word: hero wavelength index | depth | job of the batch */
#define META_HERO_MASK 0x1FFu
#define META_DEPTH_SHIFT 9u
#define META_DEPTH_MASK 0x3FFu   /* max_depth <= 1000 */
#define META_JOB_SHIFT 19u
#define MAX_JOBS 8192u           /* 13 bits of job index */

/* The scene arena: every uploaded scene lives in these arrays with global
 * indices (child words, record offsets, material / SPD / light indices are
 * rebased at upload), so one traversal launch serves rays of any scene; a ray
 * starts at its job's root node. */
struct DevScene {
  const Bvh4Node *nodes;
  const float4 *prims;
  const PrimInfo *info;
  const Xform *xforms;
  const DevMaterial *mats;
  const float *spd;
  const DevLight *lights;
  const DevLightNode *lnodes;
  const float *lweights;
  const DevJob *jobs;
  uint32_t has_xforms;    /* some scene of the batch has instance chains */
  uint32_t has_ext;       /* some scene of the batch has checker textures, cone lights or media */
  uint32_t has_media;     /* some scene of the batch has constant media */
};

/* Structure-of-arrays path state.  A pass has one slot per sample (a pixel
 * and sample index of one job).  The live paths of a bounce are kept
 * compacted: entry e of the moving arrays is the e-th live path, so the
 * traversal reads its rays contiguously; shading writes the survivors,
 * compacted again, into the other half of a ping-pong pair (n_*).  What a
 * path accumulates (radiance) and what the estimator needs (hero index) stay
 * at the path's slot. */
struct PathBuf {
  /* by entry, this bounce */
  float4 *ray_o;    /* origin, .w = the root node of the path's scene */
  float4 *ray_d;    /* unit direction, .w = the ray's time */
  float4 *thr;      /* throughput, 4 hero wavelengths */
  uint64_t *rng;    /* PCG32 state */
  uint32_t *meta;   /* META_*: hero wavelength index, depth, job */
  uint32_t *slot;   /* the path's slot */
  float *hit_t;
  uint32_t *hit_p;  /* primitive record offset of the closest hit, ~0u on a miss */
  /* by entry, next bounce (shading writes the survivors here) */
  float4 *n_ray_o, *n_ray_d, *n_thr;
  uint64_t *n_rng;
  uint32_t *n_meta, *n_slot;
  /* by slot */
  float4 *rad;      /* accumulated radiance, 4 hero wavelengths */
  uint32_t *hero;   /* hero wavelength index (for the estimator) */
  uint32_t *gcnt;   /* guided renders: diffuse vertices recorded per path this pass (else NULL) */
  float *recL;      /* guided renders, by slot x GD_SLOTS: hero radiance that arrived along each
                       training record's direction afterwards (sum of c / t0); zeroed per pass, so
                       the training round scans 4 bytes per record */
};

/* guided sampling state of a pass */
struct GuideArgs {
  uint32_t *lobes;         /* [path][GD_LWORDS]: the lobes of the path's current diffuse vertex */
  GuideRec *rec;           /* [path][GD_SLOTS] training records */
  const _Float16 *Wh;      /* fp16 operand copies of the network */
  const float *P;          /* fp32 parameters (biases) */
  float alpha;             /* probability of drawing from the lobes; 0 = plain sampling */
  uint32_t stamp;          /* pass id written into records */
  uint32_t record;         /* write training records */
  uint32_t on;             /* the batch has guided jobs: lobes/rec/gcnt are valid */
  uint32_t indirect;       /* 1: a record is not credited with emission reached straight from it
                              (direct light, which the light-tree half samples), only through a
                              specular chain or further bounces */
  unsigned long long *stats; /* stats[3] counts network evaluations */
  const uint8_t *gate;     /* [job][GD_CELLS] open cells of the guiding gate, or NULL: guide everywhere */
};

struct ShadeQueues {
  uint32_t *q[MC_COUNT];
  uint32_t *counts; /* = counter array + CNT_SHADE */
};

/* arguments of the persistent traversal kernel */
struct TraceArgs {
  uint32_t *counts;            /* counter array (queue sizes, fetch counter) */
  uint32_t in_slot;            /* extend mode: slot of the ray-queue size */
  uint32_t n_direct;           /* primary mode: number of rays (paths 0..n-1) */
  ShadeQueues sq;              /* extend mode: shading queues */
  uint32_t *spill;             /* per-thread overflow of the traversal stack */
  unsigned long long *stats;   /* counting mode: node visits, primitive tests */
  uint32_t *ids;               /* primary mode outputs */
  float *ts;
  uint32_t *ray_counts;        /* primary counting mode (nullable): per ray node visits, primitive tests */
  uint32_t lds_node_base;      /* LDS variant: nodes [base, base + lds_nodes) are cached in LDS */
  uint32_t lds_nodes;
  uint32_t lds_unit_base;      /* LDS variant: primitive float4 units [base, base + lds_units) are cached */
  uint32_t lds_units;
};

struct GenParams {
  const DevItem *items;   /* the pass' items, ordered by path_base */
  uint32_t n_items;
  uint32_t paths;         /* total paths of the pass */
};

/* one sample's XYZ contribution */
struct F3 {
  float x, y, z;
};

/* arguments of the whole-path kernel (k_paths) */
struct PathsArgs {
  uint32_t *next;              /* cursor over the pass' samples */
  uint32_t *spill;             /* per-thread overflow of the traversal stack */
  unsigned long long *stats;   /* stats[2] counts rays */
  F3 *res;                     /* by slot: the sample's contribution */
  const float4 *cie;
  uint32_t lds_node_base, lds_nodes, lds_unit_base, lds_units; /* as TraceArgs */
  uint32_t first;              /* samples a block starts with: [block * first, + first) */
  uint32_t full;               /* every ray's scene is the one in the window, and it is in there whole */
  uint32_t chunk;              /* samples a block takes from the cursor at a time, at least the block size */
};

struct ResolveParams {
  const DevItem *items;   /* the pass' items (resolve) */
  uint32_t n_items;
  uint32_t threads;       /* resolve: sum of the items' pixels */
  const DevJob *jobs;     /* finalize / zero: all jobs */
  uint32_t n_jobs;
  uint32_t pixels;        /* finalize / zero: sum of all jobs' pixels */
  float *acc32;           /* 3 per pixel */
  double *acc64;          /* 3 per pixel */
  double *acc_sq;         /* 3 per pixel */
};

/* stats: 8 x u64 = node visits, primitive tests, rays traced, network evaluations, training records used */
void launch_reset_counts(hipStream_t st, uint32_t *counts, uint32_t in_slot, uint32_t out_slot, uint64_t *stats);
void launch_set_count(hipStream_t st, uint32_t *counts, uint32_t slot, uint32_t value);
/* zero n 64-bit words with a kernel (a memset node misbehaves in captured graphs) */
void launch_zero_u64(hipStream_t st, uint64_t *p, uint32_t n);
void launch_generate(hipStream_t st, const DevScene &sc, const PathBuf &pb, const GenParams &gp);
/* persistent traversal: grid = resident blocks of the device; spill buffer of
 * trace_spill_words(blocks) words */
uint32_t trace_grid_blocks();
size_t trace_spill_words(uint32_t blocks);
/* traversal kernel variants: one ray per thread over a static grid-stride
 * loop, or persistent waves refilling lanes from an atomic work counter */
#define TRACE_SIMPLE 0
#define TRACE_PERSISTENT 1
#define TRACE_MAJORITY 4 /* only chosen by the library (guided bounces from memory) */
#define TRACE_WW 2
#define TRACE_LDS 3
/* LDS-cached traversal: dynamic LDS bytes for a cached prefix of `nodes` wide
 * nodes and `units` primitive float4, resident blocks for that size, and the
 * spill words its grid needs; mode 0 = extend, 1 = primary */
size_t lds_trace_bytes(uint32_t nodes, uint32_t units);
uint32_t lds_trace_stack_bytes();
size_t lds_trace_spill_words(uint32_t blocks);
uint32_t lds_trace_grid_blocks(size_t lds_bytes);
void launch_trace_lds(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta, uint32_t blocks,
                      size_t lds_bytes, bool counting, int mode);
void launch_extend(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta, uint32_t blocks,
                   bool counting, int variant);
void launch_primary(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta, uint32_t blocks,
                    int variant);
/* debug render modes: one ray per pixel, closest hit with per-ray counts, colours */
struct DebugArgs {
  uint32_t width, height, sample, mode;   /* mode: clv_render_mode */
  float lin_to_xyz[9];                    /* linear sRGB -> Xyz<E>, row-major */
};
void launch_generate_debug(hipStream_t st, const DevScene &sc, const PathBuf &pb, const DebugArgs &da);
void launch_primary_counting(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta, uint32_t blocks);
void launch_debug_color(hipStream_t st, const DevScene &sc, const PathBuf &pb, const DebugArgs &da,
                        const uint32_t *ray_counts, float *out);
/* resident blocks of each shading instance (index 2 * guided + extended) on the current device */
void shade_grid_blocks(uint32_t out[4]);
void launch_shade(hipStream_t st, const DevScene &sc, const PathBuf &pb, const ShadeQueues &sq, uint32_t *counts,
                  uint32_t out_slot, uint32_t max_paths, uint32_t grid_cap, const uint32_t resident[4],
                  const GuideArgs &ga);
/* learned-proposal lobes for the Lambertian queue of the current bounce */
/* allocation-free primary-hit probe (clv_primary_hits_noalloc): camera rays
 * per launch pair, traversal grid, and the device scratch that holds them */
#define NA_CHUNK 65536u
#define NA_BLOCKS 256u
#define NA_SCRATCH_BYTES 20972288u
struct NaView {
  DevJob *job;
  DevItem *item;
  uint32_t *counts;
  float *ts;         /* distances when the caller wants none */
  uint32_t *spill;   /* traversal stack overflow of the NA_BLOCKS grid */
  PathBuf pb;        /* path state of NA_CHUNK rays */
};
int na_scratch_address(void **out);
NaView na_view(void *base);
void launch_na_setup(hipStream_t st, const DevJob &jb, const DevItem &it, const NaView &v);
/* the rest of a pass' bounces in one launch (k_tail): entries of counts[ta.in_slot] */
void launch_tail(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta, uint32_t blocks,
                 const GuideArgs &ga);
uint32_t guide_photon_grid_blocks();
/* light-traced training records (k_guide_photons): n paths over the batch's
 * jobs into rec/recL[0, n), their streams keyed by (seed, round, path); grid
 * of at most `blocks` traversal blocks with a spill buffer of
 * trace_spill_words(blocks) words */
void launch_guide_photons(hipStream_t st, const DevScene &sc, uint32_t n_jobs, GuideRec *rec, float *recL, uint32_t n,
                          uint32_t stamp, uint32_t round, uint64_t seed, uint32_t *spill, uint32_t blocks,
                          uint32_t *fresh, uint32_t copies);
/* the guiding gate: the record counts of the latest round, fresh[copies][job]
 * [GD_CELLS], go into cells[job][GD_CELLS] and the job totals cell_tot[job] and
 * are cleared; then gate[job][GD_CELLS] from these */
void launch_guide_gate(hipStream_t st, uint32_t *fresh, uint32_t copies, uint32_t *cells, uint32_t *cell_tot,
                       uint8_t *gate, uint32_t n_jobs, float density);
uint32_t guide_infer_grid_blocks();
void launch_guide_infer(hipStream_t st, const DevScene &sc, const PathBuf &pb, const GuideArgs &ga,
                        const uint32_t *queue, const uint32_t *count, uint32_t max_paths, uint32_t resident);
/* guide.hip: record compaction, training steps, network probes */
void launch_guide_collect(hipStream_t st, const GuideRec *rec, const float *recL, uint32_t n, uint32_t *bcount,
                          float *bweight, uint32_t *totals, uint32_t *list, uint32_t cap, unsigned long long *used);
/* one Adam step on records [step_base, step_base + step_len) of the round's
 * list; totals[3] counts the steps taken with records (bias corrections) */
void launch_guide_step(hipStream_t st, const GuideRec *rec, const float *recL, const uint32_t *list,
                       uint32_t *totals, uint32_t cap, uint32_t step_base, uint32_t step_len, float wclip,
                       float *P, float *m, float *v, _Float16 *Wh, float *partial, float lr, float *grad_out);
void launch_guide_halves(hipStream_t st, const float *P, _Float16 *Wh);
void launch_guide_eval(hipStream_t st, const float *in, uint32_t n, const _Float16 *Wh, const float *P, float *raw,
                       float *lobes);
/* whole paths in one launch (k_paths), from a scene in LDS (full) or in
 * memory: block size, dynamic LDS, resident blocks, spill words of a grid;
 * `begin` also clears the render's counters */
uint32_t paths_block(bool full);
size_t paths_lds_bytes(bool full, uint32_t nodes, uint32_t units);
uint32_t paths_grid_blocks(size_t lds_bytes, const DevScene &sc, bool full);
size_t paths_spill_words(bool full, uint32_t blocks);
void launch_paths(hipStream_t st, const DevScene &sc, const GenParams &gp, const PathsArgs &pa, uint32_t blocks,
                  size_t lds_bytes, bool begin);
void launch_resolve_xyz(hipStream_t st, const ResolveParams &rp, const F3 *res, float *out, float *out_sq);
void launch_resolve(hipStream_t st, const PathBuf &pb, const ResolveParams &rp, const float4 *cie);
void launch_finalize(hipStream_t st, const ResolveParams &rp, float *out, float *out_sq);
void launch_zero_accum(hipStream_t st, const ResolveParams &rp);

}  // namespace clv
#endif
