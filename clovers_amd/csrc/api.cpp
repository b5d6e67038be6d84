/*
 * api.cpp -- the C ABI (include/clovers_hip.h) over the HIP renderer.
 *
 * clv_render is the drop-in for draw_cpu::draw (clovers-cli/src/draw_cpu.rs:26-98,
 * called at clovers-cli/src/render.rs:149).  A render is a sequence of passes;
 * pass p covers samples [p*k, p*k+k) of every pixel.  A plain pass is one launch
 * that runs whole paths (k_paths) and one that sums them:
 *
 *   paths                          camera, bounces and estimator of every sample
 *   resolve                        per-pixel sums, in sample order
 *
 * Guided passes, and renders that are timed or counted per launch or tuned to
 * another traversal, are wavefronts:
 *
 *   generate                       camera rays of all paths of the pass
 *   repeat max_depth+1 times:      reset counters; extend; [infer;] shade
 *   resolve                        per-sample estimator, per-pixel sums
 *
 * All launches go to the context's stream; the host never waits inside a
 * render (queue sizes stay on the device, kernels read them), so the launch
 * sequence of a pass is fixed and the driver pipelines it.
 */
#include <hip/hip_runtime.h>
#include <float.h>
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <map>
#include <memory>
#include <new>
#include <string>
#include <vector>

#include "../../include/clovers_hip.h"
#include "bvh_build.h"
#include "copyout.h"
#include "host_build.h"
#include "kernels.h"

using namespace clv;

static_assert(CLV_TRACE_SIMPLE == TRACE_SIMPLE && CLV_TRACE_PERSISTENT == TRACE_PERSISTENT && CLV_TRACE_WW == TRACE_WW &&
                  CLV_TRACE_LDS_CACHED == TRACE_LDS,
              "public and internal traversal kernel ids differ");

namespace {


/* one growable device array of the scene arena */
struct DevArray {
  char *p = nullptr;
  size_t used = 0, cap = 0;  /* bytes */
};

enum { AR_NODES, AR_PRIMS, AR_INFO, AR_XFORMS, AR_MATS, AR_SPD, AR_LIGHTS, AR_LNODES, AR_LWEIGHTS, AR_COUNT };

struct SceneRes {
  ArenaBase base;            /* element offsets of the scene in the arena */
  size_t end[AR_COUNT];      /* byte end of the scene in each array */
  uint32_t light_root = LT_EMPTY;
  uint32_t n_lights = 0;
  int32_t bg_spd = -1;
  bool has_xforms = false;
  bool has_ext = false;      /* checker textures, cone lights or constant media */
  uint32_t media_off = 0, n_media = 0;  /* constant-medium records (arena units) */
  clv_camera_init camera;
  uint32_t n_nodes = 0, n_prims = 0, prim_bytes = 0, depth = 0;
  uint32_t prim_units = 0;   /* float4 units of primitive records */
  float lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};  /* scene box (root node's child boxes) */
  double build_ms = 0.0;
};

/* the guiding network and its training buffers (allocated on first use) */
#define GUIDE_STEP 16384u /* default records per Adam step */

struct GuideState {
  float *P = nullptr, *M = nullptr, *V = nullptr;  /* fp32 parameters, Adam moments */
  _Float16 *Wh = nullptr;                          /* fp16 operand copies */
  float *partial = nullptr;                        /* gradient slices, one per 64 records of a step */
  uint32_t partial_groups = 0;
  uint32_t cap_lobes = 0;                          /* paths the lobes are kept for */
  uint32_t *lobes = nullptr;
  uint32_t cap_paths = 0;                          /* paths of a training pass: capacity of the buffers below */
  GuideRec *rec = nullptr;
  float *recL = nullptr;     /* radiance credited to each record this pass */
  uint32_t *gcnt = nullptr;
  uint32_t *list = nullptr;
  uint32_t *bcount = nullptr;
  float *bweight = nullptr;
  uint32_t *totals = nullptr;                      /* [0] valid records, [1] [2] mean weights, [3] Adam steps */
  uint32_t *host_totals = nullptr;                 /* pinned: a round's valid-record count read back */
  uint32_t stamp = 0;                              /* last pass id */
  bool init = false, trained = false;
  /* training schedule (clv_tuning) */
  uint32_t train_spp = 4;
  float alpha = 0.5f;
  float lr = 0.005f;
  uint32_t records = 2097152;
  float wclip = 1e6f;
  uint32_t rounds = 1;
  uint32_t credit = 1;       /* clv_tuning.guide_credit */
  uint32_t step = GUIDE_STEP; /* records per Adam step */
  uint32_t epochs = 1;        /* passes over a round's records */
  uint32_t warmup = 0;        /* clv_tuning.guide_warmup */
  uint32_t photons = 1u << 20; /* clv_tuning.guide_photons: light-traced records per training round */
  /* the guiding gate (guide.h GD_GRID): light-traced record counts per cell and job, their totals, the open cells */
  uint32_t *cells = nullptr, *cell_tot = nullptr;
  uint32_t *fresh = nullptr;   /* the counts of the round in flight, in gate_copies(jobs) copies of cells */
  uint8_t *gate = nullptr;
  uint32_t gate_jobs = 0;      /* jobs the buffers hold */
  bool gate_valid = false;     /* the gate has been built since the counts were cleared */
  float gate_density = 0.5f;   /* clv_tuning.guide_gate_density: a cell opens at this multiple of the job's
                                  records spread over one grid plane; 0 = no gate */
  uint32_t pre_rounds = 8;     /* clv_tuning.guide_pre_rounds: rounds on light-traced records alone before a
                                  guided render's first pass */
  uint32_t cap_photons = 0;
};

}  // namespace

struct clv_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  std::map<uint32_t, SceneRes *> scenes;
  uint32_t next_scene = 1;
  DevArray arena[AR_COUNT];
  uint32_t tile_order = 1;   /* render passes lay each sample's slots out in 8x8 pixel tiles */
  /* path state */
  uint32_t cap_paths = 0;
  PathBuf pb;                /* the view of even bounces; odd bounces swap the two entry sets */
  uint32_t *shadeq[MC_COUNT] = {nullptr};
  F3 *res = nullptr;         /* sample contributions of a whole-path pass, by slot */
  uint32_t cap_res = 0;
  /* wavefront [0] and whole-path [1] passes of an untuned context that found no memory: the smallest that failed
   * (0: none) and the device memory that was free beside them */
  struct {
    uint32_t paths = 0;
    size_t free = 0;
  } no_room[2];
  /* accumulators */
  uint32_t cap_pixels = 0;
  float *acc32 = nullptr;
  double *acc64 = nullptr, *accsq = nullptr;
  float *out = nullptr, *out_sq = nullptr;
  uint32_t *ids = nullptr;
  float *ts = nullptr;
  CopyOut copy;              /* results on their way to the caller's memory */
  /* job and pass-item tables of the current render */
  DevJob *jobs = nullptr;
  uint32_t cap_jobs = 0;
  DevItem *items = nullptr;
  uint32_t cap_items = 0;
  /* misc */
  uint32_t *counts = nullptr;
  uint64_t *stats = nullptr;
  uint32_t *spill = nullptr;      /* traversal stack overflow, one slice per launched thread */
  size_t spill_words = 0;         /* size of the spill buffer */
  size_t lds_block_bytes = 64512; /* dynamic LDS budget of one block of the LDS-cached traversal (64 KB less static use) */
  uint32_t trace_blocks = 0;      /* resident blocks of the persistent traversal */
  uint32_t infer_blocks = 1;      /* resident blocks of the network inference kernel */
  uint32_t photon_blocks = 1;     /* resident blocks of the light-traced records' kernel */
  uint32_t shade_blocks[4] = {1u << 30, 1u << 30, 1u << 30, 1u << 30}; /* resident blocks per shading instance */
  uint32_t tail_depth = 0;        /* bounce from which a pass finishes its paths in one launch (0: never) */
  void *na_scratch = nullptr;     /* this device's copy of the allocation-free probe's scratch array */
  int trace_variant = TRACE_LDS;
  bool full_grid = false;         /* one thread per possible ray instead of the resident grid */
  float4 *cie = nullptr;
  std::vector<hipEvent_t> events;
  clv_counters counters;
  uint32_t target_paths = 1u << 22;
  uint32_t grid_cap = 2048;
  GuideState guide;
  /* the last render's launch sequence as an executable graph, replayed when
   * an identical render (same signature) comes again */
  bool use_graph = true;
  hipGraphExec_t gexec = nullptr;
  std::string gsig;
  std::string last_sig;     /* signature of the previous eager render: a repeat is captured */
};

namespace {

/* the runtime keeps a failed call's error until it is asked: it is not the next call's, nor another library's */
clv_status fail(clv_ctx *c, clv_status s, const std::string &msg) {
  if (s != CLV_EINVAL) (void)hipGetLastError();
  if (c) c->err = msg;
  return s;
}

#define HIPCHK(ctx, expr)                                                                   \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess) {                                                                 \
      return fail((ctx), e_ == hipErrorOutOfMemory ? CLV_ENOMEM : CLV_EDEVICE,              \
                  std::string(#expr) + ": " + hipGetErrorString(e_));                       \
    }                                                                                       \
  } while (0)

#define CHK(expr)                       \
  do {                                  \
    clv_status s_ = (expr);             \
    if (s_ != CLV_OK) return s_;        \
  } while (0)

/* synchronises a stream when it goes out of scope: a function that queued
 * copies from its own host buffers must not let an error return free them
 * while the copies may still read them */
struct StreamDrain {
  hipStream_t s;
  ~StreamDrain() {
    if (s) (void)hipStreamSynchronize(s);
  }
};

template <typename T>
hipError_t dalloc(T **p, size_t n) {
  return hipMalloc((void **)p, n * sizeof(T) + 16);
}

void dfree(void *p) {
  if (p) (void)hipFree(p);
}

void free_paths(clv_ctx *c) {
  PathBuf &b = c->pb;
  dfree(b.ray_o); dfree(b.ray_d); dfree(b.thr); dfree(b.rng); dfree(b.meta); dfree(b.slot);
  dfree(b.n_ray_o); dfree(b.n_ray_d); dfree(b.n_thr); dfree(b.n_rng); dfree(b.n_meta); dfree(b.n_slot);
  dfree(b.hit_t); dfree(b.hit_p); dfree(b.rad); dfree(b.hero);
  for (uint32_t k = 0; k < MC_COUNT; k++) dfree(c->shadeq[k]);
  memset(&c->pb, 0, sizeof(c->pb));
  for (uint32_t k = 0; k < MC_COUNT; k++) c->shadeq[k] = nullptr;
  c->cap_paths = 0;
}

/* the path state of bounce `depth`: entries in one set, survivors to the other */
PathBuf bounce_view(const PathBuf &pb, uint32_t depth) {
  PathBuf v = pb;
  if (depth & 1u) {
    std::swap(v.ray_o, v.n_ray_o);
    std::swap(v.ray_d, v.n_ray_d);
    std::swap(v.thr, v.n_thr);
    std::swap(v.rng, v.n_rng);
    std::swap(v.meta, v.n_meta);
    std::swap(v.slot, v.n_slot);
  }
  return v;
}

clv_status ensure_spill(clv_ctx *c, size_t words) {
  if (words <= c->spill_words) return CLV_OK;
  dfree(c->spill);
  c->spill = nullptr;
  c->spill_words = 0;
  HIPCHK(c, dalloc(&c->spill, words));
  c->spill_words = words;
  return CLV_OK;
}

/* traversal launch geometry of a render for the configured variant; the LDS
 * window caches the top of scene `s` */
struct TraceGeom {
  uint32_t blocks = 0;
  size_t lds_bytes = 0;
  uint32_t lds_node_base = 0, lds_nodes = 0, lds_unit_base = 0, lds_units = 0;
  uint32_t full = 0; /* whole-path launches: the scene of every job is in the window, whole */
};

/* Whole paths in one launch per pass (k_paths) wherever the LDS-cached
 * traversal is asked for and nothing has to be seen between the bounces: no
 * guided job (the network runs between tracing and shading), no per-launch
 * timing, no counting. */
bool whole_paths(const clv_ctx *c, bool any_guide, uint32_t flags) {
  return c->trace_variant == TRACE_LDS && !any_guide && !(flags & (CLV_FLAG_TIME_KERNELS | CLV_FLAG_COUNT));
}

/* a pass of k_paths keeps 12 bytes per sample, beside the traversal stacks of its
 * resident blocks (100 MB with the scene in LDS, 136 MB from memory), so an untuned
 * context runs the samples of a whole render in one (up to 1.6 GB of contributions) */
#define DEFAULT_TARGET_PATHS (1u << 22)
#define WHOLE_TARGET_PATHS (1u << 27)

/* an untuned context's wavefront passes behind the last training round grow to
 * this many paths: the late bounces of a pass launch four kernels each for a
 * few paths (274 bytes of state and lobes per path, 9.2 GB; the guided prism
 * takes 42.2 ms with 2^24 paths, 39.3 with 2^25, 38.2 with 2^26) */
#define MERGED_TARGET_PATHS (1u << 25)

clv_status paths_geometry(clv_ctx *c, const SceneRes *s, bool one_scene, const DevScene &ds, TraceGeom *g) {
  g->full = one_scene && paths_lds_bytes(true, s->n_nodes, s->prim_units) <= c->lds_block_bytes;
  if (g->full) {
    g->lds_node_base = s->base.nodes;
    g->lds_unit_base = s->base.units;
    g->lds_nodes = s->n_nodes;
    g->lds_units = s->prim_units;
  }
  g->lds_bytes = paths_lds_bytes(g->full != 0, g->lds_nodes, g->lds_units);
  g->blocks = paths_grid_blocks(g->lds_bytes, ds, g->full != 0);
  return ensure_spill(c, paths_spill_words(g->full != 0, g->blocks));
}

/* the traversal kernel a batch runs: the tuned one, or the plain one when a
 * scene of the batch has constant media (only it has the media pass) */
int trace_variant_for(const clv_ctx *c, bool media) { return media ? TRACE_SIMPLE : c->trace_variant; }

clv_status trace_geometry(clv_ctx *c, const SceneRes *s, uint32_t full_grid_paths, TraceGeom *g, int variant) {
  if (variant == TRACE_LDS) {
    size_t budget = c->lds_block_bytes > lds_trace_stack_bytes() ? c->lds_block_bytes - lds_trace_stack_bytes() : 0;
    g->lds_node_base = s->base.nodes;
    g->lds_unit_base = s->base.units;
    g->lds_nodes = (uint32_t)std::min<size_t>(s->n_nodes, budget / sizeof(Bvh4Node));
    budget -= (size_t)g->lds_nodes * sizeof(Bvh4Node);
    g->lds_units = (uint32_t)std::min<size_t>(s->prim_units, budget / 16u);
    g->lds_bytes = lds_trace_bytes(g->lds_nodes, g->lds_units);
    g->blocks = lds_trace_grid_blocks(g->lds_bytes);
    return ensure_spill(c, lds_trace_spill_words(g->blocks));
  }
  g->blocks = c->trace_blocks;
  if (full_grid_paths && c->full_grid && variant != TRACE_PERSISTENT) g->blocks = (full_grid_paths + 255u) / 256u;
  return ensure_spill(c, trace_spill_words(g->blocks));
}

void fill_trace_args(TraceArgs *ta, const TraceGeom &g) {
  ta->lds_node_base = g.lds_node_base;
  ta->lds_nodes = g.lds_nodes;
  ta->lds_unit_base = g.lds_unit_base;
  ta->lds_units = g.lds_units;
}

clv_status ensure_paths(clv_ctx *c, uint32_t n) {
  if (n <= c->cap_paths) return CLV_OK;
  free_paths(c);
  PathBuf &b = c->pb;
  HIPCHK(c, dalloc(&b.ray_o, n));
  HIPCHK(c, dalloc(&b.ray_d, n));
  HIPCHK(c, dalloc(&b.thr, n));
  HIPCHK(c, dalloc(&b.rng, n));
  HIPCHK(c, dalloc(&b.meta, n));
  HIPCHK(c, dalloc(&b.slot, n));
  HIPCHK(c, dalloc(&b.n_ray_o, n));
  HIPCHK(c, dalloc(&b.n_ray_d, n));
  HIPCHK(c, dalloc(&b.n_thr, n));
  HIPCHK(c, dalloc(&b.n_rng, n));
  HIPCHK(c, dalloc(&b.n_meta, n));
  HIPCHK(c, dalloc(&b.n_slot, n));
  HIPCHK(c, dalloc(&b.hit_t, n));
  HIPCHK(c, dalloc(&b.hit_p, n));
  HIPCHK(c, dalloc(&b.rad, n));
  HIPCHK(c, dalloc(&b.hero, n));
  for (uint32_t k = 0; k < MC_COUNT; k++) HIPCHK(c, dalloc(&c->shadeq[k], n));
  c->cap_paths = n;
  return CLV_OK;
}

clv_status ensure_res(clv_ctx *c, uint32_t n) {
  if (n <= c->cap_res) return CLV_OK;
  dfree(c->res);
  c->res = nullptr;
  c->cap_res = 0;
  HIPCHK(c, dalloc(&c->res, n));
  c->cap_res = n;
  return CLV_OK;
}

/* bytes free on the current device */
size_t free_memory() {
  size_t free = 0, total = 0;
  return hipMemGetInfo(&free, &total) == hipSuccess ? free : 0;
}

/* gives back the buffers that hold more than `keep` paths of a pass (sample contributions, path state, lobes), which
 * any render allocates again; true if there were some */
bool free_passes(clv_ctx *c, uint32_t keep) {
  GuideState &g = c->guide;
  bool any = false;
  if (c->cap_paths > keep) {
    free_paths(c);
    any = true;
  }
  if (c->cap_res > keep) {
    dfree(c->res);
    c->res = nullptr;
    c->cap_res = 0;
    any = true;
  }
  if (g.cap_lobes > keep) {
    dfree(g.lobes);
    g.lobes = nullptr;
    g.cap_lobes = 0;
    any = true;
  }
  return any;
}

/* A context keeps the buffers of its largest passes, up to 9.2 GB.  A call that finds no memory runs again once they
 * are given back. */
template <class CALL>
clv_status with_room(clv_ctx *c, CALL call) {
  clv_status st = call();
  if (st == CLV_ENOMEM && free_passes(c, DEFAULT_TARGET_PATHS)) st = call();
  return st;
}

void free_pixels(clv_ctx *c) {
  dfree(c->acc32); dfree(c->acc64); dfree(c->accsq); dfree(c->out); dfree(c->out_sq); dfree(c->ids); dfree(c->ts);
  c->acc32 = nullptr; c->acc64 = c->accsq = nullptr; c->out = c->out_sq = nullptr; c->ids = nullptr; c->ts = nullptr;
  c->cap_pixels = 0;
}

clv_status ensure_pixels(clv_ctx *c, uint32_t n) {
  if (n <= c->cap_pixels) return CLV_OK;
  free_pixels(c);
  HIPCHK(c, dalloc(&c->acc32, 3 * (size_t)n));
  HIPCHK(c, dalloc(&c->acc64, 3 * (size_t)n));
  HIPCHK(c, dalloc(&c->accsq, 3 * (size_t)n));
  HIPCHK(c, dalloc(&c->out, 3 * (size_t)n));
  HIPCHK(c, dalloc(&c->out_sq, 3 * (size_t)n));
  HIPCHK(c, dalloc(&c->ids, (size_t)n));
  HIPCHK(c, dalloc(&c->ts, (size_t)n));
  c->cap_pixels = n;
  return CLV_OK;
}

clv_status ensure_tables(clv_ctx *c, uint32_t jobs, uint32_t items) {
  if (jobs > c->cap_jobs) {
    dfree(c->jobs);
    c->jobs = nullptr;
    c->cap_jobs = 0;
    HIPCHK(c, dalloc(&c->jobs, jobs));
    c->cap_jobs = jobs;
  }
  if (items > c->cap_items) {
    dfree(c->items);
    c->items = nullptr;
    c->cap_items = 0;
    HIPCHK(c, dalloc(&c->items, items));
    c->cap_items = items;
  }
  return CLV_OK;
}

/* append `bytes` to an arena array, growing it (a device-to-device copy of
 * what it holds) when needed; src NULL only reserves the range */
clv_status arena_append(clv_ctx *c, DevArray &a, const void *src, size_t bytes) {
  const size_t need = a.used + bytes;
  if (need > a.cap) {
    size_t cap = std::max<size_t>(std::max<size_t>(need, 2 * a.cap), 1u << 16);
    char *p = nullptr;
    HIPCHK(c, hipMalloc((void **)&p, cap));
    if (a.used) {
      hipError_t e = hipMemcpyAsync(p, a.p, a.used, hipMemcpyDeviceToDevice, c->stream);
      if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
      if (e != hipSuccess) {
        (void)hipFree(p);
        return fail(c, CLV_EDEVICE, std::string("arena growth: ") + hipGetErrorString(e));
      }
    }
    dfree(a.p);
    a.p = p;
    a.cap = cap;
  }
  if (bytes && src) HIPCHK(c, hipMemcpyAsync(a.p + a.used, src, bytes, hipMemcpyHostToDevice, c->stream));
  a.used = need;
  return CLV_OK;
}

/* r = P^-1 v for a 3x3 P (Cramer's rule) */
void inv3_apply(const double P[3][3], const double v[3], double r[3]) {
  const double det = P[0][0] * (P[1][1] * P[2][2] - P[1][2] * P[2][1]) - P[0][1] * (P[1][0] * P[2][2] - P[1][2] * P[2][0]) +
                     P[0][2] * (P[1][0] * P[2][1] - P[1][1] * P[2][0]);
  for (int k = 0; k < 3; k++) {
    double Q[3][3];
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) Q[i][j] = j == k ? v[i] : P[i][j];
    r[k] = (Q[0][0] * (Q[1][1] * Q[2][2] - Q[1][2] * Q[2][1]) - Q[0][1] * (Q[1][0] * Q[2][2] - Q[1][2] * Q[2][0]) +
            Q[0][2] * (Q[1][0] * Q[2][1] - Q[1][1] * Q[2][0])) / det;
  }
}

/* Bradford adaptation XYZ(white w) -> XYZ(E): B^-1 diag((B 1) / (B w)) B */
void bradford(const double B[3][3], const double w[3], double A[3][3]) {
  double d[3], Bi[3][3];
  for (int i = 0; i < 3; i++) d[i] = (B[i][0] + B[i][1] + B[i][2]) / (B[i][0] * w[0] + B[i][1] * w[1] + B[i][2] * w[2]);
  for (int j = 0; j < 3; j++) {
    double e[3] = {0, 0, 0}, col[3];
    e[j] = 1.0;
    inv3_apply(B, e, col);
    for (int i = 0; i < 3; i++) Bi[i][j] = col[i];
  }
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) A[i][j] = Bi[i][0] * d[0] * B[0][j] + Bi[i][1] * d[1] * B[1][j] + Bi[i][2] * d[2] * B[2][j];
}

DevScene arena_view(const clv_ctx *c) {
  DevScene d;
  memset(&d, 0, sizeof(d));
  d.nodes = (const Bvh4Node *)c->arena[AR_NODES].p;
  d.prims = (const float4 *)c->arena[AR_PRIMS].p;
  d.info = (const PrimInfo *)c->arena[AR_INFO].p;
  d.xforms = (const Xform *)c->arena[AR_XFORMS].p;
  d.mats = (const DevMaterial *)c->arena[AR_MATS].p;
  d.spd = (const float *)c->arena[AR_SPD].p;
  d.lights = (const DevLight *)c->arena[AR_LIGHTS].p;
  d.lnodes = (const DevLightNode *)c->arena[AR_LNODES].p;
  d.lweights = (const float *)c->arena[AR_LWEIGHTS].p;
  d.jobs = c->jobs;
  return d;
}

clv_status check_opts(clv_ctx *c, const clv_render_opts *o) {
  if (!o) return fail(c, CLV_EINVAL, "opts is NULL");
  if (o->width == 0 || o->height == 0) return fail(c, CLV_EINVAL, "width and height must be positive");
  if ((uint64_t)o->width * o->height > (1ull << 27)) return fail(c, CLV_EINVAL, "image larger than 2^27 pixels");
  if (o->max_depth > 1000) return fail(c, CLV_EINVAL, "max_depth above 1000");
  if (o->guiding != CLV_GUIDE_OFF && o->guiding != CLV_GUIDE_ON) return fail(c, CLV_EINVAL, "unknown guiding mode");
  return CLV_OK;
}

DevJob make_job(const SceneRes *s, const clv_camera_init &cam, const clv_render_opts *o) {
  DevJob j;
  memset(&j, 0, sizeof(j));
  j.cam = make_camera(cam, (float)o->width / (float)o->height);
  j.root = s->base.nodes;
  j.light_root = s->light_root;
  j.light_base = s->base.lights;
  j.n_lights = s->n_lights;
  j.bg_spd = s->bg_spd;
  j.width = o->width;
  j.height = o->height;
  j.max_depth = o->max_depth;
  j.seed = o->seed;
  j.spp = o->samples;
  j.fp64 = o->fp64_accum ? 1u : 0u;
  j.guiding = o->guiding;
  for (int a = 0; a < 3; a++) {
    j.lo[a] = s->lo[a];
    j.hi[a] = s->hi[a];
  }
  j.media_off = s->media_off;
  j.n_media = s->n_media;
  return j;
}

/* ------------------------------------------------------------ guiding --- */
clv_status guide_ensure_net(clv_ctx *c) {
  GuideState &g = c->guide;
  /* each by itself: a call may have run out of memory between them */
  if (!g.P) HIPCHK(c, dalloc(&g.P, GD_NPARAM));
  if (!g.M) HIPCHK(c, dalloc(&g.M, GD_NPARAM));
  if (!g.V) HIPCHK(c, dalloc(&g.V, GD_NPARAM));
  if (!g.Wh) HIPCHK(c, dalloc(&g.Wh, GD_NHALF));
  if (!g.totals) HIPCHK(c, dalloc(&g.totals, 4));
  if (!g.host_totals) {
    void *hp = nullptr;
    if (hipHostMalloc(&hp, 4 * sizeof(uint32_t), hipHostMallocDefault) == hipSuccess) g.host_totals = (uint32_t *)hp;
  }
  return CLV_OK;
}

clv_status guide_ensure_partial(clv_ctx *c, uint32_t groups) {
  GuideState &g = c->guide;
  if (groups <= g.partial_groups) return CLV_OK;
  dfree(g.partial);
  g.partial = nullptr;
  g.partial_groups = 0;
  HIPCHK(c, dalloc(&g.partial, (size_t)groups * GD_NPARAM));
  g.partial_groups = groups;
  return CLV_OK;
}

void guide_free(GuideState &g) {
  if (g.host_totals) (void)hipHostFree(g.host_totals);
  g.host_totals = nullptr;
  dfree(g.cells); dfree(g.cell_tot); dfree(g.gate); dfree(g.fresh);
  dfree(g.P); dfree(g.M); dfree(g.V); dfree(g.Wh); dfree(g.partial); dfree(g.totals);
  dfree(g.lobes); dfree(g.rec); dfree(g.recL); dfree(g.gcnt); dfree(g.list); dfree(g.bcount); dfree(g.bweight);
}

/* lobes of `paths` path slots of any pass */
clv_status guide_ensure_lobes(clv_ctx *c, uint32_t paths) {
  GuideState &g = c->guide;
  if (paths <= g.cap_lobes) return CLV_OK;
  dfree(g.lobes);
  g.lobes = nullptr;
  g.cap_lobes = 0;
  HIPCHK(c, dalloc(&g.lobes, (size_t)paths * GD_LWORDS));
  g.cap_lobes = paths;
  return CLV_OK;
}

/* record space of a training pass: GD_SLOTS per path slot, then the
 * light-traced records of a round (g.photons) */
clv_status guide_ensure_paths(clv_ctx *c, uint32_t paths) {
  GuideState &g = c->guide;
  if (paths <= g.cap_paths && g.photons <= g.cap_photons) return CLV_OK;
  dfree(g.rec); dfree(g.recL); dfree(g.gcnt); dfree(g.list); dfree(g.bcount); dfree(g.bweight);
  g.rec = nullptr; g.recL = nullptr; g.gcnt = nullptr; g.list = nullptr; g.bcount = nullptr;
  g.bweight = nullptr;
  paths = std::max(paths, g.cap_paths);
  g.cap_paths = 0;
  g.cap_photons = 0;
  const size_t slots = (size_t)paths * GD_SLOTS + g.photons;
  HIPCHK(c, dalloc(&g.rec, slots));
  HIPCHK(c, dalloc(&g.recL, slots));
  HIPCHK(c, dalloc(&g.gcnt, paths));
  HIPCHK(c, dalloc(&g.list, slots));
  /* per compaction block of 4096 records: two counts and two weight sums */
  HIPCHK(c, dalloc(&g.bcount, slots / 256 + 8));
  HIPCHK(c, dalloc(&g.bweight, slots / 256 + 8));
  HIPCHK(c, hipMemsetAsync(g.rec, 0, slots * sizeof(GuideRec), c->stream));
  HIPCHK(c, hipMemsetAsync(g.recL, 0, slots * sizeof(float), c->stream));
  g.cap_paths = paths;
  g.cap_photons = g.photons;
  return CLV_OK;
}

/* fresh parameters: He-normal hidden layers, a small output layer (broad,
 * nearly uniform lobes), zero biases, zero Adam moments */
clv_status guide_reset(clv_ctx *c, uint64_t seed) {
  CHK(with_room(c, [&] { return guide_ensure_net(c); }));
  GuideState &g = c->guide;
  std::vector<float> P(GD_NPARAM, 0.0f);
  uint64_t st = seed * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
  auto next = [&st]() {
    st += 0x9E3779B97F4A7C15ull;
    uint64_t z = st;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return ((double)(z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
  };
  auto normal = [&]() { return sqrt(-2.0 * log(next())) * cos(6.283185307179586 * next()); };
  const float he = sqrtf(2.0f / 64.0f);
  for (int k = 0; k < GD_HID * GD_IN; k++) P[GD_W1 + k] = (float)normal() * he;
  for (int k = 0; k < GD_HID * GD_HID; k++) P[GD_W2 + k] = (float)normal() * he;
  for (int k = 0; k < GD_HID * GD_HID; k++) P[GD_W3 + k] = (float)normal() * he;
  for (int k = 0; k < GD_OUT * GD_HID; k++) P[GD_W4 + k] = (float)normal() * 0.01f;
  HIPCHK(c, hipMemcpyAsync(g.P, P.data(), GD_NPARAM * sizeof(float), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemsetAsync(g.M, 0, GD_NPARAM * sizeof(float), c->stream));
  HIPCHK(c, hipMemsetAsync(g.V, 0, GD_NPARAM * sizeof(float), c->stream));
  HIPCHK(c, hipMemsetAsync(g.Wh, 0, GD_NHALF * sizeof(_Float16), c->stream));
  HIPCHK(c, hipMemsetAsync(g.totals, 0, 4 * sizeof(uint32_t), c->stream)); /* [3]: no Adam steps yet */
  launch_guide_halves(c->stream, g.P, g.Wh);
  HIPCHK(c, hipStreamSynchronize(c->stream));
  g.init = true;
  g.trained = false;
  return CLV_OK;
}

/* copies of the gate's fresh counts: the contention they relieve is a job's, so one job gets the most of them.
 * A buffer of gate_fresh_jobs(n) jobs holds the copies of a batch of n jobs and of every smaller one */
#define GATE_COPIES 16u
uint32_t gate_copies(uint32_t n_jobs) { return std::max<uint32_t>(1u, GATE_COPIES / n_jobs); }
size_t gate_fresh_jobs(uint32_t n_jobs) { return std::max<uint32_t>(GATE_COPIES, n_jobs); }

/* zero the gate's counts (a fresh network) */
clv_status guide_clear_gate(clv_ctx *c) {
  GuideState &g = c->guide;
  HIPCHK(c, hipMemsetAsync(g.cells, 0, (size_t)g.gate_jobs * GD_CELLS * sizeof(uint32_t), c->stream));
  HIPCHK(c, hipMemsetAsync(g.cell_tot, 0, (size_t)g.gate_jobs * sizeof(uint32_t), c->stream));
  HIPCHK(c, hipMemsetAsync(g.fresh, 0, gate_fresh_jobs(g.gate_jobs) * GD_CELLS * sizeof(uint32_t), c->stream));
  g.gate_valid = false;
  return CLV_OK;
}

/* gate buffers for n jobs; new ones hold no counts */
clv_status guide_ensure_gate(clv_ctx *c, uint32_t n) {
  GuideState &g = c->guide;
  if (n <= g.gate_jobs) return CLV_OK;
  dfree(g.cells); dfree(g.cell_tot); dfree(g.gate); dfree(g.fresh);
  g.cells = g.cell_tot = g.fresh = nullptr;
  g.gate = nullptr;
  g.gate_jobs = 0;
  HIPCHK(c, dalloc(&g.cells, (size_t)n * GD_CELLS));
  HIPCHK(c, dalloc(&g.cell_tot, n));
  HIPCHK(c, dalloc(&g.fresh, gate_fresh_jobs(n) * GD_CELLS));
  HIPCHK(c, dalloc(&g.gate, (size_t)n * GD_CELLS));
  g.gate_jobs = n;
  return guide_clear_gate(c);
}

/* light-traced records of a round (k_guide_photons) behind the record slots
 * of `paths` path slots */
void guide_photons(clv_ctx *c, const DevScene &ds, uint32_t n_jobs, uint32_t paths, uint32_t stamp, uint32_t round,
                   uint64_t seed) {
  GuideState &g = c->guide;
  const size_t base = (size_t)paths * GD_SLOTS;
  launch_guide_photons(c->stream, ds, n_jobs, g.rec + base, g.recL + base, g.photons, stamp, round, seed, c->spill,
                       std::min(c->photon_blocks, c->trace_blocks), g.fresh, gate_copies(n_jobs));
}

/* one training round on the records of pass `stamp` (n path slots), and
 * `extra` records behind them (the round's light-traced ones) */
void guide_train_round(clv_ctx *c, uint32_t paths, uint32_t stamp, float *grad_out, float wclip, uint32_t extra = 0) {
  GuideState &g = c->guide;
  const uint32_t cap = grad_out ? paths * GD_SLOTS : g.records;
  launch_guide_collect(c->stream, g.rec, g.recL, paths * GD_SLOTS + extra, g.bcount, g.bweight, g.totals, g.list, cap,
                       (unsigned long long *)c->stats + 4);
  const uint32_t step = grad_out ? cap : g.step;
  const uint32_t epochs = grad_out ? 1u : std::max<uint32_t>(1u, g.epochs);
  /* steps past the round's valid records are empty (the kernels skip them):
   * the count is read back so they are not launched at all -- the same
   * parameters either way */
  uint32_t used = cap;
  if (!grad_out && g.host_totals &&
      hipMemcpyAsync(g.host_totals, g.totals, sizeof(uint32_t), hipMemcpyDeviceToHost, c->stream) == hipSuccess &&
      hipStreamSynchronize(c->stream) == hipSuccess)
    used = std::min(cap, g.host_totals[0]);
  for (uint32_t e = 0; e < epochs; e++)
    for (uint32_t b = 0; b < used; b += step) {
      launch_guide_step(c->stream, g.rec, g.recL, g.list, g.totals, cap, b, std::min(step, cap - b), wclip, g.P, g.M,
                        g.V, g.Wh, g.partial, g.lr, grad_out);
    }
}

/* the batch render behind clv_render and clv_render_batch */
clv_status render_jobs(clv_ctx *c, const clv_job *jobs, uint32_t n) {
  if (n == 0 || !jobs) return fail(c, CLV_EINVAL, "no jobs");
  if (n > MAX_JOBS) return fail(c, CLV_EINVAL, "more than 8192 jobs in one batch");
  std::vector<DevJob> dj(n);
  std::vector<uint32_t> soff(n);
  std::vector<const SceneRes *> sres(n);
  uint64_t pixels = 0, samples = 0;
  uint32_t flags = 0;
  bool any_xform = false, any_ext = false, any_media = false;
  for (uint32_t k = 0; k < n; k++) {
    const clv_job &jb = jobs[k];
    CHK(check_opts(c, &jb.opts));
    if (!jb.xyz_out) return fail(c, CLV_EINVAL, "xyz_out is NULL");
    if (jb.opts.samples == 0) return fail(c, CLV_EINVAL, "samples must be positive");
    auto it = c->scenes.find(jb.scene_id);
    if (it == c->scenes.end()) return fail(c, CLV_EINVAL, "unknown scene id");
    sres[k] = it->second;
    dj[k] = make_job(it->second, jb.use_camera ? jb.camera : it->second->camera, &jb.opts);
    dj[k].pixel_base = (uint32_t)pixels;
    soff[k] = jb.opts.sample_offset;
    pixels += (uint64_t)jb.opts.width * jb.opts.height;
    samples += (uint64_t)jb.opts.width * jb.opts.height * jb.opts.samples;
    flags |= jb.opts.flags;
    any_xform = any_xform || it->second->has_xforms;
    any_ext = any_ext || it->second->has_ext;
    any_media = any_media || it->second->n_media > 0;
  }
  if (pixels > (1ull << 28)) return fail(c, CLV_EINVAL, "batch larger than 2^28 pixels");
  bool any_guide = false;
  uint64_t guide_seed = 0;
  for (uint32_t k = 0; k < n; k++)
    if (jobs[k].opts.guiding == CLV_GUIDE_ON && !any_guide) {
      any_guide = true;
      guide_seed = jobs[k].opts.seed;
    }
  if (any_guide && c->guide.warmup)
    for (uint32_t k = 0; k < n; k++)
      if ((uint64_t)jobs[k].opts.sample_offset + jobs[k].opts.samples > WARMUP_SAMPLE_BASE)
        return fail(c, CLV_EINVAL, "with guide_warmup, image sample indices stay below 2^31");
  HIPCHK(c, hipSetDevice(c->device));
  const bool frozen = (flags & CLV_FLAG_GUIDE_FROZEN) != 0;
  const bool whole = whole_paths(c, any_guide, flags);
  PassPlan pl;
  /* a frozen network is not trained: no training slices, every pass full size */
  const bool untuned = c->target_paths == DEFAULT_TARGET_PATHS;
  GuideState &gs = c->guide;
  /* the LDS window caches the scene with the most samples */
  uint32_t big = 0;
  for (uint32_t k = 1; k < n; k++)
    if ((uint64_t)dj[k].width * dj[k].height * dj[k].spp > (uint64_t)dj[big].width * dj[big].height * dj[big].spp) big = k;
  TraceGeom geom;
  DevScene ds = DevScene();
  int variant = trace_variant_for(c, any_media);
  bool one_scene = true;
  for (uint32_t k = 1; k < n; k++) one_scene = one_scene && sres[k] == sres[0];
  /* Guided bounces, unless they are measured: the window of LDS pays where it holds at least half of the only scene
   * (guided renders of 1M / 82k / 12k triangles, 1024x640, 32 spp: 43.6 / 30.2 / 21.0 ms with it, 34.8 / 25.1 / 18.9
   * from memory; 1,280 triangles, of which the window holds less than half: 14.0 / 14.4, and 3.9 / 3.6 at 320x200,
   * 16 spp) */
  if (!whole && variant == TRACE_LDS && !(flags & (CLV_FLAG_TIME_KERNELS | CLV_FLAG_COUNT)) &&
      !(one_scene && lds_trace_bytes(sres[big]->n_nodes / 2u, sres[big]->prim_units / 2u) <= c->lds_block_bytes))
    variant = TRACE_MAJORITY;
  /* the tail launch (k_tail): the resident grid of the plain traversal, never with per-launch timing or
   * counting (those measure the wavefront traversal) */
  const uint32_t tail_depth = (flags & (CLV_FLAG_TIME_KERNELS | CLV_FLAG_COUNT)) ? 0u : c->tail_depth;
  /* light-traced training records: a round before the first pass (so the
   * first samples are already guided) and one with every training pass */
  const bool photon_rounds = any_guide && !frozen && gs.photons > 0 && gs.rounds > 0;
  auto reserve = [&]() -> clv_status {
    CHK(whole ? ensure_res(c, pl.max_paths) : ensure_paths(c, pl.max_paths));
    CHK(ensure_pixels(c, (uint32_t)pixels));
    CHK(ensure_tables(c, n, (uint32_t)pl.items.size()));
    ds = arena_view(c);
    ds.has_xforms = any_xform ? 1u : 0u;
    ds.has_ext = any_ext ? 1u : 0u;
    ds.has_media = any_media ? 1u : 0u;
    geom = TraceGeom();
    if (whole) CHK(paths_geometry(c, sres[big], one_scene, ds, &geom));
    else CHK(trace_geometry(c, sres[big], pl.max_paths, &geom, variant));
    if (tail_depth || photon_rounds) CHK(ensure_spill(c, std::max(c->spill_words, trace_spill_words(c->trace_blocks))));
    if (!any_guide) return CLV_OK;
    uint32_t recorded = 0; /* the largest pass that writes training records */
    for (size_t p = 0; p < pl.paths.size(); p++)
      if (!frozen && pl.train[p]) recorded = std::max(recorded, pl.paths[p]);
    CHK(guide_ensure_lobes(c, pl.max_paths));
    CHK(guide_ensure_paths(c, recorded));
    CHK(guide_ensure_partial(c, gs.step / 64u));
    CHK(guide_ensure_net(c));
    return gs.photons ? guide_ensure_gate(c, n) : CLV_OK;
  };
  auto &no_room = c->no_room[whole ? 1 : 0];
  for (bool large = untuned, again = false;;) {
    pl = PassPlan();
    plan_passes(dj, soff, whole && large ? WHOLE_TARGET_PATHS : c->target_paths, std::max<uint32_t>(1, gs.train_spp),
                frozen ? 0u : gs.rounds, gs.warmup != 0, &pl);
    if (!whole && large) merge_passes(&pl, MERGED_TARGET_PATHS);
    if (large && no_room.paths && pl.max_paths >= no_room.paths) {
      /* a try costs what 25 allocations and frees do (60 to 110 ms for guided passes): not again before more memory
       * is free than there was */
      if (free_memory() <= no_room.free) {
        large = false;
        continue;
      }
      no_room.paths = 0;
    }
    const clv_status st = reserve();
    if (st == CLV_OK) break;
    if (st != CLV_ENOMEM || again) return st;
    /* no memory: once more without the buffers of earlier large passes, and, where these passes are large ones, at
     * the default size, which needs 50 MB beside the stacks (whole paths) to 1.2 GB (guided) */
    if (!free_passes(c, large ? 0u : DEFAULT_TARGET_PATHS) && !large) return st;
    if (large && pl.max_paths > DEFAULT_TARGET_PATHS) {
      no_room.paths = pl.max_paths;
      no_room.free = free_memory();
    }
    large = false;
    again = true;
  }
  std::vector<uint32_t> job_left(n);
  for (uint32_t k = 0; k < n; k++) job_left[k] = dj[k].spp;
  for (DevItem &it : pl.items) {
    it.order = c->tile_order;
    if (it.flags & ITEM_WARMUP) continue;
    if (job_left[it.job] == dj[it.job].spp) it.flags |= ITEM_FIRST;
    job_left[it.job] -= it.samples;
    if (job_left[it.job] == 0) it.flags |= ITEM_LAST;
  }
  const uint32_t passes = (uint32_t)pl.paths.size();
  if (any_guide) {
    const bool fresh = !(flags & CLV_FLAG_GUIDE_KEEP) || !gs.init;
    if (fresh) CHK(guide_reset(c, guide_seed));
    if (fresh && gs.photons) CHK(guide_clear_gate(c));
  }
  StreamDrain drain{c->stream}; /* dj and pl.items outlive every copy from them */
  HIPCHK(c, hipMemcpyAsync(c->jobs, dj.data(), n * sizeof(DevJob), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->items, pl.items.data(), pl.items.size() * sizeof(DevItem), hipMemcpyHostToDevice,
                           c->stream));
  const bool timing = (flags & CLV_FLAG_TIME_KERNELS) != 0;
  const bool counting = (flags & CLV_FLAG_COUNT) != 0;
  uint32_t extends = 0;
  for (uint32_t p = 0; p < passes; p++) extends += whole ? 1u : tail_depth ? std::min(pl.depth[p] + 1u, tail_depth + 1u) : pl.depth[p] + 1u;
  size_t need_events = 2 + (timing ? 2 * (size_t)extends : 0);
  while (c->events.size() < need_events) {
    hipEvent_t e;
    HIPCHK(c, hipEventCreate(&e));
    c->events.push_back(e);
  }
  ResolveParams rp;
  memset(&rp, 0, sizeof(rp));
  rp.jobs = c->jobs;
  rp.n_jobs = n;
  rp.pixels = (uint32_t)pixels;
  rp.acc32 = c->acc32;
  rp.acc64 = c->acc64;
  rp.acc_sq = c->accsq;
  ShadeQueues sq;
  for (uint32_t q = 0; q < MC_COUNT; q++) sq.q[q] = c->shadeq[q];
  sq.counts = c->counts + CNT_SHADE;
  size_t ev = 2;
  PathBuf pb = c->pb;
  GuideArgs ga;
  memset(&ga, 0, sizeof(ga));
  if (any_guide) {
    ga.lobes = gs.lobes;
    ga.rec = gs.rec;
    ga.Wh = gs.Wh;
    ga.P = gs.P;
    ga.on = 1u;
    ga.indirect = gs.credit;
    ga.stats = (unsigned long long *)c->stats;
  }
  /* timing events of the guide's launches: [start, end) pairs */
  std::vector<std::pair<hipEvent_t, hipEvent_t>> gev_infer, gev_train;
  auto guide_event = [&](std::vector<std::pair<hipEvent_t, hipEvent_t>> &v) -> hipEvent_t {
    hipEvent_t a = nullptr, b = nullptr;
    if (hipEventCreate(&a) != hipSuccess) return nullptr;
    if (hipEventCreate(&b) != hipSuccess) { (void)hipEventDestroy(a); return nullptr; }
    v.push_back({a, b});
    (void)hipEventRecord(a, c->stream);
    return b;
  };
  uint32_t rounds_run = 0;
  bool any_sq = false;
  for (uint32_t k = 0; k < n; k++) any_sq = any_sq || jobs[k].xyz_sq_out;
  /* every launch of the render; without guided jobs no host synchronisation
   * inside, so the sequence can be captured as a graph */
  auto enqueue = [&]() -> clv_status {
  if (whole) {
    for (uint32_t p = 0; p < passes; p++) {
      GenParams gp;
      memset(&gp, 0, sizeof(gp));
      gp.items = c->items + pl.first[p];
      gp.n_items = pl.first[p + 1] - pl.first[p];
      gp.paths = pl.paths[p];
      PathsArgs pa;
      memset(&pa, 0, sizeof(pa));
      pa.next = c->counts + CNT_FETCH;
      pa.spill = c->spill;
      pa.stats = (unsigned long long *)c->stats;
      pa.res = c->res;
      pa.cie = c->cie;
      pa.lds_node_base = geom.lds_node_base;
      pa.lds_nodes = geom.lds_nodes;
      pa.lds_unit_base = geom.lds_unit_base;
      pa.lds_units = geom.lds_units;
      pa.full = geom.full;
      /* a pass smaller than the grid is spread over all its blocks */
      const uint32_t block = paths_block(geom.full != 0);
      const uint32_t blocks = std::min(geom.blocks, (gp.paths + 63u) / 64u);
      pa.first = (uint32_t)std::min<uint64_t>(block, ((uint64_t)gp.paths + 64ull * blocks - 1u) / (64ull * blocks) * 64ull);
      pa.chunk = block;
      launch_paths(c->stream, ds, gp, pa, blocks, geom.lds_bytes, p == 0);
      rp.items = gp.items;
      rp.n_items = gp.n_items;
      rp.threads = pl.res[p];
      launch_resolve_xyz(c->stream, rp, c->res, c->out, any_sq ? c->out_sq : nullptr);
    }
    return CLV_OK;
  }
  launch_zero_u64(c->stream, c->stats, 8);
  launch_zero_accum(c->stream, rp);
  for (uint32_t pr = 0; photon_rounds && pr < gs.pre_rounds; pr++) {
    hipEvent_t end = timing ? guide_event(gev_train) : nullptr;
    const uint32_t st = ++gs.stamp;
    guide_photons(c, ds, n, 0, st, rounds_run, guide_seed);
    guide_train_round(c, 0, st, nullptr, gs.wclip, gs.photons);
    launch_guide_gate(c->stream, gs.fresh, gate_copies(n), gs.cells, gs.cell_tot, gs.gate, n, gs.gate_density);
    if (end) (void)hipEventRecord(end, c->stream);
    gs.trained = true;
    gs.gate_valid = true;
    rounds_run++;
  }
  for (uint32_t p = 0; p < passes; p++) {
    GenParams gp;
    memset(&gp, 0, sizeof(gp));
    gp.items = c->items + pl.first[p];
    gp.n_items = pl.first[p + 1] - pl.first[p];
    gp.paths = pl.paths[p];
    const bool recording = any_guide && !frozen && pl.train[p];
    pb.gcnt = recording ? gs.gcnt : nullptr;
    pb.recL = recording ? gs.recL : nullptr;
    launch_set_count(c->stream, c->counts, CNT_QA, gp.paths);
    launch_generate(c->stream, ds, pb, gp);
    if (any_guide) {
      /* plain sampling until the network has had a training round (or, frozen, always the network) */
      ga.alpha = (gs.trained || frozen) ? gs.alpha : 0.0f;
      ga.record = recording ? 1u : 0u;
      ga.gate = gs.photons && gs.gate_density > 0.0f && gs.gate_valid && gs.gate_jobs >= n ? gs.gate : nullptr;
      ga.stamp = ++gs.stamp;
    }
    for (uint32_t depth = 0; depth <= pl.depth[p]; depth++) {
      const PathBuf bv = bounce_view(pb, depth);
      uint32_t in = depth & 1u, out = in ^ 1u;
      uint32_t in_slot = in ? CNT_QB : CNT_QA, out_slot = out ? CNT_QB : CNT_QA;
      launch_reset_counts(c->stream, c->counts, in_slot, out_slot, c->stats);
      if (tail_depth && depth == tail_depth) {
        TraceArgs ta;
        memset(&ta, 0, sizeof(ta));
        ta.counts = c->counts;
        ta.in_slot = in_slot;
        ta.spill = c->spill;
        ta.stats = (unsigned long long *)c->stats;
        launch_tail(c->stream, ds, bv, ta, c->trace_blocks, ga);
        break;
      }
      if (timing) HIPCHK(c, hipEventRecord(c->events[ev], c->stream));
      TraceArgs ta;
      memset(&ta, 0, sizeof(ta));
      ta.counts = c->counts;
      ta.in_slot = in_slot;
      ta.sq = sq;
      ta.spill = c->spill;
      ta.stats = (unsigned long long *)c->stats;
      fill_trace_args(&ta, geom);
      if (variant == TRACE_LDS)
        launch_trace_lds(c->stream, ds, bv, ta, geom.blocks, geom.lds_bytes, counting, 0);
      else
        launch_extend(c->stream, ds, bv, ta, geom.blocks, counting, variant);
      if (timing) HIPCHK(c, hipEventRecord(c->events[ev + 1], c->stream));
      ev += timing ? 2 : 0;
      if (any_guide && ga.alpha > 0.0f) {
        hipEvent_t end = timing ? guide_event(gev_infer) : nullptr;
        launch_guide_infer(c->stream, ds, bv, ga, sq.q[MC_LAMBERTIAN], sq.counts + MC_LAMBERTIAN, gp.paths,
                           c->infer_blocks);
        if (end) (void)hipEventRecord(end, c->stream);
      }
      launch_shade(c->stream, ds, bv, sq, c->counts, out_slot, gp.paths, c->grid_cap, c->shade_blocks, ga);
    }
    rp.items = gp.items;
    rp.n_items = gp.n_items;
    rp.threads = pl.res[p];
    launch_resolve(c->stream, pb, rp, c->cie);
    if (any_guide && ga.record) {
      hipEvent_t end = timing ? guide_event(gev_train) : nullptr;
      if (photon_rounds) guide_photons(c, ds, n, gp.paths, ga.stamp, rounds_run, guide_seed);
      guide_train_round(c, gp.paths, ga.stamp, nullptr, gs.wclip, photon_rounds ? gs.photons : 0u);
      if (photon_rounds) {
        launch_guide_gate(c->stream, gs.fresh, gate_copies(n), gs.cells, gs.cell_tot, gs.gate, n, gs.gate_density);
        gs.gate_valid = true;
      }
      if (end) (void)hipEventRecord(end, c->stream);
      gs.trained = true;
      rounds_run++;
    }
  }
  launch_finalize(c->stream, rp, c->out, any_sq ? c->out_sq : nullptr);
  return CLV_OK;
  };
  /* not guided renders: a captured training round runs all the steps its record buffer could fill, most of
   * them empty (a 64-spp prism 27 ms of 72), where an eager one reads the round's count back first */
  const bool use_graph = c->use_graph && !timing && !any_guide;
  std::string sig;
  if (use_graph) {
    /* everything a launch argument of an unguided render depends on */
    auto add = [&sig](const void *p, size_t b) { sig.append((const char *)p, b); };
    add(dj.data(), dj.size() * sizeof(DevJob));
    add(pl.items.data(), pl.items.size() * sizeof(DevItem));
    add(pl.first.data(), pl.first.size() * 4);
    add(pl.paths.data(), pl.paths.size() * 4);
    add(pl.res.data(), pl.res.size() * 4);
    add(pl.depth.data(), pl.depth.size() * 4);
    const uint32_t sc[8] = {(uint32_t)whole, flags, any_sq, (uint32_t)variant, c->grid_cap, ds.has_xforms, ds.has_ext, tail_depth};
    add(sc, sizeof(sc));
    add(&geom, sizeof(geom));
    add(&pb, sizeof(pb));
    const void *ptrs[] = {c->shadeq[0], c->shadeq[1], c->shadeq[2], c->shadeq[3], c->shadeq[4], c->acc32, c->acc64,
                          c->accsq, c->out, c->out_sq, c->counts, c->stats, c->spill, c->cie, c->res, c->jobs, c->items};
    add(ptrs, sizeof(ptrs));
    for (auto &a : c->arena) add(&a.p, sizeof(a.p));
  }
  HIPCHK(c, hipEventRecord(c->events[0], c->stream));
  /* a render is captured the second time its signature comes in a row, and
   * replayed from then on; one-off renders stay eager */
  const bool repeat = use_graph && !sig.empty() && (sig == c->last_sig || sig == c->gsig);
  if (use_graph) c->last_sig = sig;
  if (repeat && c->gexec && c->gsig == sig) {
    HIPCHK(c, hipGraphLaunch(c->gexec, c->stream));
  } else {
    bool capturing = false;
    if (repeat) {
      if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
      c->gexec = nullptr;
      c->gsig.clear();
      capturing = hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal) == hipSuccess;
    }
    clv_status st = enqueue();
    if (capturing) {
      hipGraph_t g = nullptr;
      hipError_t e = hipStreamEndCapture(c->stream, &g);
      if (st == CLV_OK && e == hipSuccess) e = hipGraphInstantiate(&c->gexec, g, nullptr, nullptr, 0);
      if (g) (void)hipGraphDestroy(g);
      if (st != CLV_OK) return st;
      if (e != hipSuccess) {
        c->gexec = nullptr;
        return fail(c, CLV_EDEVICE, std::string("graph capture: ") + hipGetErrorString(e));
      }
      c->gsig = sig;
      HIPCHK(c, hipGraphLaunch(c->gexec, c->stream));
    } else if (st != CLV_OK) {
      return st;
    }
  }
  HIPCHK(c, hipEventRecord(c->events[1], c->stream));
  HIPCHK(c, hipGetLastError());
  const size_t img_bytes = sizeof(float) * 3 * (size_t)pixels;
  std::vector<CopyArray> arrays{{c->out, img_bytes}};
  std::vector<CopySeg> segs;
  for (uint32_t k = 0; k < n; k++) {
    const size_t off = sizeof(float) * 3 * (size_t)dj[k].pixel_base, cnt = sizeof(float) * 3 * (size_t)dj[k].width * dj[k].height;
    segs.push_back({0, off, cnt, jobs[k].xyz_out});
    if (jobs[k].xyz_sq_out) {
      if (arrays.size() == 1) arrays.push_back({c->out_sq, img_bytes});
      segs.push_back({1, off, cnt, jobs[k].xyz_sq_out});
    }
  }
  uint64_t stats[8];
  HIPCHK(c, c->copy.run(c->stream, arrays, segs, c->stats, stats));
  float ms = 0.0f;
  HIPCHK(c, hipEventElapsedTime(&ms, c->events[0], c->events[1]));
  clv_counters &cn = c->counters;
  cn.guide_queries = any_guide ? stats[3] : 0;
  cn.guide_rounds = rounds_run;
  cn.guide_records = any_guide ? stats[4] : 0;
  cn.guide_infer_ms = cn.guide_train_ms = 0.0;
  for (auto *v : {&gev_infer, &gev_train}) {
    double tot = 0.0;
    for (auto &e : *v) {
      float m = 0.0f;
      if (hipEventElapsedTime(&m, e.first, e.second) == hipSuccess) tot += m;
      (void)hipEventDestroy(e.first);
      (void)hipEventDestroy(e.second);
    }
    (v == &gev_infer ? cn.guide_infer_ms : cn.guide_train_ms) = tot;
  }
  cn.samples = samples;
  cn.rays = stats[2];
  cn.node_visits = counting ? stats[0] : 0;
  cn.prim_tests = counting ? stats[1] : 0;
  cn.render_ms = ms;
  cn.extend_ms = 0.0;
  if (timing) {
    for (size_t e = 2; e < ev; e += 2) {
      float m = 0.0f;
      HIPCHK(c, hipEventElapsedTime(&m, c->events[e], c->events[e + 1]));
      cn.extend_ms += m;
    }
  }
  const SceneRes *s = sres[big];
  cn.extend_launches = extends;
  cn.passes = passes;
  cn.bvh_nodes = s->n_nodes;
  cn.bvh_width = 4;
  cn.node_bytes = sizeof(Bvh4Node);
  cn.prim_bytes = s->prim_bytes;
  cn.n_prims = s->n_prims;
  cn.bvh_depth = s->depth;
  cn.build_ms = s->build_ms;
  return CLV_OK;
}

}  // namespace

extern "C" {

uint32_t clv_abi_version(void) { return CLV_ABI_VERSION; }

float clv_spectral_power(const float xyz[3], uint32_t lambda) {
  if (!xyz) return 0.0f;
  return clv::spectral_power(xyz, (int)lambda);
}

clv_status clv_wavelength_into_xyz(uint32_t lambda, float xyz_out[3]) {
  if (!xyz_out || lambda < CLV_LAMBDA_MIN || lambda >= CLV_LAMBDA_MIN + CLV_SPECTRUM) return CLV_EINVAL;
  float table[CLV_SPECTRUM * 4];
  cie_xyz_table(table);
  for (int k = 0; k < 3; k++) xyz_out[k] = table[4 * (lambda - CLV_LAMBDA_MIN) + k];
  return CLV_OK;
}

clv_status clv_create(int hip_device, clv_ctx **out) {
  if (!out) return CLV_EINVAL;
  *out = nullptr;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return CLV_EDEVICE;
  if (hip_device < 0 || hip_device >= n) return CLV_EINVAL;
  clv_ctx *c = new (std::nothrow) clv_ctx();
  if (!c) return CLV_ENOMEM;
  memset(&c->pb, 0, sizeof(c->pb));
  memset(&c->counters, 0, sizeof(c->counters));
  c->device = hip_device;
  if (hipSetDevice(hip_device) != hipSuccess || hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return CLV_EDEVICE;
  }
  c->trace_blocks = trace_grid_blocks();
  c->infer_blocks = guide_infer_grid_blocks();
  c->photon_blocks = guide_photon_grid_blocks();
  shade_grid_blocks(c->shade_blocks);
  /* the device address of the allocation-free probe's scratch array on this
   * device (the device is current); left NULL if the runtime has none */
  if (na_scratch_address(&c->na_scratch) != 0) c->na_scratch = nullptr;
  if (const char *e = getenv("CLV_TRACE_BLOCKS")) c->trace_blocks = (uint32_t)strtoul(e, nullptr, 10);
  if (const char *e = getenv("CLV_GUIDE_STEP")) c->guide.step = std::max<uint32_t>(64u, (uint32_t)strtoul(e, nullptr, 10) & ~63u);
  if (const char *e = getenv("CLV_TILE_ORDER")) c->tile_order = strcmp(e, "0") == 0 ? 0u : 1u;
  if (const char *e = getenv("CLV_GUIDE_EPOCHS")) c->guide.epochs = std::max<uint32_t>(1u, (uint32_t)strtoul(e, nullptr, 10));
  if (const char *e = getenv("CLV_TRACE_KERNEL"))
    c->trace_variant = strcmp(e, "persistent") == 0 ? TRACE_PERSISTENT
                       : strcmp(e, "ww") == 0       ? TRACE_WW
                       : strcmp(e, "simple") == 0   ? TRACE_SIMPLE
                                                    : TRACE_LDS;
  if (const char *e = getenv("CLV_TRACE_GRID")) c->full_grid = strcmp(e, "full") == 0;
  if (c->trace_blocks < 1) c->trace_blocks = 1;
  if (const char *e = getenv("CLV_LDS_BYTES")) c->lds_block_bytes = (size_t)strtoul(e, nullptr, 10);
  if (dalloc(&c->counts, CNT_TOTAL) != hipSuccess || dalloc(&c->stats, 8) != hipSuccess ||
      dalloc(&c->cie, CLV_SPECTRUM) != hipSuccess) {
    clv_destroy(c);
    return CLV_ENOMEM;
  }
  float table[CLV_SPECTRUM * 4];
  cie_xyz_table(table);
  if (hipMemcpy(c->cie, table, sizeof(table), hipMemcpyHostToDevice) != hipSuccess) {
    clv_destroy(c);
    return CLV_EDEVICE;
  }
  if (const char *e = getenv("CLV_TARGET_PATHS")) c->target_paths = (uint32_t)strtoul(e, nullptr, 10);
  if (const char *e = getenv("CLV_GRID_CAP")) c->grid_cap = (uint32_t)strtoul(e, nullptr, 10);
  if (const char *e = getenv("CLV_GRAPH")) c->use_graph = strtoul(e, nullptr, 10) != 0;
  if (const char *e = getenv("CLV_TAIL_DEPTH")) c->tail_depth = (uint32_t)strtoul(e, nullptr, 10);
  if (c->target_paths < 65536) c->target_paths = 65536;
  if (c->grid_cap < 1) c->grid_cap = 1;
  *out = c;
  return CLV_OK;
}

void clv_destroy(clv_ctx *c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto &kv : c->scenes) delete kv.second;
  for (auto &a : c->arena) dfree(a.p);
  free_paths(c);
  free_pixels(c);
  dfree(c->res);
  dfree(c->jobs);
  dfree(c->items);
  guide_free(c->guide);
  dfree(c->counts);
  dfree(c->stats);
  dfree(c->spill);
  dfree(c->cie);
  for (auto e : c->events) (void)hipEventDestroy(e);
  if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

const char *clv_last_error(const clv_ctx *c) { return c ? c->err.c_str() : "no context"; }

}  // extern "C"

namespace {

/* the device builder's inputs (records in primitive order, their offsets and
 * boxes) in temporary device buffers; the tree goes straight into the arena */
clv_status device_bvh(clv_ctx *c, const HostScene &hs, const ArenaBase &b, DeviceBvhResult *res) {
  const size_t n = hs.prim_unit.size();
  const size_t rec_bytes = hs.prims.size() * sizeof(float), unit_bytes = n * 4, box_bytes = hs.prim_box.size() * 4;
  char *tmp = nullptr;
  HIPCHK(c, hipMalloc((void **)&tmp, rec_bytes + unit_bytes + box_bytes + 512));
  float4 *src = reinterpret_cast<float4 *>(tmp);
  uint32_t *unit = reinterpret_cast<uint32_t *>(tmp + ((rec_bytes + 255) & ~(size_t)255));
  float4 *box = reinterpret_cast<float4 *>(reinterpret_cast<char *>(unit) + ((unit_bytes + 255) & ~(size_t)255));
  hipError_t e = hipMemcpyAsync(src, hs.prims.data(), rec_bytes, hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(unit, hs.prim_unit.data(), unit_bytes, hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(box, hs.prim_box.data(), box_bytes, hipMemcpyHostToDevice, c->stream);
  if (e != hipSuccess) {
    (void)hipStreamSynchronize(c->stream);
    (void)hipFree(tmp);
    return fail(c, CLV_EDEVICE, std::string("device BVH inputs: ") + hipGetErrorString(e));
  }
  DeviceBvhInput in;
  in.box = box;
  in.unit = unit;
  in.src = src;
  in.n = (uint32_t)n;
  for (int a = 0; a < 3; a++) {
    in.clo[a] = hs.clo[a];
    in.chi[a] = hs.chi[a];
  }
  std::string err;
  /* the traversal keeps at most 3 pending children per level in a 72-entry stack */
  const int st = device_build_bvh(c->stream, in, reinterpret_cast<Bvh4Node *>(c->arena[AR_NODES].p), b.nodes,
                                  reinterpret_cast<float4 *>(c->arena[AR_PRIMS].p), b.units, 23u, res, &err);
  (void)hipFree(tmp);
  if (st != CLV_OK) return fail(c, (clv_status)st, err);
  const size_t tree_units = hs.prims.size() / 4 - hs.media_units;
  if (res->units != tree_units) return fail(c, CLV_EINTERNAL, "device BVH build lost primitive records");
  /* the media records follow the tree's */
  if (hs.media_units)
    HIPCHK(c, hipMemcpyAsync(reinterpret_cast<float4 *>(c->arena[AR_PRIMS].p) + b.units + tree_units,
                             hs.prims.data() + 4 * tree_units, (size_t)hs.media_units * 16u, hipMemcpyHostToDevice,
                             c->stream));
  return CLV_OK;
}

clv_status upload_scene(clv_ctx *c, const clv_scene_desc *desc, uint32_t builder, uint32_t *scene_id) {
  HIPCHK(c, hipSetDevice(c->device));
  HostScene hs;
  std::string err;
  const bool on_device = builder == CLV_BUILD_DEVICE;
  auto t0 = std::chrono::steady_clock::now();
  int st = build_host_scene(desc, &hs, &err, on_device);
  if (st != CLV_OK) return fail(c, (clv_status)st, err);
  ArenaBase b;
  b.nodes = (uint32_t)(c->arena[AR_NODES].used / sizeof(Bvh4Node));
  b.units = (uint32_t)(c->arena[AR_PRIMS].used / 16u);
  b.info = (uint32_t)(c->arena[AR_INFO].used / sizeof(PrimInfo));
  b.xforms = (uint32_t)(c->arena[AR_XFORMS].used / sizeof(Xform));
  b.mats = (uint32_t)(c->arena[AR_MATS].used / sizeof(DevMaterial));
  b.spd = (uint32_t)(c->arena[AR_SPD].used / sizeof(float));
  b.lights = (uint32_t)(c->arena[AR_LIGHTS].used / sizeof(DevLight));
  b.lnodes = (uint32_t)(c->arena[AR_LNODES].used / sizeof(DevLightNode));
  st = rebase_host_scene(&hs, b, &err);
  if (st != CLV_OK) return fail(c, (clv_status)st, err);
  SceneRes *s = new (std::nothrow) SceneRes();
  if (!s) return fail(c, CLV_ENOMEM, "host allocation failed");
  s->base = b;
  size_t before[AR_COUNT];
  for (int k = 0; k < AR_COUNT; k++) before[k] = c->arena[k].used;
  struct Part {
    int arr;
    const void *p;
    size_t bytes;
  } parts[AR_COUNT] = {
      /* device build: reserve room for the tree (at most n - 1 nodes) and the records */
      {AR_NODES, on_device ? nullptr : hs.nodes.data(),
       (on_device ? std::max<size_t>(hs.prim_unit.size(), 2) - 1 : hs.nodes.size()) * sizeof(Bvh4Node)},
      {AR_PRIMS, on_device ? nullptr : hs.prims.data(), hs.prims.size() * sizeof(float)},
      {AR_INFO, hs.prim_info.data(), hs.prim_info.size() * sizeof(PrimInfo)},
      {AR_XFORMS, hs.xforms.data(), hs.xforms.size() * sizeof(Xform)},
      {AR_MATS, hs.materials.data(), hs.materials.size() * sizeof(DevMaterial)},
      {AR_SPD, hs.spd.data(), hs.spd.size() * sizeof(float)},
      {AR_LIGHTS, hs.lights.data(), hs.lights.size() * sizeof(DevLight)},
      {AR_LNODES, hs.light_nodes.data(), hs.light_nodes.size() * sizeof(DevLightNode)},
      {AR_LWEIGHTS, hs.light_weights.data(), hs.light_weights.size() * sizeof(float)},
  };
  clv_status r = CLV_OK;
  for (const Part &pt : parts)
    if (r == CLV_OK) r = arena_append(c, c->arena[pt.arr], pt.p, pt.bytes);
  DeviceBvhResult dres;
  if (r == CLV_OK && on_device) {
    r = device_bvh(c, hs, b, &dres);
    if (r == CLV_OK) c->arena[AR_NODES].used = ((size_t)b.nodes + dres.n_nodes) * sizeof(Bvh4Node);
  }
  if (r == CLV_OK) {
    hipError_t e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) r = fail(c, CLV_EDEVICE, hipGetErrorString(e));
  }
  if (r != CLV_OK) { /* roll the arena back to where it was, once no copy reads `hs` any more */
    (void)hipStreamSynchronize(c->stream);
    for (int k = 0; k < AR_COUNT; k++) c->arena[k].used = before[k];
    delete s;
    return r;
  }
  for (int k = 0; k < AR_COUNT; k++) s->end[k] = c->arena[k].used;
  s->n_lights = (uint32_t)hs.lights.size();
  s->light_root = hs.light_root;
  s->bg_spd = hs.background_spd;
  s->has_xforms = !hs.xforms.empty();
  for (const DevMaterial &m : hs.materials)
    s->has_ext = s->has_ext || m.tex != TX_PLAIN || m.cone != 0u || m.kind == CLV_MAT_ISOTROPIC;
  s->camera = hs.camera;
  s->n_nodes = on_device ? dres.n_nodes : (uint32_t)hs.nodes.size();
  s->prim_units = (uint32_t)(hs.prims.size() / 4);
  s->n_prims = hs.n_prims;
  s->n_media = hs.n_media;
  s->media_off = b.units + (uint32_t)(hs.prims.size() / 4) - hs.media_units;
  s->prim_bytes = hs.n_prims ? (uint32_t)(hs.prims.size() * 4 / hs.n_prims) : 0;
  s->depth = on_device ? dres.depth : hs.bvh_depth;
  s->build_ms = on_device ? std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count()
                          : hs.build_ms;
  if (on_device) {
    for (int a = 0; a < 3; a++) {
      float lo = hs.lo[a], hi = hs.hi[a];
      if (!(hi - lo > 1e-6f)) { lo -= 1.0f; hi += 1.0f; }
      s->lo[a] = lo;
      s->hi[a] = hi;
    }
  } else {
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    const Bvh4Node &root = hs.nodes[0];
    for (int k = 0; k < 4; k++) {
      if (root.child[k] == CHILD_EMPTY) continue;
      lo[0] = std::min(lo[0], root.lo_x[k]); hi[0] = std::max(hi[0], root.hi_x[k]);
      lo[1] = std::min(lo[1], root.lo_y[k]); hi[1] = std::max(hi[1], root.hi_y[k]);
      lo[2] = std::min(lo[2], root.lo_z[k]); hi[2] = std::max(hi[2], root.hi_z[k]);
    }
    for (int a = 0; a < 3; a++) {
      if (!(hi[a] - lo[a] > 1e-6f)) { lo[a] -= 1.0f; hi[a] += 1.0f; }
      s->lo[a] = lo[a];
      s->hi[a] = hi[a];
    }
  }
  c->counters.build_ms = s->build_ms;
  uint32_t id = c->next_scene++;
  c->scenes[id] = s;
  *scene_id = id;
  return CLV_OK;
}

}  // namespace

extern "C" {
clv_status clv_scene_upload(clv_ctx *c, const clv_scene_desc *desc, uint32_t *scene_id) {
  return clv_scene_upload_ex(c, desc, CLV_BUILD_HOST, scene_id);
}

clv_status clv_scene_upload_ex(clv_ctx *c, const clv_scene_desc *desc, uint32_t builder, uint32_t *scene_id) {
  if (!c || !scene_id || builder > CLV_BUILD_DEVICE) return CLV_EINVAL;
  return with_room(c, [&] { return upload_scene(c, desc, builder, scene_id); });
}

clv_status clv_scene_validate(const clv_scene_desc *desc, clv_scene_info *info) {
  if (!info) return CLV_EINVAL;
  memset(info, 0, sizeof(*info));
  HostScene hs;
  std::string err;
  int st = build_host_scene(desc, &hs, &err);
  if (st != CLV_OK) {
    snprintf(info->error, sizeof(info->error), "%s", err.c_str());
    return (clv_status)st;
  }
  info->n_objects = hs.n_objects;
  info->n_prims = hs.n_prims;
  info->n_lights = (uint32_t)hs.lights.size();
  info->bvh_nodes = (uint32_t)hs.nodes.size();
  info->bvh_depth = hs.bvh_depth;
  info->light_nodes = (uint32_t)hs.light_nodes.size();
  info->device_bytes = hs.nodes.size() * sizeof(Bvh4Node) + hs.prims.size() * sizeof(float) +
                       hs.prim_info.size() * sizeof(PrimInfo) + hs.xforms.size() * sizeof(Xform) +
                       hs.materials.size() * sizeof(DevMaterial) + hs.spd.size() * sizeof(float) +
                       hs.lights.size() * sizeof(DevLight) + hs.light_nodes.size() * sizeof(DevLightNode) +
                       hs.light_weights.size() * sizeof(float);
  info->build_ms = hs.build_ms;
  return CLV_OK;
}

/* A freed scene's arena range is reused only when it is the last one in the
 * arena (then the arena shrinks back to the end of the previous live scene);
 * freeing every scene empties the arena. */
clv_status clv_scene_free(clv_ctx *c, uint32_t scene_id) {
  if (!c) return CLV_EINVAL;
  auto it = c->scenes.find(scene_id);
  if (it == c->scenes.end()) return fail(c, CLV_EINVAL, "unknown scene id");
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  delete it->second;
  c->scenes.erase(it);
  for (int k = 0; k < AR_COUNT; k++) {
    size_t end = 0;
    for (auto &kv : c->scenes) end = std::max(end, kv.second->end[k]);
    c->arena[k].used = std::min(c->arena[k].used, end);
  }
  return CLV_OK;
}

clv_status clv_render(clv_ctx *c, uint32_t scene_id, const clv_render_opts *o, float *xyz_out, float *xyz_sq_out) {
  if (!c) return CLV_EINVAL;
  CHK(check_opts(c, o));
  clv_job j;
  memset(&j, 0, sizeof(j));
  j.scene_id = scene_id;
  j.opts = *o;
  j.xyz_out = xyz_out;
  j.xyz_sq_out = xyz_sq_out;
  return render_jobs(c, &j, 1);
}

clv_status clv_render_batch(clv_ctx *c, const clv_job *jobs, uint32_t n_jobs) {
  if (!c) return CLV_EINVAL;
  return render_jobs(c, jobs, n_jobs);
}

clv_status clv_plan_passes(const clv_job *jobs, uint32_t n, const clv_tuning *t, clv_pass_item *items, uint32_t cap,
                           uint32_t *n_items, uint32_t *n_passes) {
  if (!jobs || !t || !n_items || !n_passes || n == 0 || n > MAX_JOBS || (cap && !items)) return CLV_EINVAL;
  if (t->target_paths < 1) return CLV_EINVAL;
  std::vector<DevJob> dj(n);
  std::vector<uint32_t> soff(n);
  bool frozen = false; /* as clv_render_batch: the flags of all jobs together */
  for (uint32_t k = 0; k < n; k++) {
    const clv_render_opts &o = jobs[k].opts;
    if (o.width == 0 || o.height == 0 || (uint64_t)o.width * o.height > (1ull << 27) || o.samples == 0 ||
        o.max_depth > 1000)
      return CLV_EINVAL;
    memset(&dj[k], 0, sizeof(DevJob));
    dj[k].width = o.width;
    dj[k].height = o.height;
    dj[k].spp = o.samples;
    dj[k].max_depth = o.max_depth;
    dj[k].guiding = o.guiding;
    soff[k] = o.sample_offset;
    frozen = frozen || (o.flags & CLV_FLAG_GUIDE_FROZEN) != 0;
  }
  PassPlan pl;
  plan_passes(dj, soff, t->target_paths, std::max<uint32_t>(1, t->guide_train_spp), frozen ? 0u : t->guide_rounds,
              t->guide_warmup != 0, &pl);
  const uint32_t passes = (uint32_t)pl.paths.size();
  uint32_t w = 0;
  for (uint32_t p = 0; p < passes; p++)
    for (uint32_t i = pl.first[p]; i < pl.first[p + 1]; i++, w++) {
      if (w >= cap) continue;
      const DevItem &it = pl.items[i];
      items[w].pass = p;
      items[w].job = it.job;
      items[w].samples = it.samples;
      items[w].sample_base = it.sample_base;
      items[w].pass_paths = pl.paths[p];
      items[w].train = pl.train[p];
      items[w].warmup = (it.flags & ITEM_WARMUP) ? 1u : 0u;
    }
  *n_items = (uint32_t)pl.items.size();
  *n_passes = passes;
  return CLV_OK;
}

clv_status clv_tuning_get(const clv_ctx *c, clv_tuning *out) {
  if (!c || !out) return CLV_EINVAL;
  memset(out, 0, sizeof(*out));
  out->target_paths = c->target_paths;
  out->trace_kernel = (uint32_t)c->trace_variant;
  out->lds_bytes = (uint32_t)c->lds_block_bytes;
  out->shade_grid_cap = c->grid_cap;
  out->guide_train_spp = c->guide.train_spp;
  out->guide_alpha = c->guide.alpha;
  out->guide_lr = c->guide.lr;
  out->guide_records = c->guide.records;
  out->guide_wclip = c->guide.wclip;
  out->guide_rounds = c->guide.rounds;
  out->use_graph = c->use_graph ? 1u : 0u;
  out->guide_credit = c->guide.credit;
  out->guide_warmup = c->guide.warmup;
  out->guide_photons = c->guide.photons;
  out->guide_pre_rounds = c->guide.pre_rounds;
  out->guide_gate_density = c->guide.gate_density;
  out->tail_depth = c->tail_depth;
  return CLV_OK;
}

clv_status clv_tuning_set(clv_ctx *c, const clv_tuning *t) {
  if (!c) return CLV_EINVAL;
  if (!t) return fail(c, CLV_EINVAL, "tuning is NULL");
  if (t->target_paths < 65536 || t->target_paths > (1u << 28)) return fail(c, CLV_EINVAL, "target_paths outside [2^16, 2^28]");
  if (t->trace_kernel > CLV_TRACE_LDS_CACHED) return fail(c, CLV_EINVAL, "unknown trace kernel");
  if (t->lds_bytes > 64512) return fail(c, CLV_EINVAL, "lds_bytes above 64512");
  if (t->shade_grid_cap < 1) return fail(c, CLV_EINVAL, "shade_grid_cap must be positive");
  if (t->guide_train_spp < 1) return fail(c, CLV_EINVAL, "guide_train_spp must be positive");
  if (!(t->guide_alpha > 0.0f && t->guide_alpha < 1.0f)) return fail(c, CLV_EINVAL, "guide_alpha outside (0, 1)");
  if (!(t->guide_lr > 0.0f && t->guide_lr < 1.0f)) return fail(c, CLV_EINVAL, "guide_lr outside (0, 1)");
  if (t->guide_records < 64 || t->guide_records > (1u << 24)) return fail(c, CLV_EINVAL, "guide_records outside [64, 2^24]");
  if (!(t->guide_wclip >= 1.0f)) return fail(c, CLV_EINVAL, "guide_wclip below 1");
  if (t->guide_credit > 1u) return fail(c, CLV_EINVAL, "guide_credit is 0 or 1");
  if (t->guide_photons > (1u << 24)) return fail(c, CLV_EINVAL, "guide_photons above 2^24");
  if (t->guide_pre_rounds > 1024u) return fail(c, CLV_EINVAL, "guide_pre_rounds above 1024");
  if (!(t->guide_gate_density >= 0.0f && t->guide_gate_density <= 1e6f))
    return fail(c, CLV_EINVAL, "guide_gate_density outside [0, 1e6]");
  c->target_paths = t->target_paths;
  c->trace_variant = (int)t->trace_kernel;
  c->lds_block_bytes = t->lds_bytes;
  c->grid_cap = t->shade_grid_cap;
  c->guide.train_spp = t->guide_train_spp;
  c->guide.alpha = t->guide_alpha;
  c->guide.lr = t->guide_lr;
  c->guide.records = t->guide_records;
  c->guide.wclip = t->guide_wclip;
  c->guide.rounds = t->guide_rounds;
  c->use_graph = t->use_graph != 0;
  c->guide.credit = t->guide_credit;
  c->guide.warmup = t->guide_warmup;
  c->guide.photons = t->guide_photons;
  c->guide.pre_rounds = t->guide_pre_rounds;
  c->guide.gate_density = t->guide_gate_density;
  c->tail_depth = t->tail_depth;
  return CLV_OK;
}

clv_status clv_guide_reset(clv_ctx *c, uint64_t seed) {
  if (!c) return CLV_EINVAL;
  HIPCHK(c, hipSetDevice(c->device));
  return guide_reset(c, seed);
}

clv_status clv_guide_params(clv_ctx *c, float *out, uint32_t n) {
  if (!c) return CLV_EINVAL;
  if (!out || n < GD_NPARAM) return fail(c, CLV_EINVAL, "params_out needs CLV_GUIDE_NPARAM floats");
  HIPCHK(c, hipSetDevice(c->device));
  if (!c->guide.init) CHK(guide_reset(c, 1));
  HIPCHK(c, hipMemcpyAsync(out, c->guide.P, GD_NPARAM * sizeof(float), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CLV_OK;
}

clv_status clv_guide_set_params(clv_ctx *c, const float *in, uint32_t n) {
  if (!c) return CLV_EINVAL;
  if (!in || n != GD_NPARAM) return fail(c, CLV_EINVAL, "params need exactly CLV_GUIDE_NPARAM floats");
  HIPCHK(c, hipSetDevice(c->device));
  if (!c->guide.init) CHK(guide_reset(c, 1));
  GuideState &g = c->guide;
  HIPCHK(c, hipMemcpyAsync(g.P, in, GD_NPARAM * sizeof(float), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemsetAsync(g.M, 0, GD_NPARAM * sizeof(float), c->stream));
  HIPCHK(c, hipMemsetAsync(g.V, 0, GD_NPARAM * sizeof(float), c->stream));
  launch_guide_halves(c->stream, g.P, g.Wh);
  HIPCHK(c, hipStreamSynchronize(c->stream));
  g.trained = true;
  return CLV_OK;
}

clv_status clv_guide_eval(clv_ctx *c, const float *in, uint32_t n, float *raw, float *lobes) {
  if (!c) return CLV_EINVAL;
  if (!in || n == 0 || n > (1u << 24)) return fail(c, CLV_EINVAL, "inputs: 1..2^24 rows of 7 floats");
  HIPCHK(c, hipSetDevice(c->device));
  if (!c->guide.init) CHK(guide_reset(c, 1));
  float *din = nullptr, *draw = nullptr, *dlob = nullptr;
  clv_status st = with_room(c, [&]() -> clv_status {
    if (!din) HIPCHK(c, dalloc(&din, 7 * (size_t)n));
    if (!draw) HIPCHK(c, dalloc(&draw, (size_t)GD_OUT * n));
    if (!dlob) HIPCHK(c, dalloc(&dlob, (size_t)GD_OUT * n));
    return CLV_OK;
  });
  if (st == CLV_OK) {
    hipError_t e = hipMemcpyAsync(din, in, 7 * sizeof(float) * n, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) {
      launch_guide_eval(c->stream, din, n, c->guide.Wh, c->guide.P, draw, dlob);
      e = hipGetLastError();
    }
    if (e == hipSuccess && raw) e = hipMemcpyAsync(raw, draw, sizeof(float) * GD_OUT * n, hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess && lobes) e = hipMemcpyAsync(lobes, dlob, sizeof(float) * GD_OUT * n, hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) st = fail(c, e == hipErrorOutOfMemory ? CLV_ENOMEM : CLV_EDEVICE, hipGetErrorString(e));
  }
  dfree(din);
  dfree(draw);
  dfree(dlob);
  return st;
}

clv_status clv_guide_grad(clv_ctx *c, const float *samples, uint32_t n, float *grad_out) {
  if (!c) return CLV_EINVAL;
  if (!samples || !grad_out || n == 0 || n > (1u << 20)) return fail(c, CLV_EINVAL, "samples: 1..2^20 rows of 11 floats");
  for (uint32_t i = 0; i < n; i++)
    if (!(samples[11 * (size_t)i + 10] > 0.0f)) return fail(c, CLV_EINVAL, "sample weights must be positive");
  HIPCHK(c, hipSetDevice(c->device));
  if (!c->guide.init) CHK(guide_reset(c, 1));
  GuideState &g = c->guide;
  CHK(with_room(c, [&]() -> clv_status {
    CHK(guide_ensure_paths(c, (n + GD_SLOTS - 1) / GD_SLOTS));
    return guide_ensure_partial(c, (n + 63) / 64);
  }));
  const uint32_t stamp = ++g.stamp;
  std::vector<GuideRec> recs(n);
  std::vector<float> recL(n);
  for (uint32_t i = 0; i < n; i++) {
    const float *sm = samples + 11 * (size_t)i;
    GuideRec &r = recs[i];
    memset(&r, 0, sizeof(r));
    for (int k = 0; k < 3; k++) {
      r.p[k] = sm[k];
      r.n[k] = sm[3 + k];
      r.d[k] = sm[7 + k];
    }
    r.lam = sm[6];
    r.pdf = 1.0f;
    r.cosv = 1.0f;
    r.t0 = 1.0f;
    recL[i] = sm[10];
    r.stamp = stamp;
  }
  float *dgrad = nullptr;
  HIPCHK(c, dalloc(&dgrad, GD_NPARAM));
  hipError_t e = hipMemcpyAsync(g.rec, recs.data(), n * sizeof(GuideRec), hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(g.recL, recL.data(), n * sizeof(float), hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) {
    launch_guide_collect(c->stream, g.rec, g.recL, n, g.bcount, g.bweight, g.totals, g.list, n, nullptr);
    launch_guide_step(c->stream, g.rec, g.recL, g.list, g.totals, n, 0, n, FLT_MAX, g.P, g.M, g.V, g.Wh, g.partial, g.lr,
                      dgrad);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(grad_out, dgrad, GD_NPARAM * sizeof(float), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  dfree(dgrad);
  if (e != hipSuccess) return fail(c, CLV_EDEVICE, hipGetErrorString(e));
  return CLV_OK;
}

clv_status clv_autotune(clv_ctx *c, const clv_job *jobs, uint32_t n, uint64_t trial_samples, clv_tuning *best_out) {
  if (!c) return CLV_EINVAL;
  if (!jobs || n == 0 || n > MAX_JOBS) return fail(c, CLV_EINVAL, "no jobs");
  if (trial_samples == 0) trial_samples = 1ull << 26;
  uint64_t total = 0;
  for (uint32_t k = 0; k < n; k++) {
    CHK(check_opts(c, &jobs[k].opts));
    total += (uint64_t)jobs[k].opts.width * jobs[k].opts.height * jobs[k].opts.samples;
  }
  /* the shortened batch: every job keeps its shape, with its samples scaled */
  std::vector<clv_job> trial(jobs, jobs + n);
  std::vector<std::vector<float>> bufs(n);
  uint64_t tsamples = 0;
  for (uint32_t k = 0; k < n; k++) {
    clv_render_opts &o = trial[k].opts;
    uint64_t spp = total > trial_samples ? (uint64_t)o.samples * trial_samples / total : o.samples;
    o.samples = (uint32_t)std::max<uint64_t>(1, spp);
    o.flags = 0;
    bufs[k].resize(3 * (size_t)o.width * o.height);
    trial[k].xyz_out = bufs[k].data();
    trial[k].xyz_sq_out = nullptr;
    tsamples += (uint64_t)o.width * o.height * o.samples;
  }
  clv_tuning start;
  CHK(clv_tuning_get(c, &start));
  struct Cand {
    uint32_t target, kernel, lds;
  };
  std::vector<Cand> cands;
  bool any_guided = false;
  for (uint32_t k = 0; k < n; k++) any_guided = any_guided || jobs[k].opts.guiding == CLV_GUIDE_ON;
  for (uint32_t lg = 22; lg <= 26; lg++) { /* 2^22: the automatic size */
    const uint32_t tgt = 1u << lg;
    if (lg > 22 && (uint64_t)(tgt >> 1) >= tsamples) break; /* larger passes than the work change nothing */
    /* whole paths: the automatic size holds the trial in one pass, so another size that does is the same render here,
     * though not where the batch has more samples than its trial */
    if (any_guided || lg == 22 || tgt < tsamples) {
      cands.push_back({tgt, CLV_TRACE_LDS_CACHED, 64512});
      cands.push_back({tgt, CLV_TRACE_LDS_CACHED, 16384});
    }
    cands.push_back({tgt, CLV_TRACE_SIMPLE, 64512});
  }
  clv_tuning best = start;
  double best_ms = 1e300;
  bool warmed = false;
  const bool graph0 = c->use_graph;
  c->use_graph = false; /* trials never repeat: no capture */
  for (const Cand &cd : cands) {
    clv_tuning t = start;
    t.target_paths = cd.target;
    t.trace_kernel = cd.kernel;
    t.lds_bytes = cd.lds;
    CHK(clv_tuning_set(c, &t));
    clv_status st = render_jobs(c, trial.data(), n);
    if (st == CLV_ENOMEM) continue; /* too large a pass for the device: skip */
    if (st != CLV_OK) {
      (void)clv_tuning_set(c, &start);
      c->use_graph = graph0;
      return st;
    }
    if (!warmed) { /* first trial also pays allocation and first-launch costs: repeat it */
      warmed = true;
      st = render_jobs(c, trial.data(), n);
      if (st != CLV_OK) {
        (void)clv_tuning_set(c, &start);
        c->use_graph = graph0;
        return st;
      }
    }
    const double ms = c->counters.render_ms;
    if (ms < best_ms) {
      best_ms = ms;
      best = t;
    }
  }
  /* the best shape with the late bounces in one launch (k_tail): fewer launches where few paths are
   * left, which pays on small images; not for batches with guided jobs, whose vertices in the tail
   * sample the plain mixture, nor for whole paths in one launch, which have no tail */
  CHK(clv_tuning_set(c, &best));
  if (!any_guided && best_ms < 1e300 && !whole_paths(c, false, 0u)) {
    const clv_tuning shape = best;
    for (uint32_t d = 2; d <= 4; d++) {
      clv_tuning t = shape;
      t.tail_depth = d;
      CHK(clv_tuning_set(c, &t));
      clv_status st = render_jobs(c, trial.data(), n);
      if (st != CLV_OK) {
        (void)clv_tuning_set(c, &start);
        c->use_graph = graph0;
        return st;
      }
      const double ms = c->counters.render_ms;
      if (ms < best_ms) {
        best_ms = ms;
        best = t;
      }
    }
  }
  best.use_graph = graph0 ? 1u : 0u;
  CHK(clv_tuning_set(c, &best));
  if (best_out) *best_out = best;
  return CLV_OK;
}

clv_status clv_primary_hits(clv_ctx *c, uint32_t scene_id, const clv_render_opts *o, uint32_t *ids, float *ts) {
  if (!c) return CLV_EINVAL;
  CHK(check_opts(c, o));
  if (!ids) return fail(c, CLV_EINVAL, "prim_id_out is NULL");
  auto it = c->scenes.find(scene_id);
  if (it == c->scenes.end()) return fail(c, CLV_EINVAL, "unknown scene id");
  HIPCHK(c, hipSetDevice(c->device));
  const uint32_t W = o->width, H = o->height, WH = W * H;
  TraceGeom geom;
  const int variant = trace_variant_for(c, it->second->n_media > 0);
  CHK(with_room(c, [&]() -> clv_status {
    CHK(ensure_paths(c, WH));
    CHK(ensure_pixels(c, WH));
    CHK(ensure_tables(c, 1, 1));
    return trace_geometry(c, it->second, 0, &geom, variant);
  }));
  DevJob jb = make_job(it->second, it->second->camera, o);
  DevItem item;
  memset(&item, 0, sizeof(item));
  item.pixels = WH;
  item.samples = 1;
  item.sample_base = o->sample_offset;
  StreamDrain drain{c->stream}; /* jb and item outlive the copies from them */
  HIPCHK(c, hipMemcpyAsync(c->jobs, &jb, sizeof(jb), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->items, &item, sizeof(item), hipMemcpyHostToDevice, c->stream));
  DevScene ds = arena_view(c);
  ds.has_xforms = it->second->has_xforms ? 1u : 0u;
  ds.has_ext = it->second->has_ext ? 1u : 0u;
  ds.has_media = it->second->n_media > 0 ? 1u : 0u;
  GenParams gp;
  memset(&gp, 0, sizeof(gp));
  gp.items = c->items;
  gp.n_items = 1;
  gp.paths = WH;
  launch_generate(c->stream, ds, c->pb, gp);
  launch_set_count(c->stream, c->counts, CNT_FETCH, 0u);
  TraceArgs ta;
  memset(&ta, 0, sizeof(ta));
  ta.counts = c->counts;
  ta.n_direct = WH;
  ta.ids = c->ids;
  ta.ts = c->ts;
  ta.spill = c->spill;
  fill_trace_args(&ta, geom);
  if (variant == TRACE_LDS)
    launch_trace_lds(c->stream, ds, c->pb, ta, geom.blocks, geom.lds_bytes, false, 1);
  else
    launch_primary(c->stream, ds, c->pb, ta, geom.blocks, variant);
  HIPCHK(c, hipGetLastError());
  const size_t bytes = sizeof(uint32_t) * (size_t)WH;
  std::vector<CopyArray> arrays{{c->ids, bytes}};
  std::vector<CopySeg> segs{{0, 0, bytes, ids}};
  if (ts) {
    arrays.push_back({c->ts, bytes});
    segs.push_back({1, 0, bytes, ts});
  }
  HIPCHK(c, c->copy.run(c->stream, arrays, segs, nullptr, nullptr));
  return CLV_OK;
}

static_assert(NA_SCRATCH_BYTES == CLV_NOALLOC_SCRATCH_BYTES, "the header states the scratch size");

clv_status clv_primary_hits_noalloc(clv_ctx *c, uint32_t scene_id, const clv_render_opts *o, uint32_t *ids, float *ts) {
  if (!c) return CLV_EINVAL;
  CHK(check_opts(c, o));
  if (!ids) return fail(c, CLV_EINVAL, "prim_id_out is NULL");
  auto it = c->scenes.find(scene_id);
  if (it == c->scenes.end()) return fail(c, CLV_EINVAL, "unknown scene id");
  const uint64_t WH = (uint64_t)o->width * o->height;
  if (WH > CLV_NOALLOC_MAX_PIXELS)
    return fail(c, CLV_EINVAL, "clv_primary_hits_noalloc covers at most CLV_NOALLOC_MAX_PIXELS pixels per call");
  if (!c->na_scratch) return fail(c, CLV_EDEVICE, "no device scratch array on this device");
  HIPCHK(c, hipSetDevice(c->device));
  for (void *p : {(void *)ids, (void *)ts}) {
    if (!p) continue;
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess || a.type != hipMemoryTypeDevice || a.device != c->device) {
      (void)hipGetLastError();
      return fail(c, CLV_EINVAL, "prim_id_out and t_out must be device memory of the context's device");
    }
  }
  const SceneRes *s = it->second;
  const NaView v = na_view(c->na_scratch);
  const DevJob jb = make_job(s, s->camera, o);
  DevScene ds = arena_view(c);
  ds.jobs = v.job;
  ds.has_xforms = s->has_xforms ? 1u : 0u;
  ds.has_ext = s->has_ext ? 1u : 0u;
  ds.has_media = s->n_media > 0 ? 1u : 0u;
  /* chunks of NA_CHUNK pixels: the chunk's item starts the slot numbering at
   * its first pixel (path_base wraps to -p0), so slot i is pixel p0 + i */
  for (uint32_t p0 = 0; p0 < (uint32_t)WH; p0 += NA_CHUNK) {
    const uint32_t n = std::min<uint32_t>(NA_CHUNK, (uint32_t)WH - p0);
    DevItem item;
    memset(&item, 0, sizeof(item));
    item.path_base = 0u - p0;
    item.pixels = (uint32_t)WH;
    item.samples = 1;
    item.sample_base = o->sample_offset;
    launch_na_setup(c->stream, jb, item, v);
    GenParams gp;
    memset(&gp, 0, sizeof(gp));
    gp.items = v.item;
    gp.n_items = 1;
    gp.paths = n;
    launch_generate(c->stream, ds, v.pb, gp);
    TraceArgs ta;
    memset(&ta, 0, sizeof(ta));
    ta.counts = v.counts;
    ta.n_direct = n;
    ta.ids = ids + p0;
    ta.ts = ts ? ts + p0 : v.ts;
    ta.spill = v.spill;
    launch_primary(c->stream, ds, v.pb, ta, NA_BLOCKS, TRACE_SIMPLE);
  }
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CLV_OK;
}

clv_status clv_render_debug(clv_ctx *c, uint32_t scene_id, const clv_render_opts *o, uint32_t mode, float *xyz_out) {
  if (!c) return CLV_EINVAL;
  CHK(check_opts(c, o));
  if (!xyz_out) return fail(c, CLV_EINVAL, "xyz_out is NULL");
  if (mode < CLV_MODE_NORMAL_MAP || mode > CLV_MODE_PRIMITIVE_TEST_COUNT)
    return fail(c, CLV_EINVAL, "mode is not a debug mode (path tracing is clv_render)");
  auto it = c->scenes.find(scene_id);
  if (it == c->scenes.end()) return fail(c, CLV_EINVAL, "unknown scene id");
  HIPCHK(c, hipSetDevice(c->device));
  const uint32_t W = o->width, H = o->height, WH = W * H;
  const uint32_t blocks = c->trace_blocks;
  CHK(with_room(c, [&]() -> clv_status {
    CHK(ensure_paths(c, WH));
    CHK(ensure_pixels(c, WH));
    CHK(ensure_tables(c, 1, 1));
    return ensure_spill(c, trace_spill_words(blocks));
  }));
  DevJob jb = make_job(it->second, it->second->camera, o);
  StreamDrain drain{c->stream}; /* jb outlives the copy from it */
  HIPCHK(c, hipMemcpyAsync(c->jobs, &jb, sizeof(jb), hipMemcpyHostToDevice, c->stream));
  DevScene ds = arena_view(c);
  ds.has_xforms = it->second->has_xforms ? 1u : 0u;
  ds.has_ext = it->second->has_ext ? 1u : 0u;
  ds.has_media = it->second->n_media > 0 ? 1u : 0u;
  DebugArgs da;
  memset(&da, 0, sizeof(da));
  da.width = W;
  da.height = H;
  da.sample = o->sample_offset;
  da.mode = mode;
  /* LinSrgb -> Xyz<E>: the sRGB primaries' matrix, then Bradford D65 -> E */
  {
    const double xy[3][2] = {{0.64, 0.33}, {0.30, 0.60}, {0.15, 0.06}};
    const double wt[3] = {0.95047, 1.0, 1.08883};
    const double B[3][3] = {{0.8951, 0.2664, -0.1614}, {-0.7502, 1.7135, 0.0367}, {0.0389, -0.0685, 1.0296}};
    double P[3][3], M[3][3], A[3][3];
    for (int k = 0; k < 3; k++) {
      P[0][k] = xy[k][0] / xy[k][1];
      P[1][k] = 1.0;
      P[2][k] = (1.0 - xy[k][0] - xy[k][1]) / xy[k][1];
    }
    double S[3];
    inv3_apply(P, wt, S);
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) M[i][j] = P[i][j] * S[j];
    bradford(B, wt, A);
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) da.lin_to_xyz[3 * i + j] = (float)(A[i][0] * M[0][j] + A[i][1] * M[1][j] + A[i][2] * M[2][j]);
  }
  launch_generate_debug(c->stream, ds, c->pb, da);
  launch_zero_u64(c->stream, c->stats, 8);
  TraceArgs ta;
  memset(&ta, 0, sizeof(ta));
  ta.counts = c->counts;
  ta.n_direct = WH;
  ta.ids = c->ids;
  ta.ts = c->ts;
  ta.spill = c->spill;
  ta.stats = (unsigned long long *)c->stats;
  uint32_t *rc = reinterpret_cast<uint32_t *>(c->acc64);  /* 2 words per ray within the 6 the pixel holds */
  ta.ray_counts = rc;
  launch_primary_counting(c->stream, ds, c->pb, ta, blocks);
  launch_debug_color(c->stream, ds, c->pb, da, rc, c->out);
  HIPCHK(c, hipGetLastError());
  const size_t bytes = sizeof(float) * 3 * (size_t)WH;
  uint64_t st[8];
  HIPCHK(c, c->copy.run(c->stream, {{c->out, bytes}}, {{0, 0, bytes, xyz_out}}, c->stats, st));
  clv_counters cn;
  memset(&cn, 0, sizeof(cn));
  cn.samples = WH;
  cn.rays = WH;
  cn.node_visits = st[0];
  cn.prim_tests = st[1];
  c->counters = cn;
  return CLV_OK;
}

clv_status clv_counters_get(const clv_ctx *c, clv_counters *out) {
  if (!c || !out) return CLV_EINVAL;
  *out = c->counters;
  return CLV_OK;
}

}  // extern "C"
