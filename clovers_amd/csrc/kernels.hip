/*
 * kernels.hip -- spectral path tracer for MI355X (gfx950).
 *
 * The reference evaluates one camera sample with a recursive function
 * (clovers-cli/src/trace.rs:21-122) per pixel per row thread
 * (draw_cpu.rs:101-146).  Here a plain pass is one launch whose blocks carry
 * paths in registers from the camera to their end (k_paths).  Where something
 * happens between the bounces (the guiding network, timing, counting), every
 * sample is a path slot in HBM and a bounce is two kernels over all live paths:
 *
 *   extend  closest hit of every queued ray (4-wide BVH, short per-lane stack
 *           in LDS); each hit is appended to one of five shading queues by
 *           material class (miss / emitter / Lambertian / metal / glass) with
 *           one wave-aggregated atomic per class -- ballot + popcount prefix.
 *   shade   one launch over the concatenated class queues in 64-aligned
 *           chunks, so every wave runs a single material's code; surviving
 *           paths are appended to the next ray queue the same way.
 *
 * The iterative form accumulates L += T * emitted at each vertex and
 * multiplies T by the vertex weight, which is the reference's recursion
 * unrolled: specular vertices contribute atten * L_next (trace.rs:74-79), diffuse
 * vertices emitted + atten * pdf_bsdf / pdf_mix * L_next (trace.rs:116-119).
 * `resolve` applies the per-sample estimator of draw_cpu.rs:130-142 and sums
 * samples per pixel in sample order.
 */
#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include "clv_layout.h"
#include "copyout.h"
#include "kernels.h"

namespace clv {

#define PI_F 3.14159265358979323846f
#define EPS_ACNE 0.001f   /* EPSILON_SHADOW_ACNE, lib.rs:114 */
#define EPS_RECT 0.0001f  /* EPSILON_RECT_THICKNESS, lib.rs:116 */
#define MISS_WORD 0xFFFFFFFFu

/* ------------------------------------------------------------- helpers --- */
struct V {
  float x, y, z;
};
__device__ __forceinline__ V mk(float x, float y, float z) { V r; r.x = x; r.y = y; r.z = z; return r; }
__device__ __forceinline__ V operator+(V a, V b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ V operator-(V a, V b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ V operator-(V a) { return mk(-a.x, -a.y, -a.z); }
__device__ __forceinline__ V operator*(float s, V a) { return mk(s * a.x, s * a.y, s * a.z); }
__device__ __forceinline__ V operator/(V a, float s) { return mk(a.x / s, a.y / s, a.z / s); }
__device__ __forceinline__ float dot(V a, V b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V cross(V a, V b) { return mk(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x); }
__device__ __forceinline__ V unit(V a) { return a / sqrtf(dot(a, a)); }
__device__ __forceinline__ V xyz(float4 f) { return mk(f.x, f.y, f.z); }
__device__ __forceinline__ float comp(V a, int i) { return i == 0 ? a.x : (i == 1 ? a.y : a.z); }
__device__ __forceinline__ uint32_t as_u(float f) { return __float_as_uint(f); }

/* PCG32 (O'Neill 2014), bit-identical to the oracle's per-path streams */
__device__ __forceinline__ uint32_t pcg_next(uint64_t &s) {
  uint64_t old = s;
  s = old * 6364136223846793005ull + 1442695040888963407ull;
  uint32_t xs = (uint32_t)(((old >> 18u) ^ old) >> 27u);
  uint32_t rot = (uint32_t)(old >> 59u);
  return (xs >> rot) | (xs << ((-rot) & 31u));
}
__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
__device__ __forceinline__ uint64_t pcg_for_path(uint64_t seed, uint32_t pixel, uint32_t sample) {
  uint64_t s = splitmix64(seed ^ splitmix64(((uint64_t)sample << 32) | (uint64_t)pixel));
  (void)pcg_next(s);
  return s;
}
__device__ __forceinline__ float rnd(uint64_t &s) { return (float)(pcg_next(s) >> 8) * 0x1p-24f; }
__device__ __forceinline__ bool coin(uint64_t &s) { return (pcg_next(s) >> 31) != 0u; }
__device__ __forceinline__ float rnd_pm1(uint64_t &s) { return 2.0f * rnd(s) - 1.0f; }
/* the free-flight uniform of a constant medium, in [0, 1) like rnd: a hash of
 * the path's stream state at the bounce and the medium's object id (the
 * reference draws it from the path's generator inside the traversal, in its
 * own tree's order, constant_medium.rs:103) */
__device__ __forceinline__ float medium_u01(uint64_t state, uint32_t id) {
  const uint64_t h = splitmix64(state ^ (((uint64_t)id + 1ull) * 0xD1B54A32D192ED03ull));
  return (float)(uint32_t)(h >> 40) * 0x1p-24f;
}

/* wave-aggregated append of `item` to queue q (counter *cnt) when pred */
__device__ __forceinline__ void wave_append(bool pred, uint32_t item, uint32_t *q, uint32_t *cnt) {
  uint64_t mask = __ballot(pred);
  if (mask == 0) return;
  uint32_t lane = __lane_id();
  uint32_t leader = (uint32_t)__ffsll((unsigned long long)mask) - 1u;
  uint32_t base = 0;
  if (lane == leader) base = atomicAdd(cnt, (uint32_t)__popcll(mask));
  base = __shfl(base, (int)leader);
  uint64_t below = mask & ((1ull << lane) - 1ull);
  if (pred) q[base + (uint32_t)__popcll(below)] = item;
}

/* Block-aggregated append to queue `cls` (cls >= NC: no append): the
 * lane's position in the queue (~0u if none).  Each wave counts its lanes
 * per queue with a ballot and writes the counts to LDS; NC threads turn them
 * into per-wave offsets and do one global atomic per queue for the whole
 * block.  Every thread of the block must call this (it synchronises the
 * block).  `lds` holds NC * (BLOCK/64) + NC words.  block_append also stores
 * `item` at that position. */
template <int NC, int BLOCK>
__device__ __forceinline__ uint32_t block_append_pos(uint32_t cls, uint32_t *counters, uint32_t *lds) {
  constexpr int WAVES = BLOCK / 64;
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  const uint64_t lt = (1ull << lane) - 1ull;
  uint32_t rank = 0;
#pragma unroll
  for (int c = 0; c < NC; c++) {
    uint64_t m = __ballot(cls == (uint32_t)c);
    if (lane == 0) lds[c * WAVES + wave] = (uint32_t)__popcll(m);
    if (cls == (uint32_t)c) rank = (uint32_t)__popcll(m & lt);
  }
  __syncthreads();
  if (threadIdx.x < (uint32_t)NC) {
    const uint32_t c = threadIdx.x;
    uint32_t sum = 0;
    for (int w = 0; w < WAVES; w++) {
      uint32_t t = lds[c * WAVES + w];
      lds[c * WAVES + w] = sum;
      sum += t;
    }
    lds[NC * WAVES + c] = sum ? atomicAdd(&counters[c], sum) : 0u;
  }
  __syncthreads();
  const uint32_t pos = cls < (uint32_t)NC ? lds[NC * WAVES + cls] + lds[cls * WAVES + wave] + rank : 0xFFFFFFFFu;
  __syncthreads();
  return pos;
}
template <int NC, int BLOCK>
__device__ __forceinline__ void block_append(uint32_t cls, uint32_t item, uint32_t *const *queues, uint32_t *counters,
                                             uint32_t *lds) {
  const uint32_t pos = block_append_pos<NC, BLOCK>(cls, counters, lds);
  if (cls < (uint32_t)NC) queues[cls][pos] = item;
}

/* -------------------------------------------------- primitive tests --- */
/* Sphere::hit (objects/sphere.rs:70-125): strict t bounds, near root first */
__device__ __forceinline__ bool sphere_t(V c, float r, V o, V d, float tmin, float tmax, float &t) {
  V oc = o - c;
  float a = dot(d, d);
  float half_b = dot(oc, d);
  float cc = dot(oc, oc) - r * r;
  float disc = half_b * half_b - a * cc;
  if (!(disc > 0.0f)) return false;
  float root = sqrtf(disc);
  float t0 = (-half_b - root) / a;
  if (t0 < tmax && t0 > tmin) { t = t0; return true; }
  float t1 = (-half_b + root) / a;
  if (t1 < tmax && t1 > tmin) { t = t1; return true; }
  return false;
}

/* Quad::hit (objects/quad.rs:88-132): |n.d| < 1e-4 rejected, inclusive t and (a, b) bounds */
/* Quad::hit (quad.rs:88-132) and Triangle::hit (triangle.rs:120-166): the
 * plane distance, then the plane coordinates (alpha, beta) of the hit point,
 * inside if both are in [0, 1] (and alpha + beta <= 1 for a triangle,
 * triangle.rs:229-234), computed with the reference's operations so hits and
 * distances are the reference's own, including where a ray meets a shared
 * edge and the rounding puts it outside both triangles */
template <bool TRI>
__device__ __forceinline__ bool plane_t(const float4 *rec, V o, V d, float tmin, float tmax, float &t) {
  float4 f0 = rec[0], f1 = rec[1], f2 = rec[2], f3 = rec[3], f4 = rec[4];
  V q = xyz(f0), u = xyz(f1), v = xyz(f2), n = xyz(f3), w = xyz(f4);
  float denom = dot(n, d);
  if (fabsf(denom) < EPS_RECT) return false;
  float tt = (-f2.w - dot(n, o)) / denom;
  if (tt < tmin || tt > tmax) return false;
  V p = o + tt * d;
  V ph = p - q;
  float alpha = dot(w, cross(ph, v));
  float beta = dot(w, cross(u, ph));
  if (!(alpha >= 0.0f && alpha <= 1.0f && beta >= 0.0f && beta <= 1.0f)) return false;
  if (TRI && !(alpha + beta <= 1.0f)) return false;
  t = tt;
  return true;
}


/* RotateY/Translate chain, outermost op first (rotate.rs:97-113, translate.rs:60-66) */
__device__ __forceinline__ void xform_ray(const Xform &x, V &o, V &d) {
  for (uint32_t k = 0; k < x.n_ops; k++) {
    const XformOp &op = x.ops[k];
    if (op.kind == XF_TRANSLATE) {
      o = o - mk(op.a, op.b, op.c);
    } else {
      float s = op.a, c = op.b;
      o = mk(c * o.x - s * o.z, o.y, s * o.x + c * o.z);
      d = unit(mk(c * d.x - s * d.z, d.y, s * d.x + c * d.z));
    }
  }
}

/* Boxy::hit (boxy.rs:87-104) over its six quad records: the closest side */
__device__ __forceinline__ bool box_t(const float4 *sides, V o, V d, float tmin, float tmax, float &t) {
  bool any = false;
  float closest = tmax;
  for (int k = 0; k < 6; k++) {
    float tt;
    if (plane_t<false>(sides + PREC_QUAD * k, o, d, tmin, closest, tt)) {
      closest = tt;
      any = true;
    }
  }
  t = closest;
  return any;
}

#define EPS_MEDIUM 0.0001f /* EPSILON_CONSTANT_MEDIUM, lib.rs:119 */

/* ConstantMedium::hit (constant_medium.rs:65-126): the boundary's entry
 * over (-inf, inf) and exit after it, clipped to [tmin, tmax] and to 0, an
 * exponential free flight of mean 1/density along the ray's length */
__device__ __forceinline__ bool medium_t(const DevScene &sc, const float4 *rec, V o, V d, float tmin, float tmax,
                                         uint64_t state, float &t) {
  const float4 f0 = rec[0];
  float t1, t2;
  if (as_u(f0.y) == MED_SPHERE) {
    const float4 b = rec[2];
    if (!sphere_t(xyz(b), b.w, o, d, -INFINITY, INFINITY, t1)) return false;
    if (!sphere_t(xyz(b), b.w, o, d, t1 + EPS_MEDIUM, INFINITY, t2)) return false;
  } else {
    if (!box_t(rec + 2, o, d, -INFINITY, INFINITY, t1)) return false;
    if (!box_t(rec + 2, o, d, t1 + EPS_MEDIUM, INFINITY, t2)) return false;
  }
  if (t1 < tmin) t1 = tmin;
  if (t2 > tmax) t2 = tmax;
  if (t1 >= t2) return false;
  if (t1 < 0.0f) t1 = 0.0f;
  const float len = sqrtf(dot(d, d));
  const float inside = (t2 - t1) * len;
  const float u = medium_u01(state, sc.info[as_u(rec[1].w)].report_id);
  const float hd = f0.x * logf(u);
  if (hd > inside) return false;
  t = t1 + hd / len;
  return true;
}

/* test one primitive record of a BVH leaf (media are not in the tree); on a
 * hit inside [tmin, tbest] update tbest */
__device__ __forceinline__ uint32_t prim_units(uint32_t type) { return PREC_OF(type); }

template <bool HAS_XFORM>
__device__ __forceinline__ bool test_prim(const DevScene &sc, const float4 *rec, uint32_t hdr, V o, V d, float time,
                                          float tmin, float tmax, float &t) {
  uint32_t type = hdr & PT_TYPE_MASK;
  uint32_t xf = hdr >> PT_XF_SHIFT;
  if (HAS_XFORM && xf) xform_ray(sc.xforms[xf - 1u], o, d);
  if (type == PT_SPHERE) {
    float4 f0 = rec[0], f1 = rec[1];
    return sphere_t(xyz(f0), f1.x, o, d, tmin, tmax, t);
  }
  if (type == PT_TRI) return plane_t<true>(rec, o, d, tmin, tmax, t);
  if (type == PT_MSPHERE) { /* MovingSphere::hit (moving_sphere.rs:106-160): the sphere at the ray's time */
    float4 f0 = rec[0], f1 = rec[1], f2 = rec[2];
    return sphere_t(xyz(f0) + time * xyz(f2), f1.x, o, d, tmin, tmax, t);
  }
  return plane_t<false>(rec, o, d, tmin, tmax, t);
}

/* ------------------------------------------------------ traversal --- */
/* Per-lane traversal stack: the top STACK_LDS entries live in LDS
 * (interleaved so that a wave's lanes hit distinct banks), deeper entries in
 * a per-thread slice of a global buffer.  The host refuses BVHs whose depth
 * could need more than STACK_TOTAL entries (3 pending children per level). */
#define STACK_LDS 16
#define STACK_TOTAL 72
#define STACK_GLOBAL (STACK_TOTAL - STACK_LDS)
#define TRACE_BLOCK 256

/* The LDS part of a stack is read and written through pointers typed for the
 * LDS address space: with generic pointers the compiler merges a pop's two
 * loads (LDS or global slice) into one flat load, which waits on both the LDS
 * and the vector-memory counters. */
typedef __attribute__((address_space(3))) uint32_t lds_u32;
__device__ __forceinline__ uint32_t lds_load(const uint32_t *p) { return *(const lds_u32 *)p; }
__device__ __forceinline__ void lds_store(uint32_t *p, uint32_t v) { *(lds_u32 *)p = v; }

/* state of one lane's ray */
struct Lane {
  V o, d, inv, oi;
  float tb;          /* closest accepted distance so far (the reference starts at f32::MAX, trace.rs:44) */
  float time;        /* the ray's instant in [0, 1): moving spheres are tested where they are then */
  uint32_t best;     /* record offset of the closest hit, MISS_WORD if none */
  uint32_t word;     /* node / leaf word being processed, CHILD_EMPTY when the traversal is over */
  uint32_t path;
  int sp;
  bool live;
};

/* a lane's traversal state for the ray o + t d at instant `time`, from the
 * scene root `root` */
__device__ __forceinline__ void lane_start_ray(Lane &L, V o, V d, float time, uint32_t root) {
  L.o = o;
  L.d = d;
  L.time = time;
  V dd = mk(fabsf(L.d.x) < 1e-20f ? copysignf(1e-20f, L.d.x) : L.d.x,
            fabsf(L.d.y) < 1e-20f ? copysignf(1e-20f, L.d.y) : L.d.y,
            fabsf(L.d.z) < 1e-20f ? copysignf(1e-20f, L.d.z) : L.d.z);
  L.inv = mk(1.0f / dd.x, 1.0f / dd.y, 1.0f / dd.z);
  L.oi = mk(L.o.x * L.inv.x, L.o.y * L.inv.y, L.o.z * L.inv.z);
  L.tb = FLT_MAX;
  L.best = MISS_WORD;
  /* a ray with a NaN component misses at the root, as in the reference, where
   * both child entry distances come out None (aabb.rs:135-155,
   * bvh/hitable_trait.rs:43-46); without this the NaN-blind slab test below
   * would accept every box and walk the whole tree */
  const float chk = L.o.x + L.o.y + L.o.z + L.d.x + L.d.y + L.d.z;
  L.word = (chk == chk) ? root : CHILD_EMPTY;
  L.sp = 0;
  L.live = true;
}
__device__ __forceinline__ void lane_start(Lane &L, const PathBuf &pb, uint32_t path) {
  float4 o4 = pb.ray_o[path], d4 = pb.ray_d[path];
  lane_start_ray(L, xyz(o4), xyz(d4), d4.w, as_u(o4.w)); /* .w: the ray's root node, its job's scene in the arena */
  L.path = path;
}

__device__ __forceinline__ void lane_push(Lane &L, uint32_t w, uint32_t *lst, uint32_t *gst) {
  if (L.sp < STACK_LDS) lds_store(lst + (uint32_t)L.sp * TRACE_BLOCK, w);
  else if (L.sp < STACK_TOTAL) gst[L.sp - STACK_LDS] = w;
  else return; /* unreachable: the host bounds the BVH depth */
  L.sp++;
}

__device__ __forceinline__ void lane_pop(Lane &L, const uint32_t *lst, const uint32_t *gst) {
  if (L.sp == 0) { L.word = CHILD_EMPTY; return; }
  L.sp--;
  if (L.sp < STACK_LDS) L.word = lds_load(lst + (uint32_t)L.sp * TRACE_BLOCK);
  else L.word = gst[L.sp - STACK_LDS];
}

/* entry distance of the ray into each of a node's four child boxes (rows
 * 0-5 of the node at nf: lo/hi per axis, 4 children each), FLT_MAX where it
 * misses the box or the box starts beyond the closest hit so far.  The
 * conservative slab test of aabb.rs:54-155: entry clamped to the acne
 * epsilon, exit to just past the closest hit.  Both builders give an empty
 * child slot lo = FLT_MAX, hi = -FLT_MAX, which this test never enters (its
 * entry distance is at least FLT_MAX on every axis and its exit at most
 * -FLT_MAX), so it needs no check of the child word. */
__device__ __forceinline__ void slab4(const Lane &L, const float4 *nf, float tn[4]) {
  /* the near plane per axis is row lo (0, 2, 4) where the direction is
   * positive, hi (1, 3, 5) where it is negative, the far plane the other row
   * of the pair; rows picked by the signs give each axis's entry and exit
   * distances without a min/max pair per axis (a box has lo <= hi and the
   * multiply-add is monotone, so they are the same values) */
  const uint32_t rx = as_u(L.inv.x) >> 31, ry = 2u + (as_u(L.inv.y) >> 31), rz = 4u + (as_u(L.inv.z) >> 31);
  const float4 nx = nf[rx], fx = nf[rx ^ 1u], ny = nf[ry], fy = nf[ry ^ 1u], nz = nf[rz], fz = nf[rz ^ 1u];
  const float nxa[4] = {nx.x, nx.y, nx.z, nx.w}, fxa[4] = {fx.x, fx.y, fx.z, fx.w};
  const float nya[4] = {ny.x, ny.y, ny.z, ny.w}, fya[4] = {fy.x, fy.y, fy.z, fy.w};
  const float nza[4] = {nz.x, nz.y, nz.z, nz.w}, fza[4] = {fz.x, fz.y, fz.z, fz.w};
  const float tfar_lim = L.tb * 1.00000024f;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const float x0 = fmaf(nxa[k], L.inv.x, -L.oi.x), x1 = fmaf(fxa[k], L.inv.x, -L.oi.x);
    const float y0 = fmaf(nya[k], L.inv.y, -L.oi.y), y1 = fmaf(fya[k], L.inv.y, -L.oi.y);
    const float z0 = fmaf(nza[k], L.inv.z, -L.oi.z), z1 = fmaf(fza[k], L.inv.z, -L.oi.z);
    const float tnear = fmaxf(fmaxf(x0, y0), fmaxf(z0, EPS_ACNE));
    const float tfar = fminf(fminf(x1, y1), fminf(z1, tfar_lim));
    tn[k] = tnear <= tfar ? tnear : FLT_MAX;
  }
}

/* the same distances from all six rows with a min/max pair per axis, for
 * the traversals that read nodes from global memory: their six row loads
 * share one address (immediate offsets) and no per-lane row offsets stay in
 * registers; on the 1M-triangle mesh, whose traversal waits on node fetches,
 * the row-picked form was 1% slower */
template <class RAY>
__device__ __forceinline__ void slab4_minmax(const RAY &L, const float4 *nf, const uint32_t cw[4], float tn[4]) {
  const float4 lx = nf[0], hx = nf[1], ly = nf[2], hy = nf[3], lz = nf[4], hz = nf[5];
  const float lxa[4] = {lx.x, lx.y, lx.z, lx.w}, hxa[4] = {hx.x, hx.y, hx.z, hx.w};
  const float lya[4] = {ly.x, ly.y, ly.z, ly.w}, hya[4] = {hy.x, hy.y, hy.z, hy.w};
  const float lza[4] = {lz.x, lz.y, lz.z, lz.w}, hza[4] = {hz.x, hz.y, hz.z, hz.w};
  const float tfar_lim = L.tb * 1.00000024f;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const float x0 = fmaf(lxa[k], L.inv.x, -L.oi.x), x1 = fmaf(hxa[k], L.inv.x, -L.oi.x);
    const float y0 = fmaf(lya[k], L.inv.y, -L.oi.y), y1 = fmaf(hya[k], L.inv.y, -L.oi.y);
    const float z0 = fmaf(lza[k], L.inv.z, -L.oi.z), z1 = fmaf(hza[k], L.inv.z, -L.oi.z);
    const float tnear = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), EPS_ACNE));
    const float tfar = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), tfar_lim));
    const bool hit = (tnear <= tfar) && (cw[k] != CHILD_EMPTY);
    tn[k] = hit ? tnear : FLT_MAX;
  }
}

/* one interior node: test the four child boxes, continue with the nearest
 * hit child, push the others far-to-near */
__device__ __forceinline__ void lane_node(Lane &L, const DevScene &sc, uint32_t *lst, uint32_t *gst) {
  const Bvh4Node *nd = sc.nodes + L.word;
  const float4 *nf = reinterpret_cast<const float4 *>(nd);
  uint4 ch = reinterpret_cast<const uint4 *>(nd)[6];
  uint32_t cw[4] = {ch.x, ch.y, ch.z, ch.w};
  float tn[4];
  slab4_minmax(L, nf, cw, tn);
#define CSWAP(a, b)                                                       \
  {                                                                       \
    const bool s_ = tn[b] < tn[a];                                        \
    const float ta_ = tn[a], tb_ = tn[b];                                 \
    const uint32_t ca_ = cw[a], cb_ = cw[b];                              \
    tn[a] = s_ ? tb_ : ta_; tn[b] = s_ ? ta_ : tb_;                       \
    cw[a] = s_ ? cb_ : ca_; cw[b] = s_ ? ca_ : cb_;                       \
  }
  CSWAP(0, 1) CSWAP(2, 3) CSWAP(0, 2) CSWAP(1, 3) CSWAP(1, 2)
#undef CSWAP
#pragma unroll
  for (int k = 3; k >= 1; k--)
    if (tn[k] < FLT_MAX) lane_push(L, cw[k], lst, gst);
  if (tn[0] < FLT_MAX) L.word = cw[0];
  else lane_pop(L, lst, gst);
}

/* one leaf: test its primitives; every primitive keeps its own acceptance
 * rule against the current closest distance, as in the reference (inclusive
 * for quads and triangles, strict for spheres) */
__device__ __forceinline__ uint32_t lane_leaf(Lane &L, const DevScene &sc, bool any_xform) {
  uint32_t cnt = ((L.word >> 28) & 7u) + 1u;
  uint32_t off = L.word & LEAF_OFFSET_MASK;
  for (uint32_t k = 0; k < cnt; k++) {
    const float4 *rec = sc.prims + off;
    uint32_t hdr = as_u(rec[0].w);
    float t;
    bool h = any_xform ? test_prim<true>(sc, rec, hdr, L.o, L.d, L.time, EPS_ACNE, L.tb, t)
                       : test_prim<false>(sc, rec, hdr, L.o, L.d, L.time, EPS_ACNE, L.tb, t);
    if (h) {
      L.tb = t;
      L.best = off;
    }
    off += prim_units(hdr & PT_TYPE_MASK);
  }
  return cnt;
}

/* one primitive of the current leaf; the leaf word keeps the primitives left
 * (the same order as lane_leaf, so the same hits).  Returns true when the
 * leaf is done (the caller pops the stack).  One primitive per step keeps a
 * lane on a full leaf from holding up the lanes taking node steps. */
__device__ __forceinline__ bool lane_leaf_step(Lane &L, const DevScene &sc, bool any_xform) {
  const uint32_t cnt = ((L.word >> 28) & 7u) + 1u;
  const uint32_t off = L.word & LEAF_OFFSET_MASK;
  const float4 *rec = sc.prims + off;
  const uint32_t hdr = as_u(rec[0].w);
  float t;
  const bool h = any_xform ? test_prim<true>(sc, rec, hdr, L.o, L.d, L.time, EPS_ACNE, L.tb, t)
                           : test_prim<false>(sc, rec, hdr, L.o, L.d, L.time, EPS_ACNE, L.tb, t);
  if (h) {
    L.tb = t;
    L.best = off;
  }
  if (cnt == 1u) return true;
  L.word = (L.word & ~(LEAF_OFFSET_MASK | (7u << 28))) | ((cnt - 2u) << 28) | (off + prim_units(hdr & PT_TYPE_MASK));
  return false;
}

/* After the surface traversal: the job's constant media, each tested against
 * the closest surface so far (a medium's hit needs its boundary inside
 * [tmin, tmax], so the tree's box culling never changes its outcome, and its
 * uniform is keyed by the medium, so the order of the tests does not matter).
 * Only the traversal instance for batches with media runs this. */
__device__ __forceinline__ void lane_media(Lane &L, const DevScene &sc, uint32_t meta, uint64_t state) {
  const DevJob &jb = sc.jobs[meta >> META_JOB_SHIFT];
  if (jb.n_media == 0) return;
  uint32_t off = jb.media_off;
  for (uint32_t k = 0; k < jb.n_media; k++) {
    const float4 *rec = sc.prims + off;
    const uint32_t hdr = as_u(rec[0].w), xf = hdr >> PT_XF_SHIFT;
    V o = L.o, d = L.d;
    if (xf) xform_ray(sc.xforms[xf - 1u], o, d);
    float t;
    if (medium_t(sc, rec, o, d, EPS_ACNE, L.tb, state, t)) {
      L.tb = t;
      L.best = off;
    }
    off += as_u(rec[0].z);
  }
}

/* ------------------------------------------------------------ kernels --- */
/* before a bounce: count the rays about to be traced, clear the shading
 * queues and the next ray queue (a kernel, not a memset, so it can live in a
 * captured graph) */
__global__ void k_reset_counts(uint32_t *counts, uint32_t in_slot, uint32_t out_slot, unsigned long long *stats) {
  uint32_t i = threadIdx.x;
  if (i == 0) stats[2] += (unsigned long long)counts[in_slot];
  __syncthreads();
  if (i < MC_COUNT) counts[CNT_SHADE + i] = 0u;
  if (i == 0) counts[out_slot] = 0u;
  if (i == 1) counts[CNT_FETCH] = 0u;
}

__global__ void k_zero_u64(uint64_t *p, uint32_t n) {
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0ull;
}

__global__ void k_set_count(uint32_t *counts, uint32_t slot, uint32_t value) {
  if (threadIdx.x == 0 && blockIdx.x == 0) counts[slot] = value;
}

/* Device memory to pinned host memory, a chunk of COPY_CHUNK bytes a block: the
 * chunk's flag is raised behind its last store, so that the host takes it on
 * while the next ones are under way.  The link bounds it: 8 MB in 164 us,
 * 51 GB/s. */
#define CO_THREADS 256
__global__ __launch_bounds__(CO_THREADS) void k_copy_out(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst,
                                                         uint64_t words, uint32_t *flags, uint32_t stamp,
                                                         const uint64_t *stats, uint64_t *stats_out) {
  const uint64_t base = (uint64_t)blockIdx.x * (COPY_CHUNK / 4);
  const uint64_t end = base + COPY_CHUNK / 4 < words ? base + COPY_CHUNK / 4 : words;
  if (stats && blockIdx.x == 0 && threadIdx.x < 8) stats_out[threadIdx.x] = stats[threadIdx.x];
  if (end - base == COPY_CHUNK / 4) {
    const uint4 *s = reinterpret_cast<const uint4 *>(src + base);
    uint4 *d = reinterpret_cast<uint4 *>(dst + base);
    uint4 v[COPY_CHUNK / 16 / CO_THREADS];
#pragma unroll
    for (uint32_t k = 0; k < COPY_CHUNK / 16 / CO_THREADS; k++) v[k] = s[k * CO_THREADS + threadIdx.x];
#pragma unroll
    for (uint32_t k = 0; k < COPY_CHUNK / 16 / CO_THREADS; k++) d[k * CO_THREADS + threadIdx.x] = v[k];
  } else {
    for (uint64_t i = base + threadIdx.x; i < end; i += CO_THREADS) dst[i] = src[i];
  }
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(flags + blockIdx.x, stamp, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

/* index of the last entry of a table ordered by `key` whose key is <= v */
template <typename T>
__device__ __forceinline__ uint32_t find_entry(const T *tab, uint32_t n, uint32_t v, uint32_t T::*key) {
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1u) {
    uint32_t mid = (lo + hi) >> 1;
    if (tab[mid].*key <= v) lo = mid;
    else hi = mid;
  }
  return lo;
}

/* camera sample of sampler/random.rs:20-32 and Camera::get_ray (camera.rs:103-126);
 * path slot i belongs to the pass item whose range holds it */
/* row-major pixel index (row 0 = top) of the q-th slot of a sample in tile
 * order: bands of 8 rows top to bottom, 8x8 tiles left to right within a
 * band, row-major within a tile; the last band and the last tile of a band
 * are shorter / narrower when H or W is not a multiple of 8.  A bijection of
 * [0, W*H): a wave's 64 rays cover one tile instead of 64 pixels of a row. */
__device__ __forceinline__ uint32_t tile_pixel(uint32_t q, uint32_t W, uint32_t H) {
  const uint32_t band = q / (8u * W);
  const uint32_t q1 = q - band * 8u * W;
  const uint32_t hb = min(8u, H - 8u * band);
  const uint32_t tc = q1 / (8u * hb);
  const uint32_t q2 = q1 - tc * 8u * hb;
  const uint32_t tw = min(8u, W - 8u * tc);
  const uint32_t yi = q2 / tw;
  return (8u * band + yi) * W + 8u * tc + (q2 - yi * tw);
}

/* the camera sample of path slot i of a pass: its ray, the state of its
 * stream after the sampler's draws, and its meta word (depth 0) */
__device__ __forceinline__ uint32_t camera_sample(const DevScene &sc, const GenParams &gp, uint32_t i, V &org, V &dir,
                                                  float &time, uint64_t &s) {
  const DevItem it = gp.items[find_entry(gp.items, gp.n_items, i, &DevItem::path_base)];
  const DevJob &jb = sc.jobs[it.job];
  const uint32_t W = jb.width, H = jb.height;
  uint32_t k = i - it.path_base;
  uint32_t j = k / it.pixels, o = k - j * it.pixels;
  if (it.order) o = tile_pixel(o, W, H);
  uint32_t r = o / W, x = o - r * W;
  uint32_t y = H - 1u - r;
  uint32_t sample = it.sample_base + j;
  s = pcg_for_path(jb.seed, x + y * W, sample);
  float ox = rnd(s), oy = rnd(s);
  float lx, ly;
  for (;;) {
    lx = rnd_pm1(s);
    ly = rnd_pm1(s);
    if (lx * lx + ly * ly <= 1.0f) break;
  }
  time = rnd(s); /* the ray's instant (sampler/random.rs:23); carried in ray_d.w */
  uint32_t wl = (uint32_t)(((uint64_t)pcg_next(s) * 400ull) >> 32);
  float u = ((float)x + ox) / (float)W;
  float v = ((float)y + oy) / (float)H;
  const DevCamera &c = jb.cam;
  lx *= c.lens_radius;
  ly *= c.lens_radius;
  V cu = mk(c.u[0], c.u[1], c.u[2]), cv = mk(c.v[0], c.v[1], c.v[2]);
  V off = lx * cu + ly * cv;
  org = mk(c.origin[0], c.origin[1], c.origin[2]);
  dir = mk(c.llc[0], c.llc[1], c.llc[2]) + u * mk(c.horizontal[0], c.horizontal[1], c.horizontal[2]) +
        v * mk(c.vertical[0], c.vertical[1], c.vertical[2]) - org - off;
  dir = unit(dir);
  org = org + off;
  return wl | (it.job << META_JOB_SHIFT);
}

__global__ __launch_bounds__(256) void k_generate(DevScene sc, PathBuf pb, GenParams gp) {
  uint32_t n = gp.paths;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    V org, dir;
    float time;
    uint64_t s;
    const uint32_t meta = camera_sample(sc, gp, i, org, dir, time, s);
    const uint32_t root = sc.jobs[meta >> META_JOB_SHIFT].root;
    /* slot i is entry i of the first bounce */
    pb.ray_o[i] = make_float4(org.x, org.y, org.z, __uint_as_float(root));
    pb.ray_d[i] = make_float4(dir.x, dir.y, dir.z, time);
    pb.thr[i] = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    pb.rng[i] = s;
    pb.meta[i] = meta;
    pb.slot[i] = i;
    pb.rad[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    pb.hero[i] = meta & META_HERO_MASK;
    if (pb.gcnt) {
      pb.gcnt[i] = 0u;
#pragma unroll
      for (uint32_t k = 0; k < GD_SLOTS; k++) pb.recL[(size_t)i * GD_SLOTS + k] = 0.0f;
    }
  }
}

/* ------------------------------------------- LDS-cached traversal --- */
/* The same one-ray-per-thread traversal, with the top of the scene in LDS.
 * Incoherent rays make every lane's node load hit a different cache line, and
 * the vector-memory pipeline serialises such loads; LDS serves them at
 * bank speed.  Each block copies the first `lds_nodes` wide nodes (the tree
 * is numbered breadth-first, so this is its top) and the first `lds_units`
 * float4 of primitive records into LDS, then traverses.  768-thread blocks
 * (12 waves) amortise the copy; the per-lane stack keeps 8 entries in LDS
 * and the rest in a global per-thread slice. */
#define LT_BLOCK 768
#define LT_STACK_LDS 8
#define LT_STACK_GLOBAL (STACK_TOTAL - LT_STACK_LDS)

template <int BLOCK, int DEPTH>
struct LStack {
  uint32_t *lst;   /* LDS: DEPTH entries per lane, stride BLOCK */
  uint32_t *gst;   /* global slice: the entries from DEPTH on */
  __device__ __forceinline__ void push(Lane &L, uint32_t w) const {
    if (L.sp < DEPTH) lds_store(lst + (uint32_t)L.sp * BLOCK, w);
    else if (L.sp < STACK_TOTAL) gst[L.sp - DEPTH] = w;
    else return; /* unreachable: the host bounds the BVH depth */
    L.sp++;
  }
  __device__ __forceinline__ void pop(Lane &L) const {
    if (L.sp == 0) { L.word = CHILD_EMPTY; return; }
    L.sp--;
    if (L.sp < DEPTH) L.word = lds_load(lst + (uint32_t)L.sp * BLOCK);
    else L.word = gst[L.sp - DEPTH];
  }
};

/* one interior node whose 8 float4 start at nf (LDS or global) */
template <class STACK>
__device__ __forceinline__ void lnode_at(Lane &L, const float4 *nf, const STACK &S) {
  float4 cf = nf[6];
  uint32_t cw[4] = {as_u(cf.x), as_u(cf.y), as_u(cf.z), as_u(cf.w)};
  float tn[4];
  slab4(L, nf, tn);
#define CSWAP(a, b)                                                       \
  {                                                                       \
    const bool s_ = tn[b] < tn[a];                                        \
    const float ta_ = tn[a], tb_ = tn[b];                                 \
    const uint32_t ca_ = cw[a], cb_ = cw[b];                              \
    tn[a] = s_ ? tb_ : ta_; tn[b] = s_ ? ta_ : tb_;                       \
    cw[a] = s_ ? cb_ : ca_; cw[b] = s_ ? ca_ : cb_;                       \
  }
  CSWAP(0, 1) CSWAP(2, 3) CSWAP(0, 2) CSWAP(1, 3) CSWAP(1, 2)
#undef CSWAP
#pragma unroll
  for (int k = 3; k >= 1; k--)
    if (tn[k] < FLT_MAX) S.push(L, cw[k]);
  if (tn[0] < FLT_MAX) L.word = cw[0];
  else S.pop(L);
}

/* one primitive record at rec (LDS or global) */
__device__ __forceinline__ void lprim_at(Lane &L, const DevScene &sc, const float4 *rec, uint32_t off, bool any_xform,
                                         uint32_t &units) {
  uint32_t hdr = as_u(rec[0].w);
  float t;
  bool h = any_xform ? test_prim<true>(sc, rec, hdr, L.o, L.d, L.time, EPS_ACNE, L.tb, t)
                     : test_prim<false>(sc, rec, hdr, L.o, L.d, L.time, EPS_ACNE, L.tb, t);
  if (h) {
    L.tb = t;
    L.best = off;
  }
  units = prim_units(hdr & PT_TYPE_MASK);
}

/* the part of the scene a block keeps in LDS */
struct LdsWindow {
  const float4 *nodes, *prims;
  uint32_t nn, nb;   /* nodes [nb, nb + nn) */
  uint32_t nu, ub;   /* primitive units [ub, ub + nu) */
};

/* a lane's whole traversal */
template <bool COUNT, class STACK>
__device__ __forceinline__ void lds_traverse(Lane &L, const DevScene &sc, const LdsWindow &w, const STACK &S,
                                             bool any_xform, uint32_t &nvisit, uint32_t &ntest) {
  while (L.word != CHILD_EMPTY) {
    if (!(L.word & CHILD_LEAF)) {
      const uint32_t rel = L.word - w.nb; /* wraps above nn for nodes below the window */
      if (rel < w.nn) lnode_at(L, w.nodes + rel * 8u, S);
      else lnode_at(L, reinterpret_cast<const float4 *>(sc.nodes + L.word), S);
      if (COUNT) nvisit++;
    } else {
      /* one primitive per step: a lane on a leaf of 8 does not hold up the
       * lanes taking node steps; the leaf word keeps the primitives left
       * (the same order, so the same hits) */
      const uint32_t cnt = ((L.word >> 28) & 7u) + 1u;
      const uint32_t off = L.word & LEAF_OFFSET_MASK;
      uint32_t units;
      if (off >= w.ub && off + PREC_QUAD <= w.ub + w.nu)
        lprim_at(L, sc, w.prims + (off - w.ub), off, any_xform, units);
      else
        lprim_at(L, sc, sc.prims + off, off, any_xform, units);
      if (COUNT) ntest++;
      if (cnt > 1u) L.word = (L.word & ~(LEAF_OFFSET_MASK | (7u << 28))) | ((cnt - 2u) << 28) | (off + units);
      else S.pop(L);
    }
  }
}

template <bool COUNT, int MODE>
__global__ __launch_bounds__(LT_BLOCK) void k_trace_lds(DevScene sc, PathBuf pb, TraceArgs ta) {
  extern __shared__ float4 smem[];
  const uint32_t nn = ta.lds_nodes, nu = ta.lds_units, nb = ta.lds_node_base, ub = ta.lds_unit_base;
  float4 *cnodes = smem;
  float4 *cprims = smem + nn * 8u;
  const LdsWindow win = {cnodes, cprims, nn, nb, nu, ub};
  LStack<LT_BLOCK, LT_STACK_LDS> S;
  S.lst = reinterpret_cast<uint32_t *>(cprims + nu) + threadIdx.x;
  S.gst = ta.spill + (size_t)(blockIdx.x * LT_BLOCK + threadIdx.x) * LT_STACK_GLOBAL;
  {
    const float4 *gn = reinterpret_cast<const float4 *>(sc.nodes + nb);
    for (uint32_t k = threadIdx.x; k < nn * 8u; k += LT_BLOCK) cnodes[k] = gn[k];
    for (uint32_t k = threadIdx.x; k < nu; k += LT_BLOCK) cprims[k] = sc.prims[ub + k];
  }
  __syncthreads();
  __shared__ uint32_t agg[MC_COUNT * (LT_BLOCK / 64) + MC_COUNT];
  const uint32_t n = MODE == 0 ? ta.counts[ta.in_slot] : ta.n_direct;
  const bool any_xform = sc.has_xforms != 0;
  uint32_t nvisit = 0, ntest = 0;
  for (uint32_t base = blockIdx.x * LT_BLOCK; base < n; base += gridDim.x * LT_BLOCK) {
    const uint32_t i = base + threadIdx.x;
    const bool active = i < n;
    Lane L;
    L.live = false;
    L.best = MISS_WORD;
    L.path = 0;
    if (active) lane_start(L, pb, i);
    else L.word = CHILD_EMPTY;
    lds_traverse<COUNT>(L, sc, win, S, any_xform, nvisit, ntest);
    if (MODE == 0) {
      uint32_t cls = MC_COUNT;
      if (active) {
        pb.hit_t[L.path] = L.tb;
        pb.hit_p[L.path] = L.best;
        cls = L.best != MISS_WORD ? sc.mats[sc.info[as_u(sc.prims[L.best + 1u].w)].material].mclass : MC_MISS;
      }
      block_append<MC_COUNT, LT_BLOCK>(cls, L.path, ta.sq.q, ta.sq.counts, agg);
    } else if (active) {
      if (L.best == MISS_WORD) {
        ta.ids[L.path] = 0xFFFFFFFFu;
        ta.ts[L.path] = INFINITY;
      } else {
        ta.ids[L.path] = sc.info[as_u(sc.prims[L.best + 1u].w)].report_id;
        ta.ts[L.path] = L.tb;
      }
    }
  }
  if (COUNT) {
    atomicAdd(ta.stats + 0, (unsigned long long)nvisit);
    atomicAdd(ta.stats + 1, (unsigned long long)ntest);
  }
}

/* Closest-hit kernel, one ray per thread: the block's threads take rays
 * base + threadIdx.x in a grid-stride loop; each thread runs its ray to
 * completion (node or leaf per step).  Results as in k_trace below. */
/* ORDER: a node or a primitive per lane and turn; while-while; or, for guided
 * bounces in scenes that are not in LDS, a turn of nodes or of primitives, by
 * what most lanes have (uneven batch of 6 scenes 14.3 ms; 15.2 with both each
 * turn, 17.8 through the LDS window of its largest job's scene) */
#define ORDER_BOTH 0
#define ORDER_WW 1
#define ORDER_MAJORITY 2
/* MEDIA: the instance for batches with constant media (the media pass after
 * the tree raises the traversal's registers, so the other instances leave it
 * out; batches with media always trace with this kernel) */
template <bool COUNT, int MODE, int ORDER, bool MEDIA = false>
/* 7 waves per SIMD for the rendering instances: the traversal waits on
 * dependent node fetches, and 72 VGPRs (a few spilled outside the node loop)
 * let 7 waves hide that latency instead of the 6 that 76 VGPRs allow */
__global__ __launch_bounds__(TRACE_BLOCK) __attribute__((amdgpu_waves_per_eu((COUNT || MEDIA) ? 1 : 8))) void k_trace_simple(DevScene sc, PathBuf pb, TraceArgs ta) {
  __shared__ uint32_t lds_stack[STACK_LDS * TRACE_BLOCK];
  __shared__ uint32_t agg[MC_COUNT * (TRACE_BLOCK / 64) + MC_COUNT];
  const uint32_t n = MODE == 0 ? ta.counts[ta.in_slot] : ta.n_direct;
  uint32_t *lst = lds_stack + threadIdx.x;
  uint32_t *gst = ta.spill + (size_t)(blockIdx.x * TRACE_BLOCK + threadIdx.x) * STACK_GLOBAL;
  const bool any_xform = sc.has_xforms != 0;
  uint32_t nvisit = 0, ntest = 0;
  for (uint32_t base = blockIdx.x * TRACE_BLOCK; base < n; base += gridDim.x * TRACE_BLOCK) {
    const uint32_t i = base + threadIdx.x;
    const bool active = i < n;
    Lane L;
    L.live = false;
    L.best = MISS_WORD;
    L.path = 0;
    if (active) lane_start(L, pb, i);
    else L.word = CHILD_EMPTY;
    const uint32_t v0 = nvisit, t0 = ntest;
    if (ORDER == ORDER_WW) {
      /* while-while: the wave descends interior nodes until every lane holds
       * a leaf (or is done), then all lanes test their leaf together */
      while (__any(L.word != CHILD_EMPTY)) {
        while (__any(!(L.word & CHILD_LEAF))) {
          if (!(L.word & CHILD_LEAF)) {
            lane_node(L, sc, lst, gst);
            if (COUNT) nvisit++;
          }
        }
        if (L.word != CHILD_EMPTY) {
          uint32_t c = lane_leaf(L, sc, any_xform);
          if (COUNT) ntest += c;
          lane_pop(L, lst, gst);
        }
      }
    } else if (ORDER == ORDER_MAJORITY) {
      for (;;) {
        const bool leaf = L.word >= CHILD_LEAF && L.word != CHILD_EMPTY, node = L.word < CHILD_LEAF;
        const uint32_t nn = (uint32_t)__popcll(__ballot(node)), nl = (uint32_t)__popcll(__ballot(leaf));
        if (nn + nl == 0u) break;
        if (nn >= nl) {
          if (node) lane_node(L, sc, lst, gst);
        } else if (leaf) {
          if (lane_leaf_step(L, sc, any_xform)) lane_pop(L, lst, gst);
        }
      }
    } else {
      while (L.word != CHILD_EMPTY) {
        if (!(L.word & CHILD_LEAF)) {
          lane_node(L, sc, lst, gst);
          if (COUNT) nvisit++;
        } else {
          if (COUNT) ntest++;
          if (lane_leaf_step(L, sc, any_xform)) lane_pop(L, lst, gst);
        }
      }
    }
    if (MEDIA && active) lane_media(L, sc, pb.meta[L.path], pb.rng[L.path]);
    if (MODE == 0) {
      uint32_t cls = MC_COUNT;
      if (active) {
        pb.hit_t[L.path] = L.tb;
        pb.hit_p[L.path] = L.best;
        cls = L.best != MISS_WORD ? sc.mats[sc.info[as_u(sc.prims[L.best + 1u].w)].material].mclass : MC_MISS;
      }
      block_append<MC_COUNT, TRACE_BLOCK>(cls, L.path, ta.sq.q, ta.sq.counts, agg);
    } else if (active) {
      if (L.best == MISS_WORD) {
        ta.ids[L.path] = 0xFFFFFFFFu;
        ta.ts[L.path] = INFINITY;
      } else {
        ta.ids[L.path] = sc.info[as_u(sc.prims[L.best + 1u].w)].report_id;
        ta.ts[L.path] = L.tb;
      }
      pb.hit_t[L.path] = L.tb;
      pb.hit_p[L.path] = L.best;
      if (COUNT && ta.ray_counts) {
        ta.ray_counts[2u * L.path] = nvisit - v0;
        ta.ray_counts[2u * L.path + 1u] = ntest - t0;
      }
    }
  }
  if (COUNT) {
    atomicAdd(ta.stats + 0, (unsigned long long)nvisit);
    atomicAdd(ta.stats + 1, (unsigned long long)ntest);
  }
}

/* Persistent closest-hit kernel.  Each wave keeps 64 rays in flight; a lane
 * whose ray is finished takes the next one from the queue (one atomic per
 * wave per refill), so waves stay full through the tail of a bounce.  Each
 * iteration descends interior nodes until every lane holds a leaf
 * (while-while), then tests one leaf per lane.  Finished rays are written out
 * and, in the extend mode, appended to the shading queue of their material
 * class with wave-aggregated atomics.
 *   MODE_EXTEND:  rays are entries 0 .. counts[in_slot] of the path state
 *   MODE_PRIMARY: rays are paths 0 .. n_direct, results go to ids/ts */
#define MODE_EXTEND 0
#define MODE_PRIMARY 1

template <bool COUNT, int MODE>
__global__ __launch_bounds__(TRACE_BLOCK) void k_trace(DevScene sc, PathBuf pb, TraceArgs ta) {
  __shared__ uint32_t lds_stack[STACK_LDS * TRACE_BLOCK];
  const uint32_t n = MODE == MODE_EXTEND ? ta.counts[ta.in_slot] : ta.n_direct;
  const uint32_t lane = __lane_id();
  const uint64_t lt_mask = (1ull << lane) - 1ull;
  uint32_t *lst = lds_stack + threadIdx.x;
  uint32_t *gst = ta.spill + (size_t)(blockIdx.x * TRACE_BLOCK + threadIdx.x) * STACK_GLOBAL;
  const bool any_xform = sc.has_xforms != 0;
  uint32_t nvisit = 0, ntest = 0;
  bool exhausted = false;
  Lane L;
  L.live = false;
  L.word = CHILD_EMPTY;
  L.path = 0;
  L.sp = 0;
  L.tb = FLT_MAX;
  L.best = MISS_WORD;
  for (;;) {
    if (!exhausted) {
      uint64_t idle = __ballot(!L.live);
      if (idle) {
        uint32_t leader = (uint32_t)__ffsll((unsigned long long)idle) - 1u;
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(ta.counts + CNT_FETCH, (uint32_t)__popcll(idle));
        base = __shfl(base, (int)leader);
        if (base >= n) exhausted = true;
        if (!L.live) {
          uint32_t idx = base + (uint32_t)__popcll(idle & lt_mask);
          if (idx < n) lane_start(L, pb, idx);
        }
      }
    }
    if (!__any(L.live)) {
      if (exhausted) break;
      continue;
    }
    /* descend interior nodes until every live lane holds a leaf or is done */
    while (__any(L.live && !(L.word & CHILD_LEAF))) {
      if (L.live && !(L.word & CHILD_LEAF)) {
        lane_node(L, sc, lst, gst);
        if (COUNT) nvisit++;
      }
    }
    if (L.live && L.word != CHILD_EMPTY) {
      uint32_t c = lane_leaf(L, sc, any_xform);
      if (COUNT) ntest += c;
      lane_pop(L, lst, gst);
    }
    const bool fin = L.live && L.word == CHILD_EMPTY;
    if (MODE == MODE_EXTEND) {
      uint32_t cls = MC_MISS;
      if (fin) {
        pb.hit_t[L.path] = L.tb;
        pb.hit_p[L.path] = L.best;
        if (L.best != MISS_WORD) cls = sc.mats[sc.info[as_u(sc.prims[L.best + 1u].w)].material].mclass;
      }
#pragma unroll
      for (uint32_t c = 0; c < MC_COUNT; c++) wave_append(fin && cls == c, L.path, ta.sq.q[c], ta.sq.counts + c);
    } else if (fin) {
      if (L.best == MISS_WORD) {
        ta.ids[L.path] = 0xFFFFFFFFu;
        ta.ts[L.path] = INFINITY;
      } else {
        ta.ids[L.path] = sc.info[as_u(sc.prims[L.best + 1u].w)].report_id;
        ta.ts[L.path] = L.tb;
      }
    }
    if (fin) L.live = false;
  }
  if (COUNT) {
    atomicAdd(ta.stats + 0, (unsigned long long)nvisit);
    atomicAdd(ta.stats + 1, (unsigned long long)ntest);
  }
}

/* ------------------------------------------------------------ shading --- */
struct Hit {
  V p, n;       /* position, normal oriented against the ray */
  bool front;
  uint32_t material;
  float u, v;   /* surface coordinates (only for surface-checker materials) */
};

/* Sphere::get_uv (sphere.rs:58-65), MovingSphere::get_uv (moving_sphere.rs:93-101) */
__device__ __forceinline__ void sphere_uv(V p, V c, float r, float &u, float &v) {
  V t = (p - c) / r;
  float phi = atan2f(t.z, t.x);
  float theta = asinf(t.y);
  u = 1.0f - (phi + PI_F) / (2.0f * PI_F);
  v = (theta + PI_F / 2.0f) / PI_F;
}

/* Reconstruct the reference's HitRecord for the hit primitive: run the wrapper
 * chain forward, evaluate the primitive's record, then unwind RotateY
 * (rotate.rs:115-158: rotate back, set_face_normal with the rotated ray) and
 * Translate (translate.rs:68-77: shift back, set_face_normal with the moved ray). */
template <bool UV, bool XF = true>
__device__ Hit hit_record(const DevScene &sc, uint32_t off, V o, V d, float time, float t) {
  const float4 *rec = sc.prims + off;
  float4 f0 = rec[0], f1 = rec[1];
  uint32_t hdr = as_u(f0.w), type = hdr & PT_TYPE_MASK, xf = XF ? hdr >> PT_XF_SHIFT : 0u;
  Hit h;
  h.material = sc.info[as_u(f1.w)].material;
  h.u = h.v = 0.0f;
  V dirs[4];
  uint32_t nops = 0;
  const Xform *x = sc.xforms;
  if (xf) {
    x = &sc.xforms[xf - 1u];
    nops = x->n_ops;
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) {
      if (k < nops) {
        const XformOp &op = x->ops[k];
        if (op.kind == XF_TRANSLATE) {
          o = o - mk(op.a, op.b, op.c);
        } else {
          float s = op.a, c = op.b;
          o = mk(c * o.x - s * o.z, o.y, s * o.x + c * o.z);
          d = unit(mk(c * d.x - s * d.z, d.y, s * d.x + c * d.z));
        }
      }
      dirs[k] = d;
    }
  }
  V p = o + t * d;
  V outward;
  const bool want_uv = UV && sc.mats[h.material].tex == TX_SURFACE;
  if (type == PT_MEDIUM) {
    /* the reference gives a medium hit a random unit normal and front_face = true
     * (constant_medium.rs:108-109); nothing reads them for an Isotropic phase
     * function, so a fixed one is used and the stream is not drawn from */
    outward = -unit(d);
  } else if (type == PT_SPHERE || type == PT_MSPHERE) {
    V c = type == PT_SPHERE ? xyz(f0) : xyz(f0) + time * xyz(rec[2]);
    outward = unit((p - c) / f1.x);
    if (want_uv) sphere_uv(p, c, f1.x, h.u, h.v);
  } else {
    outward = xyz(rec[3]);
    if (want_uv) {
      /* (u, v) = the plane coordinates (alpha, beta) of quad.rs:108-128 / triangle.rs:143-160 */
      const V q = xyz(f0), eu = xyz(f1), ev = xyz(rec[2]), w = xyz(rec[4]);
      V ph = p - q;
      h.u = dot(w, cross(ph, ev));
      h.v = dot(w, cross(eu, ph));
    }
  }
  bool front = dot(d, outward) < 0.0f;
  V n = front ? outward : -outward;
#pragma unroll
  for (int k = 3; k >= 0; k--) {
    if (k < (int)nops) {
      const XformOp &op = x->ops[k];
      if (op.kind == XF_TRANSLATE) {
        p = p + mk(op.a, op.b, op.c);
      } else {
        float s = op.a, c = op.b;
        p = mk(c * p.x + s * p.z, p.y, -s * p.x + c * p.z);
        n = unit(mk(c * n.x + s * n.z, n.y, -s * n.x + c * n.z));
      }
      front = dot(dirs[k], n) < 0.0f;
      n = front ? n : -n;
    }
  }
  h.p = p;
  h.n = n;
  h.front = front;
  return h;
}

__device__ __forceinline__ V reflect(V v, V n) { return unit(v - 2.0f * dot(v, n) * n); }
__device__ __forceinline__ V refract(V v, V n, float ratio) {
  float ct = fminf(-dot(v, n), 1.0f);
  V par = ratio * (v + ct * n);
  V perp = -sqrtf(1.0f - dot(par, par)) * n;
  return unit(par + perp);
}
__device__ __forceinline__ float schlick(float cosine, float idx) {
  float r0 = (1.0f - idx) / (1.0f + idx);
  r0 = r0 * r0;
  return r0 + (1.0f - r0) * powf(1.0f - cosine, 5.0f);
}
/* ThinFilm::interference (thin_film.rs:31-54) */
__device__ __forceinline__ float interference(const DevMaterial &m, V d, V n, int wl) {
  float n_ratio = 1.0f / m.film_ior;
  float c1 = -dot(d, n);
  float s1 = sqrtf(1.0f - c1 * c1);
  float s2 = n_ratio * s1;
  float c2 = sqrtf(1.0f - (s2 * s2));
  float opd = 2.0f * m.film_ior * m.film_thickness * c2;
  float mm = opd / (float)wl;
  return 1.0f + cosf(mm * 2.0f * PI_F);
}

/* ONB::build_from_w (onb.rs:23-40) */
struct Onb {
  V u, v, w;
};
__device__ __forceinline__ Onb onb_from_w(V w) {
  V a = fabsf(w.x) > 0.9f ? mk(0.0f, 1.0f, 0.0f) : mk(1.0f, 0.0f, 0.0f);
  Onb b;
  b.v = unit(cross(w, a));
  b.u = unit(cross(w, b.v));
  b.w = w;
  return b;
}
__device__ __forceinline__ V onb_local(const Onb &b, V a) { return unit(a.x * b.u + a.y * b.v + a.z * b.w); }

/* UnitSphere (Marsaglia 1972), as random_unit_vector (random.rs:11-15) */
__device__ __forceinline__ V random_unit_vector(uint64_t &s) {
  for (;;) {
    float x1 = rnd_pm1(s), x2 = rnd_pm1(s);
    float sum = x1 * x1 + x2 * x2;
    if (sum >= 1.0f) continue;
    float f = 2.0f * sqrtf(1.0f - sum);
    return unit(mk(x1 * f, x2 * f, 1.0f - 2.0f * sum));
  }
}

/* light pdf of one MIS leaf (quad.rs:140-165, triangle.rs:176-201, sphere.rs:133-158) */
__device__ float light_pdf(const DevLight &L, V o, V d) {
  if (L.type == PT_SPHERE) {
    V c = mk(L.q[0], L.q[1], L.q[2]);
    float r = L.u[0];
    float t;
    if (!sphere_t(c, r, o, d, EPS_ACNE, INFINITY, t)) return 0.0f;
    V oc = c - o;
    float ctm = sqrtf(1.0f - r * r / dot(oc, oc));
    float solid = 2.0f * PI_F * (1.0f - ctm);
    return 1.0f / solid;
  }
  V q = mk(L.q[0], L.q[1], L.q[2]), u = mk(L.u[0], L.u[1], L.u[2]), v = mk(L.v[0], L.v[1], L.v[2]);
  V n = mk(L.n[0], L.n[1], L.n[2]), w = mk(L.w[0], L.w[1], L.w[2]);
  float denom = dot(n, d);
  if (fabsf(denom) < EPS_RECT) return 0.0f;
  float t = (-L.n[3] - dot(n, o)) / denom;
  if (t < EPS_ACNE || t > INFINITY) return 0.0f;
  V p = o + t * d;
  V ph = p - q;
  float alpha = dot(w, cross(ph, v));
  float beta = dot(w, cross(u, ph));
  bool in = alpha >= 0.0f && alpha <= 1.0f && beta >= 0.0f && beta <= 1.0f;
  if (L.type == PT_TRI) in = in && (alpha + beta <= 1.0f);
  if (!in) return 0.0f;
  float dist2 = t * t * dot(d, d);
  float cosine = fabsf(dot(d, n)) / sqrtf(dot(d, d)); /* |d . oriented normal| */
  return dist2 / (cosine * L.w[3]);
}

/* random point / direction towards one MIS leaf (quad.rs:168-172, triangle.rs:204-220, sphere.rs:160-187) */
__device__ V light_sample(const DevLight &L, V o, uint64_t &s) {
  if (L.type == PT_SPHERE) {
    V c = mk(L.q[0], L.q[1], L.q[2]);
    float r = L.u[0];
    V off = c - o;
    float dist2 = dot(off, off);
    Onb b = onb_from_w(unit(off));
    float r1 = rnd(s), r2 = rnd(s);
    float z = 1.0f + r2 * (sqrtf(1.0f - r * r / dist2) - 1.0f);
    float phi = 2.0f * PI_F * r1;
    float x = cosf(phi) * sqrtf(1.0f - z * z);
    float y = sinf(phi) * sqrtf(1.0f - z * z);
    return onb_local(b, unit(mk(x, y, z)));
  }
  float a = rnd(s), bb = rnd(s);
  if (L.type == PT_TRI && a + bb > 1.0f) {
    a = 1.0f - a;
    bb = 1.0f - bb;
  }
  V q = mk(L.q[0], L.q[1], L.q[2]), u = mk(L.u[0], L.u[1], L.u[2]), v = mk(L.v[0], L.v[1], L.v[2]);
  V point = q + (a * u) + (bb * v);
  return point - o;
}

/* HitablePDF over the MIS tree: sampling descends with a fair coin wherever
 * both children exist (bvh/hitable_trait.rs:113-127); the pdf is the
 * 2^-depth weighted sum over leaves, i.e. the nested midpoints of :89-111. */
__device__ V tree_sample(const DevScene &sc, const DevJob &jb, V o, uint64_t &s) {
  uint32_t w = jb.light_root;
  while (!(w & LT_LEAF)) {
    const DevLightNode &nd = sc.lnodes[w];
    if (nd.child[1] == LT_EMPTY) w = nd.child[0];
    else if (nd.child[0] == LT_EMPTY) w = nd.child[1];
    else w = coin(s) ? nd.child[0] : nd.child[1];
  }
  return light_sample(sc.lights[w & ~LT_LEAF], o, s);
}
__device__ float tree_pdf(const DevScene &sc, const DevJob &jb, V o, V d) {
  float p = 0.0f;
  for (uint32_t l = jb.light_base; l < jb.light_base + jb.n_lights; l++) {
    float w = sc.lweights[l];
    if (w > 0.0f) p += w * light_pdf(sc.lights[l], o, d);
  }
  return p;
}

/* the SPD a hit reads from a material's texture: the plain table, or a
 * checker's even/odd cell table (spatial_checker.rs:74-88 by world position,
 * surface_checker.rs:72-84 by surface coordinates) */
__device__ __forceinline__ int32_t tex_spd(const DevMaterial &m, int32_t even, const Hit &h) {
  if (m.tex == TX_PLAIN) return even;
  const float k = m.density_pi;
  const float sines = m.tex == TX_SPATIAL ? sinf(k * h.p.x) * sinf(k * h.p.y) * sinf(k * h.p.z)
                                          : sinf(k * h.u) * sinf(k * h.v);
  return sines < 0.0f ? m.odd_spd : even;
}

__device__ __forceinline__ void rotate_wl(uint32_t hero_idx, int wl[4]) {
#pragma unroll
  for (int j = 0; j < 4; j++) wl[j] = CLV_LAMBDA_MIN + (int)((hero_idx + 100u * (uint32_t)j) % 400u);
}

/* a radiance sample c0 (hero wavelength, already times the path throughput)
 * reached the path: credit it to the path's open training records, each as
 * c0 / (throughput right after that vertex) = radiance along its direction */
#define GD_SPECULAR 0x80000000u /* gcnt flag: a specular vertex since the latest record */
__device__ __forceinline__ void gd_credit(const PathBuf &pb, const GuideArgs &ga, uint32_t slot, float c0) {
  if (!(c0 > 0.0f)) return;
  const uint32_t g = pb.gcnt[slot], cnt = g & ~GD_SPECULAR;
  const uint32_t m = cnt < GD_SLOTS ? cnt : GD_SLOTS;
  for (uint32_t k = (ga.indirect && !(g & GD_SPECULAR)) ? 1u : 0u; k < m; k++) {
    const size_t j = (size_t)slot * GD_SLOTS + ((cnt - 1u - k) % GD_SLOTS);
    const float t0 = ga.rec[j].t0;
    if (t0 > 0.0f) pb.recL[j] += c0 / t0;
  }
}

/* the state a surviving path carries into the next bounce */
struct NextPath {
  float4 o, d, thr;
  uint64_t rng;
  uint32_t meta, slot;
};

/* a hit position normalised to the job's scene box ([-1, 1]^3): the guiding
 * network's input and the gate's cell coordinates */
__device__ __forceinline__ void gd_norm_pos(const DevJob &jb, V p, float out[3]) {
  out[0] = 2.0f * (p.x - jb.lo[0]) / (jb.hi[0] - jb.lo[0]) - 1.0f;
  out[1] = 2.0f * (p.y - jb.lo[1]) / (jb.hi[1] - jb.lo[1]) - 1.0f;
  out[2] = 2.0f * (p.z - jb.lo[2]) / (jb.hi[2] - jb.lo[2]) - 1.0f;
}
/* the gate is open at the vertex the entry's ray reaches, o + t d (GuideArgs.gate
 * NULL: everywhere).  The point is the ray's, not the hit record's, so the
 * inference kernel decides without reconstructing the hit; the shading kernel
 * decides from the same entry with the same operations, so they agree. */
__device__ __forceinline__ bool gd_gate_open(const GuideArgs &ga, const DevJob &jb, uint32_t job, float4 o4, float4 d4,
                                             float t) {
  if (!ga.gate) return true;
  const V p = xyz(o4) + t * xyz(d4);
  float pn[3];
  gd_norm_pos(jb, p, pn);
  return ga.gate[(size_t)job * GD_CELLS + gd_cell(pn)] != 0;
}

/* the scattered direction at a metal (metal.rs:26-52) or glass vertex
 * (dielectric.rs:35-70, dispersive.rs:68-115: the index at the hero
 * wavelength), drawing from the path's stream */
template <bool METAL>
__device__ __forceinline__ V specular_dir(const DevMaterial &m, V d, const Hit &h, uint32_t hero_idx, uint64_t &s) {
  if (METAL) {
    V r = reflect(d, h.n);
    return unit(r + m.fuzz * random_unit_vector(s));
  }
  float n_ior;
  if (m.kind == CLV_MAT_DISPERSIVE) {
    float wm = (float)(CLV_LAMBDA_MIN + (int)hero_idx) / 1000.0f;
    n_ior = m.cauchy_a + (m.cauchy_b / (wm * wm));
  } else {
    n_ior = m.ior;
  }
  float ratio = h.front ? 1.0f / n_ior : n_ior;
  float ct = fminf(-dot(d, h.n), 1.0f);
  float st = sqrtf(1.0f - ct * ct);
  if (ratio * st > 1.0f) return reflect(d, h.n);
  float rp = schlick(ct, ratio);
  return (rnd(s) < rp) ? reflect(d, h.n) : refract(d, h.n, ratio);
}

/* what shading reads of a path and of the hit of its ray */
struct ShadeIn {
  float4 o4, d4;     /* as in PathBuf: .w = root node; the ray's instant */
  float4 T;          /* throughput */
  uint64_t rng;
  uint32_t meta, slot;
  float t;           /* hit distance */
  uint32_t hit;      /* hit record */
};

/* how a shading step ended: the path is over and adds nothing, it goes on, or
 * it is over with the radiance it found (a path has at most one such vertex,
 * its last: nothing that emits scatters) */
#define SH_DEAD 0
#define SH_GOES_ON 1
#define SH_LIT 2

/* One shading step of the path `in` (entry i of the wavefront: where its
 * lobes are); its next state goes to `nx`, emitted radiance to `L`.  EXT adds
 * what only some scenes need (checker textures, surface coordinates, cone
 * lights), XF instance chains; batches without them use the leaner
 * instantiations.  MC_MISS reads only T, meta and slot. */
template <uint32_t CLS, bool GUIDE, bool EXT, bool XF>
__device__ __forceinline__ int shade_vertex(const DevScene &sc, const PathBuf &pb, const ShadeIn &in, uint32_t i,
                                            const GuideArgs &ga, NextPath &nx, float4 &L) {
  const uint32_t meta = in.meta, slot = in.slot;
  uint32_t hero_idx = meta & META_HERO_MASK;
  uint32_t depth = (meta >> META_DEPTH_SHIFT) & META_DEPTH_MASK;
  const DevJob &jb = sc.jobs[meta >> META_JOB_SHIFT];
  int wl[4];
  rotate_wl(hero_idx, wl);
  float4 T = in.T;
  if (CLS == MC_MISS) {
    const float *bg = sc.spd + jb.bg_spd;
    L.x = T.x * bg[wl[0] - CLV_LAMBDA_MIN];
    L.y = T.y * bg[wl[1] - CLV_LAMBDA_MIN];
    L.z = T.z * bg[wl[2] - CLV_LAMBDA_MIN];
    L.w = T.w * bg[wl[3] - CLV_LAMBDA_MIN];
    if (GUIDE && ga.record && jb.guiding) gd_credit(pb, ga, slot, T.x * bg[wl[0] - CLV_LAMBDA_MIN]);
    return SH_LIT;
  }
  const float4 o4 = in.o4, d4 = in.d4;
  V o = xyz(o4), d = xyz(d4);
  const float t = in.t;
  Hit h = hit_record<EXT, XF>(sc, in.hit, o, d, d4.w, t);
  const DevMaterial &m = sc.mats[h.material];
  if (CLS == MC_LIGHT) { /* DiffuseLight / ConeLight: emit on the front face (inside the cone), never scatter */
    bool lit = h.front;
    if (EXT && lit && m.cone) { /* cone_light.rs:46-53 */
      const float c = -dot(d, h.n) / (sqrtf(dot(d, d)) * sqrtf(dot(h.n, h.n)));
      lit = !(c >= -1.0f && c <= 1.0f && c < m.cone_cos);
    }
    if (lit) {
      const float *e = sc.spd + (EXT ? tex_spd(m, m.emit_spd, h) : m.emit_spd);
      L.x = T.x * e[wl[0] - CLV_LAMBDA_MIN];
      L.y = T.y * e[wl[1] - CLV_LAMBDA_MIN];
      L.z = T.z * e[wl[2] - CLV_LAMBDA_MIN];
      L.w = T.w * e[wl[3] - CLV_LAMBDA_MIN];
      if (GUIDE && ga.record && jb.guiding) gd_credit(pb, ga, slot, T.x * e[wl[0] - CLV_LAMBDA_MIN]);
      return SH_LIT;
    }
    return SH_DEAD;
  }
  uint64_t s = in.rng;
  /* attenuation (trace.rs:61-70; materials.rs:90-102) */
  const bool wdep = m.thin_film || m.kind == CLV_MAT_DISPERSIVE;
  float att[4];
  {
    const float *alb = m.albedo_spd >= 0 ? sc.spd + (EXT ? tex_spd(m, m.albedo_spd, h) : m.albedo_spd) : nullptr;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (wdep && j > 0) { att[j] = 0.0f; continue; }
      float k = alb ? alb[wl[j] - CLV_LAMBDA_MIN] : 1.0f;
      float tf = m.thin_film ? interference(m, d, h.n, wl[j]) : 1.0f;
      att[j] = k * tf;
    }
  }
  V nd;
  if (CLS == MC_LAMBERTIAN && EXT && m.kind == CLV_MAT_ISOTROPIC) {
    /* MixturePDF(HitablePDF(lights), SpherePDF) -- isotropic.rs:21-39, pdf.rs:144-168; never guided,
     * no training record (a medium vertex counts like a specular one for the credit rule) */
    if (GUIDE && ga.record && ga.indirect && jb.guiding) {
      const uint32_t g = pb.gcnt[slot];
      if (g && !(g & GD_SPECULAR)) pb.gcnt[slot] = g | GD_SPECULAR;
    }
    V gen = coin(s) ? tree_sample(sc, jb, h.p, s) : random_unit_vector(s);
    nd = unit(gen);
    const float sp = 1.0f / (4.0f * PI_F);
    const float mis = 0.5f * tree_pdf(sc, jb, h.p, nd) + 0.5f * sp;
    T.x = T.x * att[0] * sp / mis;
    T.y = T.y * att[1] * sp / mis;
    T.z = T.z * att[2] * sp / mis;
    T.w = T.w * att[3] * sp / mis;
  } else if (CLS == MC_LAMBERTIAN) {
    /* MixturePDF(HitablePDF(lights), CosinePDF(normal)) -- trace.rs:80-120, pdf.rs:106-141 */
    Onb b = onb_from_w(h.n);
    /* guided: the light-tree half of the mixture stays; the cosine half draws
     * from the learned lobes with probability alpha (one-sample MIS over all
     * three densities).  Unguided jobs draw exactly the plain sequence. */
    float pn[3] = {0.0f, 0.0f, 0.0f};
    if (GUIDE && ga.on && jb.guiding) gd_norm_pos(jb, h.p, pn);
    const bool guided = GUIDE && ga.on && jb.guiding && ga.alpha > 0.0f &&
                        gd_gate_open(ga, jb, meta >> META_JOB_SHIFT, o4, d4, t);
    const uint32_t *lob = guided ? ga.lobes + (size_t)i * GD_LWORDS : nullptr;
    const float alpha = guided ? ga.alpha : 0.0f;
    V gen;
    if (coin(s)) {
      gen = tree_sample(sc, jb, h.p, s);
    } else if (guided && rnd(s) < alpha) {
      float gx, gy, gz;
      const float u0 = rnd(s), u1 = rnd(s), u2 = rnd(s);
      gd_sample(lob, u0, u1, u2, gx, gy, gz);
      gen = mk(gx, gy, gz);
    } else {
      float r1 = rnd(s), r2 = rnd(s);
      float z = sqrtf(1.0f - r2);
      float phi = 2.0f * PI_F * r1;
      gen = onb_local(b, mk(cosf(phi) * sqrtf(r2), sinf(phi) * sqrtf(r2), z));
    }
    nd = unit(gen);
    float lp = tree_pdf(sc, jb, h.p, nd);
    V ndn = unit(nd);
    float cs = dot(ndn, b.w);
    float cp = cs <= 0.0f ? 0.0f : cs / PI_F;
    if (guided) cp = alpha * gd_pdf(lob, ndn.x, ndn.y, ndn.z) + (1.0f - alpha) * cp;
    float mis = 0.5f * lp + 0.5f * cp;
    float c2 = dot(h.n, ndn);
    if (c2 < 0.0f) return SH_DEAD; /* scattering_pdf None: return emitted (0 for Lambertian) */
    float spdf = c2 / PI_F;
    T.x = T.x * att[0] * spdf / mis;
    T.y = T.y * att[1] * spdf / mis;
    T.z = T.z * att[2] * spdf / mis;
    T.w = T.w * att[3] * spdf / mis;
    if (GUIDE && ga.record && jb.guiding && depth + 1u <= jb.max_depth) {
      const uint32_t cnt = pb.gcnt[slot] & ~GD_SPECULAR;
      GuideRec r;
      r.p[0] = pn[0];
      r.p[1] = pn[1];
      r.p[2] = pn[2];
      r.n[0] = h.n.x;
      r.n[1] = h.n.y;
      r.n[2] = h.n.z;
      r.d[0] = ndn.x;
      r.d[1] = ndn.y;
      r.d[2] = ndn.z;
      r.lam = (float)hero_idx / 400.0f;
      r.pdf = mis;
      r.cosv = c2;
      r.t0 = T.x;
      r.src = GD_SRC_CAMERA;
      r.stamp = ga.stamp;
      r.pad = 0u;
      ga.rec[(size_t)slot * GD_SLOTS + cnt % GD_SLOTS] = r;
      pb.recL[(size_t)slot * GD_SLOTS + cnt % GD_SLOTS] = 0.0f;
      pb.gcnt[slot] = cnt + 1u;
    }
  } else {
    if (GUIDE && ga.record && ga.indirect && jb.guiding) {
      const uint32_t g = pb.gcnt[slot];
      if (g && !(g & GD_SPECULAR)) pb.gcnt[slot] = g | GD_SPECULAR;
    }
    nd = specular_dir<CLS == MC_METAL>(m, d, h, hero_idx, s);
    T.x *= att[0];
    T.y *= att[1];
    T.z *= att[2];
    T.w *= att[3];
  }
  if (depth + 1u > jb.max_depth) return SH_DEAD; /* trace() at depth > max_depth returns 0 */
  nx.thr = T;
  nx.o = make_float4(h.p.x, h.p.y, h.p.z, o4.w); /* .w: root node of the path's scene */
  nx.d = make_float4(nd.x, nd.y, nd.z, d4.w);    /* .w: the ray's instant stays with the path */
  nx.rng = s;
  nx.meta = (meta & ~(META_DEPTH_MASK << META_DEPTH_SHIFT)) | ((depth + 1u) << META_DEPTH_SHIFT);
  nx.slot = slot;
  return SH_GOES_ON;
}

/* the wavefront's shading step: the path at entry i of the path state; returns
 * true if the path continues */
template <uint32_t CLS, bool GUIDE, bool EXT>
__device__ __forceinline__ bool shade_path(const DevScene &sc, const PathBuf &pb, uint32_t i, const GuideArgs &ga,
                                           NextPath &nx) {
  ShadeIn in;
  in.meta = pb.meta[i];
  in.slot = pb.slot[i];
  in.T = pb.thr[i];
  if (CLS != MC_MISS) {
    in.o4 = pb.ray_o[i];
    in.d4 = pb.ray_d[i];
    in.t = pb.hit_t[i];
    in.hit = pb.hit_p[i];
    in.rng = pb.rng[i];
  }
  float4 L;
  const int r = shade_vertex<CLS, GUIDE, EXT, true>(sc, pb, in, i, ga, nx, L);
  if (r == SH_LIT) {
    float4 sum = pb.rad[in.slot];
    sum.x += L.x;
    sum.y += L.y;
    sum.z += L.z;
    sum.w += L.w;
    pb.rad[in.slot] = sum;
  }
  return r == SH_GOES_ON;
}

/* the plain instance is compiled for 7 waves per SIMD (72 VGPRs, none
 * spilled; the compiler alone takes 88 and 5 waves), the extended one for 6
 * (80 VGPRs; at 7 it spills), the guided one for 5 (96 VGPRs; 111 and 4
 * waves left alone); the guided extended one keeps the compiler's choice
 * (it spills at 5).  The shading kernel waits on chains of dependent loads,
 * so more waves in flight pay */
template <bool GUIDE, bool EXT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(GUIDE ? (EXT ? 1 : 5) : (EXT ? 6 : 7)))) void k_shade(
    DevScene sc, PathBuf pb, ShadeQueues sq, uint32_t *counts, uint32_t out_slot, GuideArgs ga) {
  __shared__ uint32_t agg[1 * 4 + 1];
  __shared__ NextPath stage[256]; /* survivors' state across the compaction (keeps it out of registers) */
  uint32_t c[MC_COUNT], chunks[MC_COUNT + 1];
  chunks[0] = 0;
#pragma unroll
  for (uint32_t k = 0; k < MC_COUNT; k++) {
    c[k] = sq.counts[k];
    chunks[k + 1] = chunks[k] + (c[k] + 63u) / 64u;
  }
  const uint32_t total = chunks[MC_COUNT];
  const uint32_t lane = threadIdx.x & 63u;
  /* block-uniform loop: each iteration the block's 4 waves take 4 consecutive 64-path chunks */
  for (uint32_t first = blockIdx.x * 4u; first < total; first += gridDim.x * 4u) {
    const uint32_t wv = first + (threadIdx.x >> 6);
    bool cont = false;
    if (wv < total) {
      uint32_t cls = 0;
#pragma unroll
      for (uint32_t k = 1; k < MC_COUNT; k++)
        if (wv >= chunks[k]) cls = k;
      cls = __builtin_amdgcn_readfirstlane(cls);
      uint32_t idx = (wv - chunks[cls]) * 64u + lane;
      if (idx < c[cls]) {
        const uint32_t path = sq.q[cls][idx];
        NextPath &nx = stage[threadIdx.x];
        switch (cls) {
          case MC_MISS: cont = shade_path<MC_MISS, GUIDE, EXT>(sc, pb, path, ga, nx); break;
          case MC_LIGHT: cont = shade_path<MC_LIGHT, GUIDE, EXT>(sc, pb, path, ga, nx); break;
          case MC_LAMBERTIAN: cont = shade_path<MC_LAMBERTIAN, GUIDE, EXT>(sc, pb, path, ga, nx); break;
          case MC_METAL: cont = shade_path<MC_METAL, GUIDE, EXT>(sc, pb, path, ga, nx); break;
          default: cont = shade_path<MC_GLASS, GUIDE, EXT>(sc, pb, path, ga, nx); break;
        }
      }
    }
    /* survivors are compacted into the next bounce's entries, in block order */
    const uint32_t e = block_append_pos<1, 256>(cont ? 0u : 1u, counts + out_slot, agg);
    if (cont) {
      const NextPath &nx = stage[threadIdx.x];
      pb.n_ray_o[e] = nx.o;
      pb.n_ray_d[e] = nx.d;
      pb.n_thr[e] = nx.thr;
      pb.n_rng[e] = nx.rng;
      pb.n_meta[e] = nx.meta;
      pb.n_slot[e] = nx.slot;
    }
  }
}

/* one sample's XYZ contribution (the estimator of draw_cpu.rs:130-142) from
 * its radiance at the four wavelengths that follow the hero */
__device__ __forceinline__ void sample_xyz(const float4 *cie, float4 L, uint32_t hero, float c[3]) {
  c[0] = c[1] = c[2] = 0.0f;
  if (L.y == 0.0f && L.z == 0.0f && L.w == 0.0f) {
    float4 x = cie[hero];
    c[0] = x.x * L.x;
    c[1] = x.y * L.x;
    c[2] = x.z * L.x;
  } else {
    float Ls[4] = {L.x, L.y, L.z, L.w};
#pragma unroll
    for (int q = 0; q < 4; q++) {
      float p = Ls[q];
      if (isnormal(p) && !signbit(p)) {
        float4 x = cie[(hero + 100u * (uint32_t)q) % 400u];
        c[0] += x.x * p / 4.0f;
        c[1] += x.y * p / 4.0f;
        c[2] += x.z * p / 4.0f;
      }
    }
  }
}

/* -------------------------------------- traversal of the whole-path kernel --- */
typedef __attribute__((address_space(3))) float4 lds_f4;
/* the 32-bit LDS address of a shared-memory pointer */
__device__ __forceinline__ uint32_t lds_addr(const void *p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)p; }
__device__ __forceinline__ uint32_t lds_ld(uint32_t a) { return *(const lds_u32 *)(uintptr_t)a; }
__device__ __forceinline__ void lds_st(uint32_t a, uint32_t v) { *(lds_u32 *)(uintptr_t)a = v; }
__device__ __forceinline__ float4 lds_ld4(uint32_t a) {
  const __attribute__((address_space(3))) float *p = (const __attribute__((address_space(3))) float *)(uintptr_t)a;
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 v = *(const __attribute__((address_space(3))) f4 *)p;
  return make_float4(v.x, v.y, v.z, v.w);
}

/* A lane's ray on its way through the tree.  FULL: the scene lies in the
 * block's LDS and its child words were rewritten for it (interior: byte offset
 * of the node, leaf: unit offset in the window); else they are arena words. */
struct Trav {
  V o, d, inv, oi;
  uint32_t rx, ry, rz;   /* byte offset of the near-plane row per axis */
  float tb, time;
  float a, ra;           /* d.d and its reciprocal (sphere tests of rays that are not transformed) */
  uint32_t best, word;
  uint32_t sp;           /* LDS address of the next free stack entry; entry 0 holds CHILD_EMPTY */
};

/* n / a, correctly rounded, from ra = RN(1/a): a quotient and two residual
 * corrections (Markstein 1990, "Computation of elementary functions on the IBM
 * RISC System/6000 processor"), half the operations of a full division.  For
 * 1/2 < a < 2 and quotients far from the ends of the range; elsewhere the
 * result is still outside every [tmin, tmax] it is compared with, or NaN. */
__device__ __forceinline__ float div_by(float n, float a, float ra) {
  float q = n * ra;
  q = fmaf(fmaf(-a, q, n), ra, q);
  return fmaf(fmaf(-a, q, n), ra, q);
}

/* sphere_t for the ray's own d.d and its reciprocal */
__device__ __forceinline__ bool sphere_hit(V c, float r, const Trav &L, float tmin, float tmax, float &t) {
  V oc = L.o - c;
  float half_b = dot(oc, L.d);
  float cc = dot(oc, oc) - r * r;
  float disc = half_b * half_b - L.a * cc;
  if (!(disc > 0.0f)) return false;
  float root = sqrtf(disc);
  float t0 = div_by(-half_b - root, L.a, L.ra);
  if (t0 < tmax && t0 > tmin) { t = t0; return true; }
  float t1 = div_by(-half_b + root, L.a, L.ra);
  if (t1 < tmax && t1 > tmin) { t = t1; return true; }
  return false;
}

/* entries of a stack: the pending children the host allows, CHILD_EMPTY below them, and the word of a ray that is
 * left on its way above them */
#define TRAV_TOTAL (STACK_TOTAL + 2)
template <int BLOCK, int DEPTH>
struct TravStack {
  uint32_t lst;      /* LDS address of the lane's entry 0; entries are BLOCK words apart */
  uint32_t *spill;   /* this block's slices */
  static constexpr uint32_t STRIDE = 4u * BLOCK, N = DEPTH;
  __device__ __forceinline__ uint32_t *deep(uint32_t e) const {
    return spill + (size_t)threadIdx.x * (TRAV_TOTAL - DEPTH) + (e - DEPTH);
  }
  __device__ __forceinline__ void start(Trav &L) const {
    lds_st(lst, CHILD_EMPTY);
    L.sp = lst + STRIDE;
  }
  /* a ray that is left on its way: its word on top of the stack, the stack's end in entry 0 */
  __device__ __forceinline__ void leave(const Trav &L) const {
    const uint32_t e = (L.sp - lst) / STRIDE;
    if (e < DEPTH) lds_st(L.sp, L.word);
    else *deep(e) = L.word;
    lds_st(lst, L.sp);
  }
  __device__ __forceinline__ void resume(Trav &L) const {
    L.sp = lds_ld(lst);
    lds_st(lst, CHILD_EMPTY);
    const uint32_t e = (L.sp - lst) / STRIDE;
    L.word = e < DEPTH ? lds_ld(L.sp) : *deep(e);
  }
  /* the children at distances tn[1..3] that were hit (sorted: hits first), far to near */
  __device__ __forceinline__ void push3(Trav &L, const uint32_t cw[4], const float tn[4]) const {
    if (__any(L.sp > lst + (DEPTH - 3) * STRIDE)) { /* some lane may leave its LDS part */
#pragma unroll
      for (int k = 3; k >= 1; k--)
        if (tn[k] < FLT_MAX) {
          const uint32_t e = (L.sp - lst) / STRIDE;
          if (e < DEPTH) lds_st(L.sp, cw[k]);
          else if (e < TRAV_TOTAL) *deep(e) = cw[k]; /* always: the host bounds the BVH depth */
          L.sp += STRIDE;
        }
    } else { /* stores without branches; the stack grows past the ones that were hit */
#pragma unroll
      for (int k = 3; k >= 1; k--) {
        lds_st(L.sp, cw[k]);
        L.sp += tn[k] < FLT_MAX ? STRIDE : 0u;
      }
    }
  }
  __device__ __forceinline__ void pop(Trav &L) const {
    L.sp -= STRIDE;
    if (__any(L.sp > lst + (DEPTH - 1) * STRIDE)) {
      const uint32_t e = (L.sp - lst) / STRIDE;
      L.word = e < DEPTH ? lds_ld(L.sp) : *deep(e);
    } else {
      L.word = lds_ld(L.sp);
    }
  }
};

#define TRAV_SORT4(tn, cw)                                                \
  do {                                                                    \
    auto swp = [&](int a, int b) {                                        \
      const bool s_ = tn[b] < tn[a];                                      \
      const float ta_ = tn[a], tb_ = tn[b];                               \
      const uint32_t ca_ = cw[a], cb_ = cw[b];                            \
      tn[a] = s_ ? tb_ : ta_; tn[b] = s_ ? ta_ : tb_;                     \
      cw[a] = s_ ? cb_ : ca_; cw[b] = s_ ? ca_ : cb_;                     \
    };                                                                    \
    swp(0, 1); swp(2, 3); swp(0, 2); swp(1, 3); swp(1, 2);                \
  } while (0)

/* after the slab tests of a node: on to the nearest child hit, the others on the stack */
template <class STACK>
__device__ __forceinline__ void trav_next(Trav &L, float tn[4], uint32_t cw[4], const STACK &S) {
  TRAV_SORT4(tn, cw);
  S.push3(L, cw, tn);
  if (tn[0] < FLT_MAX) L.word = cw[0];
  else S.pop(L);
}

/* one node of the window, at LDS address p: near and far planes per axis picked by the ray's signs (slab4) */
template <class STACK>
__device__ __forceinline__ void trav_node_lds(Trav &L, uint32_t p, const STACK &S) {
  const uint32_t px = p + L.rx, py = p + L.ry, pz = p + L.rz;
  const float4 cf = lds_ld4(p + 96u);
  const float4 nx = lds_ld4(px), fx = lds_ld4(px ^ 16u), ny = lds_ld4(py), fy = lds_ld4(py ^ 16u), nz = lds_ld4(pz),
               fz = lds_ld4(pz ^ 16u);
  const float nxa[4] = {nx.x, nx.y, nx.z, nx.w}, fxa[4] = {fx.x, fx.y, fx.z, fx.w};
  const float nya[4] = {ny.x, ny.y, ny.z, ny.w}, fya[4] = {fy.x, fy.y, fy.z, fy.w};
  const float nza[4] = {nz.x, nz.y, nz.z, nz.w}, fza[4] = {fz.x, fz.y, fz.z, fz.w};
  const float tfar_lim = L.tb * 1.00000024f;
  uint32_t cw[4] = {as_u(cf.x), as_u(cf.y), as_u(cf.z), as_u(cf.w)};
  float tn[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const float x0 = fmaf(nxa[k], L.inv.x, -L.oi.x), x1 = fmaf(fxa[k], L.inv.x, -L.oi.x);
    const float y0 = fmaf(nya[k], L.inv.y, -L.oi.y), y1 = fmaf(fya[k], L.inv.y, -L.oi.y);
    const float z0 = fmaf(nza[k], L.inv.z, -L.oi.z), z1 = fmaf(fza[k], L.inv.z, -L.oi.z);
    const float tnear = fmaxf(fmaxf(x0, y0), fmaxf(z0, EPS_ACNE));
    const float tfar = fminf(fminf(x1, y1), fminf(z1, tfar_lim));
    tn[k] = tnear <= tfar ? tnear : FLT_MAX;
  }
  trav_next(L, tn, cw, S);
}

/* one node in global memory */
template <class STACK>
__device__ __forceinline__ void trav_node_global(Trav &L, const Bvh4Node *nd, const STACK &S) {
  const float4 *nf = reinterpret_cast<const float4 *>(nd);
  const uint4 ch = reinterpret_cast<const uint4 *>(nd)[6];
  uint32_t cw[4] = {ch.x, ch.y, ch.z, ch.w};
  float tn[4];
  slab4_minmax(L, nf, cw, tn);
  trav_next(L, tn, cw, S);
}

/* rays of a wave that are left on their way: less than one in PS_LEAVE (mesh of 1M triangles: 63.6 ms without,
 * 57.5 at 32, 53.0 at 16, 49.6 at 8, 48.0 at 4, 48.3 at 3) */
#define PS_LEAVE 4u
/* The closest hit of a ray (L.tb, L.best: an arena record offset), from its
 * start or, with `resumed`, from where it was left.  A few rays of a wave go on
 * for long: over a third of the steps are taken for less than a quarter of its
 * lanes.  From memory, a wave leaves once fewer than 1 / PS_LEAVE of the rays it
 * came with are on their way: those keep their stacks, best hits and lanes
 * (false) and go on beside the wave's next rays; a wave with a handful finishes
 * them.  In LDS the steps are too short for that: the rounds that the leftovers
 * fill less cost more than they save (sphere field 28.6 -> 30.2 ms, prism 16.1
 * -> 18.8). */
template <bool FULL, bool XF, class STACK>
__device__ __forceinline__ bool trav_ray(Trav &L, const DevScene &sc, const LdsWindow &w, const STACK &S, uint32_t root,
                                         bool resumed) {
  const uint32_t few = FULL ? 0u : (uint32_t)__popcll(__ballot(true)) / PS_LEAVE;
  {
    Lane s;
    lane_start_ray(s, L.o, L.d, L.time, FULL ? 0u : root);
    L.inv = s.inv;
    L.oi = s.oi;
    L.word = s.word;
  }
  if (resumed) {
    S.resume(L);
  } else {
    L.tb = FLT_MAX;
    L.best = MISS_WORD;
    S.start(L);
  }
  if (FULL) {
    L.rx = (as_u(L.inv.x) >> 31) * 16u;
    L.ry = (as_u(L.inv.y) >> 31) * 16u + 32u;
    L.rz = (as_u(L.inv.z) >> 31) * 16u + 64u;
    L.a = dot(L.d, L.d);
    L.ra = 1.0f / L.a;
    const uint32_t nodes = lds_addr(w.nodes), prims = lds_addr(w.prims);
    for (;;) {
      /* a primitive in an instance costs several nodes: while two lanes or more wait with one for every lane at
       * a node, the wave tests primitives (features room 3.34 -> 3.23 ms; without instances both each turn:
       * prism 16.3, by that rule 17.1) */
      const bool node = !(L.word & CHILD_LEAF);
      bool nodes_now = true;
      if (XF) {
        const uint64_t going = __ballot(L.word != CHILD_EMPTY);
        if (going == 0u) break;
        const uint32_t nn = (uint32_t)__popcll(__ballot(node));
        nodes_now = 3u * nn >= (uint32_t)__popcll(going);
      } else if (L.word == CHILD_EMPTY) {
        break;
      }
      if (node) {
        if (nodes_now) trav_node_lds(L, nodes + L.word, S);
      } else if (!XF || (!nodes_now && L.word != CHILD_EMPTY)) {
        /* one primitive per step: a lane on a leaf of 8 does not hold up the
         * lanes taking node steps; the leaf word counts its primitives down
         * and its offset up (the same order, so the same hits) */
        const uint32_t off = L.word & LEAF_OFFSET_MASK, p = prims + off * 16u;
        const bool last = ((L.word >> 28) & 7u) == 0u;
        const float4 f0 = lds_ld4(p), f1 = lds_ld4(p + 16u), *rec = w.prims + off;
        const uint32_t hdr = as_u(f0.w), type = hdr & PT_TYPE_MASK;
        float t;
        bool h;
        if (XF && (hdr >> PT_XF_SHIFT)) h = test_prim<true>(sc, rec, hdr, L.o, L.d, L.time, EPS_ACNE, L.tb, t);
        else if (type == PT_SPHERE) h = sphere_hit(xyz(f0), f1.x, L, EPS_ACNE, L.tb, t);
        else if (type == PT_MSPHERE) h = sphere_hit(xyz(f0) + L.time * xyz(rec[2]), f1.x, L, EPS_ACNE, L.tb, t);
        else if (type == PT_TRI) h = plane_t<true>(rec, L.o, L.d, EPS_ACNE, L.tb, t);
        else h = plane_t<false>(rec, L.o, L.d, EPS_ACNE, L.tb, t);
        if (h) {
          L.tb = t;
          L.best = off + w.ub;
        }
        if (last) S.pop(L);
        else L.word += prim_units(type) - (1u << 28);
      }
    }
  } else {
    /* nodes and records come from L2 and beyond, the lanes of a wave from as
     * many places; the wave takes node steps while most of its lanes have one
     * to take, then leaf steps, so that each round of fetches serves more
     * lanes */
    for (;;) {
      const bool leaf = L.word >= CHILD_LEAF && L.word != CHILD_EMPTY, node = L.word < CHILD_LEAF;
      const uint32_t nn = (uint32_t)__popcll(__ballot(node)), nl = (uint32_t)__popcll(__ballot(leaf));
      if (nn + nl <= few) { /* few: 0 for less than PS_LEAVE */
        if (nn + nl == 0u || !(node || leaf)) break;
        S.leave(L);
        return false;
      }
      if (nn >= nl) {
        if (node) trav_node_global(L, sc.nodes + L.word, S);
      } else if (leaf) {
        const uint32_t off = L.word & LEAF_OFFSET_MASK;
        const bool last = ((L.word >> 28) & 7u) == 0u;
        const float4 *rec = sc.prims + off;
        const uint32_t hdr = as_u(rec[0].w);
        float t;
        if (test_prim<XF>(sc, rec, hdr, L.o, L.d, L.time, EPS_ACNE, L.tb, t)) {
          L.tb = t;
          L.best = off;
        }
        if (last) S.pop(L);
        else L.word += prim_units(hdr & PT_TYPE_MASK) - (1u << 28);
      }
    }
  }
  return true;
}

/* ------------------------------------------------- whole paths, one launch --- */
/* A plain render's pass in one launch.  The wavefront above moves every path
 * through HBM twice per bounce and launches three kernels per bounce, and from
 * the fourth bounce or so on those launches hold a few percent of the paths.
 * Here a resident block carries BLOCK paths in registers from the camera to
 * their end.  One turn of its loop is one bounce:
 *
 *   trace    every lane follows its ray (the LDS-cached traversal);
 *   sort     the block's paths change lanes so that they lie in the order of
 *            their material classes: per-wave ballots give every path its place,
 *            its 17 words of state travel through LDS in two rounds (a ray that
 *            is still on its way keeps its lane).  A wave
 *            then shades one class, or two where a boundary falls inside it;
 *   shade    shade_vertex, as the wavefront; a path that ends writes its
 *            sample's XYZ contribution at its slot (k_resolve_xyz sums the
 *            samples of a pixel in sample order, so no result depends on which
 *            block ran a path, or when);
 *   refill   lanes without a path take the next camera samples.  Misses and
 *            emitters sort first and always end, so whole waves get fresh
 *            samples, 64 neighbours in tile order, and stay coherent.
 *
 * Samples come from a pass-wide cursor in chunks that a block takes ahead of
 * need (one global atomic per chunk).  The exchange rounds use the memory of
 * the traversal stacks, which are empty then.  Every path runs the same
 * operations on the same stream as in the wavefront: the same image, bit for
 * bit.
 *
 * FULL: the scene of every job lies in the block's LDS, its child words
 * rewritten to LDS offsets; else nodes and records come from memory.  In LDS
 * the kernel is bound by VALU issue: 512-thread blocks, three to a CU beside
 * a sphere field's 33 KB, at 6 waves per SIMD (80 VGPRs); 768 threads take
 * 29.4 ms where 512 take 29.2 and leave less room for larger scenes, 512
 * threads at 5 waves and no spills 36.4.  From memory it waits on node
 * fetches (with stacks and spills 5.2 TB/s behind L2, as a large copy): two-wave
 * blocks at 8 waves per SIMD, and rays that are left on their way while the
 * others are shaded (trav_ray): the 1M-triangle mesh takes 46.8
 * ms, 48.9 in blocks of 256 threads, 47.9 of 64, 49.4 at 6 waves (before rays
 * were left: 63.6, and 68.6 / 69.1 with node and leaf steps taken in another
 * order than by majority: node-first / both each turn).  XF, EXT and
 * MEDIA leave out of the registers what a batch has none of: without XF the
 * sphere field goes from 32.7 to 29.2 ms.
 *
 * A wave is refilled once 16 of its lanes are free: below that the camera
 * code costs more than the idle lanes (sphere field 32.8 ms at 1, 31.4 at 8 and
 * 16, 31.8 at 32, 33.9 at 64); what is left over sorts to the block's end.  From
 * memory, once 4 are: tracing is more of the time there (mesh 48.2 ms at 16, 47.1
 * at 8, 46.8 at 4 and 1).
 *
 * Whole calls, before this kernel -> now: sphere field 1920x1080 64 spp 60.5
 * -> 29.2 ms, prism 1024^2 64 spp 33.1 -> 16.7, mesh 4 views 8 spp 138.5 -> 49,
 * Cornell 256^2 16 spp 0.695 -> 0.58. */
#define PS_REFILL 16u
#define PS_REFILL_GLOBAL 4u
#define PS_WORDS 9 /* LDS words per lane: stack entries, or one round of the exchange */
/* lanes of mask m below this one */
__device__ __forceinline__ uint32_t below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

template <int BLOCK, bool EXT, bool MEDIA, bool FULL, bool XF>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(MEDIA ? 4 : (FULL ? 6 : 8)))) void k_paths(DevScene sc, GenParams gp,
                                                                                      PathsArgs pa) {
  constexpr uint32_t WAVES = BLOCK / 64;
  static_assert((MC_COUNT + 1) * WAVES <= 64, "one lane of a wave per (class or free, wave) count");
  extern __shared__ __attribute__((aligned(128))) float4 scene[]; /* rows of a plane pair differ in address bit 4 */
  __shared__ uint32_t cnt[64];   /* paths per (class, wave), then lanes per wave whose ray is not on its way */
  __shared__ uint8_t nth[BLOCK]; /* per wave: its n-th such lane */
  __shared__ uint32_t pool[4];   /* sample ids at hand: [0] base and [1] length of the first range, [2] base of the
                                    second (pa.chunk long), [3] ids taken since the ranges were set */
  const LdsWindow win = {scene, scene + pa.lds_nodes * 8u, pa.lds_nodes, pa.lds_node_base, pa.lds_units, pa.lds_unit_base};
  const uint32_t tid = threadIdx.x, lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t *ex = reinterpret_cast<uint32_t *>(scene + pa.lds_nodes * 8u + pa.lds_units);
  TravStack<BLOCK, PS_WORDS> S;
  S.lst = lds_addr(ex + tid);
  S.spill = pa.spill + (size_t)blockIdx.x * BLOCK * (TRAV_TOTAL - PS_WORDS);
  {
    const float4 *gn = reinterpret_cast<const float4 *>(sc.nodes + win.nb);
    auto local = [&](float f) { /* a child word for FULL (struct Trav) */
      const uint32_t c = as_u(f);
      return __uint_as_float(c == CHILD_EMPTY ? c : (c & CHILD_LEAF) ? c - win.ub : (c - win.nb) * 128u);
    };
    for (uint32_t k = tid; k < win.nn * 8u; k += BLOCK) {
      float4 v = gn[k];
      if (FULL && (k & 7u) == 6u) v = make_float4(local(v.x), local(v.y), local(v.z), local(v.w));
      scene[k] = v;
    }
    for (uint32_t k = tid; k < win.nu; k += BLOCK) scene[win.nn * 8u + k] = sc.prims[win.ub + k];
    if (tid == 0) {
      pool[0] = 0u;
      pool[1] = 0u;
      pool[2] = 0u;
      pool[3] = pa.chunk; /* both ranges used up */
    }
  }
  __syncthreads();
  const uint32_t n = gp.paths;
  uint32_t rays = 0;
  bool exhausted = false; /* thread 0: the pass-wide cursor has passed the last sample */
  /* the lane's path */
  ShadeIn ps;
  ps.T = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
  ps.rng = 0;
  ps.meta = 0;
  ps.slot = tid < pa.first ? blockIdx.x * pa.first + tid : 0xFFFFFFFFu;
  V o = mk(0.0f, 0.0f, 0.0f), d = o;
  float time = 0.0f;
  bool alive = ps.slot < n;
  uint64_t under = 0; /* the wave's lanes whose ray was left on its way */
  ps.t = 0.0f;
  ps.hit = 0;
  if (alive) ps.meta = camera_sample(sc, gp, ps.slot, o, d, time, ps.rng);
  for (;;) {
    /* trace */
    uint32_t cls = MC_COUNT;
    Trav L;
    L.tb = ps.t;
    L.best = ps.hit;
    const bool resumed = ((under >> lane) & 1u) != 0u;
    bool done = true;
    rays += (uint32_t)__popcll(__ballot(alive && !resumed));
    if (alive) {
      L.o = o;
      L.d = d;
      L.time = time;
      done = trav_ray<FULL, XF>(L, sc, win, S, FULL ? 0u : sc.jobs[ps.meta >> META_JOB_SHIFT].root, resumed);
      if (done) {
        if (MEDIA) {
          Lane m;
          m.o = o;
          m.d = d;
          m.tb = L.tb;
          m.best = L.best;
          lane_media(m, sc, ps.meta, ps.rng);
          L.tb = m.tb;
          L.best = m.best;
        }
        cls = L.best != MISS_WORD ? sc.mats[sc.info[as_u(sc.prims[L.best + 1u].w)].material].mclass : MC_MISS;
      } else {
        ps.t = L.tb;
        ps.hit = L.best;
      }
    }
    under = __ballot(!done);
    /* each path's place in class order */
    uint32_t rank = 0;
#pragma unroll
    for (uint32_t c = 0; c < MC_COUNT; c++) {
      const uint64_t m = __ballot(cls == c);
      if (lane == 0) cnt[c * WAVES + wave] = (uint32_t)__popcll(m);
      if (cls == c) rank = below(m);
    }
    const uint32_t own_free = below(~under);
    if (lane == 0) cnt[MC_COUNT * WAVES + wave] = 64u - (uint32_t)__popcll(under);
    if (!FULL && done) nth[wave * 64u + own_free] = (uint8_t)lane;
    __syncthreads();
    if (tid == 0 && pool[3] >= pool[1]) { /* the first range is used up: the rest of the second follows, and a new one */
      const uint32_t over = pool[3] - pool[1];
      pool[0] = pool[2] + over;
      pool[1] = pa.chunk - over;
      pool[3] = 0u;
      uint32_t base = n;
      if (!exhausted) base = atomicAdd(pa.next, pa.chunk);
      exhausted = base >= n;
      pool[2] = base;
    }
    uint32_t sum = lane < (MC_COUNT + 1) * WAVES ? cnt[lane] : 0u;
    const uint32_t own = sum;
#pragma unroll
    for (uint32_t k = 1; k < 64u; k <<= 1) {
      const uint32_t up = __shfl_up(sum, k);
      if (lane >= k) sum += up;
    }
    const uint32_t total = __builtin_amdgcn_readlane(sum, MC_COUNT * WAVES - 1);
    const uint32_t left = BLOCK + total - __builtin_amdgcn_readlane(sum, 63); /* rays on their way */
    if (total + left == 0u) break; /* the same in every wave: nothing left to trace, and the last refill found no sample */
    const uint32_t excl = sum - own;
    uint32_t start[MC_COUNT];
#pragma unroll
    for (uint32_t c = 1; c < MC_COUNT; c++) start[c] = __builtin_amdgcn_readlane(excl, c * WAVES);
    /* the place in class order is that of the lane among those without a ray on its way */
    const uint32_t at = FULL ? tid : own_free + __builtin_amdgcn_readlane(excl, MC_COUNT * WAVES + wave) - total;
    uint32_t dest = __shfl(excl, (int)(min(cls, MC_COUNT - 1u) * WAVES + wave)) + rank;
    if (!FULL) {
      uint32_t first = 0, in = 0; /* the wave that holds the place, and its first one */
#pragma unroll
      for (uint32_t k = 1; k < WAVES; k++) {
        const uint32_t f = __builtin_amdgcn_readlane(excl, MC_COUNT * WAVES + k) - total;
        if (dest >= f) {
          first = f;
          in = k * 64u;
        }
      }
      if (cls < MC_COUNT) dest = in + nth[in + dest - first];
    }
    /* the paths change lanes */
    uint32_t *w = ex + dest;
    const uint32_t *r = ex + tid;
    const bool moves = cls < MC_COUNT;
    const bool shades = done && at < total;
    alive = shades || !done;
    if (moves) {
      lds_store(w, as_u(o.x));
      lds_store(w + BLOCK, as_u(o.y));
      lds_store(w + 2 * BLOCK, as_u(o.z));
      lds_store(w + 3 * BLOCK, as_u(d.x));
      lds_store(w + 4 * BLOCK, as_u(d.y));
      lds_store(w + 5 * BLOCK, as_u(d.z));
      lds_store(w + 6 * BLOCK, as_u(time));
      lds_store(w + 7 * BLOCK, as_u(L.tb));
      lds_store(w + 8 * BLOCK, L.best);
    }
    __syncthreads();
    if (shades) {
      o = mk(__uint_as_float(lds_load(r)), __uint_as_float(lds_load(r + BLOCK)), __uint_as_float(lds_load(r + 2 * BLOCK)));
      d = mk(__uint_as_float(lds_load(r + 3 * BLOCK)), __uint_as_float(lds_load(r + 4 * BLOCK)),
             __uint_as_float(lds_load(r + 5 * BLOCK)));
      time = __uint_as_float(lds_load(r + 6 * BLOCK));
      ps.t = __uint_as_float(lds_load(r + 7 * BLOCK));
      ps.hit = lds_load(r + 8 * BLOCK);
    }
    __syncthreads();
    if (moves) {
      lds_store(w, as_u(ps.T.x));
      lds_store(w + BLOCK, as_u(ps.T.y));
      lds_store(w + 2 * BLOCK, as_u(ps.T.z));
      lds_store(w + 3 * BLOCK, as_u(ps.T.w));
      lds_store(w + 4 * BLOCK, (uint32_t)ps.rng);
      lds_store(w + 5 * BLOCK, (uint32_t)(ps.rng >> 32));
      lds_store(w + 6 * BLOCK, ps.meta);
      lds_store(w + 7 * BLOCK, ps.slot);
    }
    __syncthreads();
    if (shades) {
      ps.T = make_float4(__uint_as_float(lds_load(r)), __uint_as_float(lds_load(r + BLOCK)),
                         __uint_as_float(lds_load(r + 2 * BLOCK)), __uint_as_float(lds_load(r + 3 * BLOCK)));
      ps.rng = (uint64_t)lds_load(r + 4 * BLOCK) | ((uint64_t)lds_load(r + 5 * BLOCK) << 32);
      ps.meta = lds_load(r + 6 * BLOCK);
      ps.slot = lds_load(r + 7 * BLOCK);
    }
    __syncthreads(); /* the exchange is over: the memory is the stacks' again */
    /* shade */
    if (shades) {
      ps.o4 = make_float4(o.x, o.y, o.z, 0.0f);
      ps.d4 = make_float4(d.x, d.y, d.z, time);
      uint32_t c = 0;
#pragma unroll
      for (uint32_t k = 1; k < MC_COUNT; k++) c += at >= start[k] ? 1u : 0u;
      NextPath nx;
      float4 lit = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      int end;
      const PathBuf pb = PathBuf();
      const GuideArgs ga = GuideArgs();
      switch (c) {
        case MC_MISS: end = shade_vertex<MC_MISS, false, EXT, XF>(sc, pb, ps, 0u, ga, nx, lit); break;
        case MC_LIGHT: end = shade_vertex<MC_LIGHT, false, EXT, XF>(sc, pb, ps, 0u, ga, nx, lit); break;
        case MC_LAMBERTIAN: end = shade_vertex<MC_LAMBERTIAN, false, EXT, XF>(sc, pb, ps, 0u, ga, nx, lit); break;
        case MC_METAL: end = shade_vertex<MC_METAL, false, EXT, XF>(sc, pb, ps, 0u, ga, nx, lit); break;
        default: end = shade_vertex<MC_GLASS, false, EXT, XF>(sc, pb, ps, 0u, ga, nx, lit); break;
      }
      if (end == SH_GOES_ON) {
        o = mk(nx.o.x, nx.o.y, nx.o.z);
        d = mk(nx.d.x, nx.d.y, nx.d.z);
        ps.T = nx.thr;
        ps.rng = nx.rng;
        ps.meta = nx.meta;
      } else {
        alive = false;
        F3 c3 = {0.0f, 0.0f, 0.0f};
        if (end == SH_LIT) sample_xyz(pa.cie, lit, ps.meta & META_HERO_MASK, &c3.x);
        pa.res[ps.slot] = c3;
      }
    }
    /* refill */
    const uint64_t idle = __ballot(!alive);
    if ((uint32_t)__popcll(idle) >= (FULL ? PS_REFILL : PS_REFILL_GLOBAL)) {
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(&pool[3], (uint32_t)__popcll(idle));
      base = __builtin_amdgcn_readfirstlane(base);
      if (!alive) {
        const uint32_t k = base + below(idle), len = pool[1];
        ps.slot = k < len ? pool[0] + k : pool[2] + (k - len);
        alive = ps.slot < n;
        if (alive) {
          ps.meta = camera_sample(sc, gp, ps.slot, o, d, time, ps.rng);
          ps.T = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
        }
      }
    }
  }
  if (lane == 0 && rays) atomicAdd(pa.stats + 2, (unsigned long long)rays);
}

/* the counters of a pass of k_paths: the sample cursor starts behind the
 * blocks' first samples; with `stats`, the render's counters too */
__global__ void k_paths_begin(uint32_t *next, uint32_t value, unsigned long long *stats) {
  if (threadIdx.x == 0) *next = value;
  if (stats && threadIdx.x < 8u) stats[threadIdx.x] = 0ull;
}

/* the per-pixel sums of a pass of k_paths, in sample order, one thread per
 * (pass item, pixel).  A job whose samples are all in one pass goes straight
 * to its means; sums of others wait in the accumulators between passes.  The
 * second moments are summed only where some job returns them. */
__global__ __launch_bounds__(256) void k_resolve_xyz(ResolveParams rp, const F3 *res, float *out, float *out_sq) {
  for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < rp.threads; g += gridDim.x * blockDim.x) {
    const DevItem it = rp.items[find_entry(rp.items, rp.n_items, g, &DevItem::res_base)];
    const uint32_t q = g - it.res_base; /* slot within a sample */
    const DevJob &jb = rp.jobs[it.job];
    const uint32_t o = it.order ? tile_pixel(q, jb.width, jb.height) : q;
    const bool fp64 = jb.fp64 != 0;
    const uint32_t a = 3u * (jb.pixel_base + o);
    float a32[3] = {0.0f, 0.0f, 0.0f};
    double a64[3] = {0.0, 0.0, 0.0}, sq[3] = {0.0, 0.0, 0.0};
    if (!(it.flags & ITEM_FIRST))
      for (int k = 0; k < 3; k++) {
        sq[k] = rp.acc_sq[a + k];
        if (fp64) a64[k] = rp.acc64[a + k];
        else a32[k] = rp.acc32[a + k];
      }
    auto add = [&](F3 c) {
      const float v[3] = {c.x, c.y, c.z};
      for (int k = 0; k < 3; k++) {
        if (fp64) a64[k] += (double)v[k];
        else a32[k] += v[k];
        if (out_sq) sq[k] += (double)v[k] * (double)v[k];
      }
    };
    /* 8 samples are read before any is added, so that their loads are in
     * flight together */
    const F3 *p = res + it.path_base + q;
    uint32_t j = 0;
    for (; j + 8u <= it.samples; j += 8u) {
      F3 b[8];
#pragma unroll
      for (uint32_t u = 0; u < 8u; u++) b[u] = p[(size_t)(j + u) * it.pixels];
#pragma unroll
      for (uint32_t u = 0; u < 8u; u++) add(b[u]);
    }
    for (; j < it.samples; j++) add(p[(size_t)j * it.pixels]);
    if (it.flags & ITEM_LAST) {
      for (int k = 0; k < 3; k++) {
        out[a + k] = fp64 ? (float)(a64[k] / (double)jb.spp) : a32[k] / (float)jb.spp;
        if (out_sq) out_sq[a + k] = (float)(sq[k] / (double)jb.spp);
      }
    } else {
      for (int k = 0; k < 3; k++) {
        rp.acc_sq[a + k] = sq[k];
        if (fp64) rp.acc64[a + k] = a64[k];
        else rp.acc32[a + k] = a32[k];
      }
    }
  }
}

/* The tail of a pass.  From bounce `tail_depth` on, few paths are left and
 * each further bounce would cost a traversal and a shading launch for a
 * handful of rays, so one launch finishes them: every thread traces and
 * shades its path, bounce after bounce, until it ends.  It runs the same
 * traversal (lane_start / lane_node / lane_leaf, the media pass) and the same
 * shade_path as the wavefront bounces, and a path's stream and state move
 * through the same entry, so every path gives the same bytes as in the
 * wavefront.  Guided jobs sample with the plain mixture here (no lobes are
 * evaluated for these vertices); their training records are still written
 * and credited.  stats[2] counts the rays it traces. */
template <bool GUIDE, bool EXT, bool MEDIA>
__global__ __launch_bounds__(TRACE_BLOCK) void k_tail(DevScene sc, PathBuf pb, TraceArgs ta, GuideArgs ga) {
  __shared__ uint32_t lds_stack[STACK_LDS * TRACE_BLOCK];
  const uint32_t n = ta.counts[ta.in_slot];
  uint32_t *lst = lds_stack + threadIdx.x;
  uint32_t *gst = ta.spill + (size_t)(blockIdx.x * TRACE_BLOCK + threadIdx.x) * STACK_GLOBAL;
  const bool any_xform = sc.has_xforms != 0;
  ga.alpha = 0.0f; /* no lobes for tail vertices */
  uint32_t rays = 0;
  for (uint32_t i = blockIdx.x * TRACE_BLOCK + threadIdx.x; i < n; i += gridDim.x * TRACE_BLOCK) {
    for (bool first = true;; first = false) {
      if (!first) rays++; /* the entry's first ray was counted with the bounce it entered the tail in */
      Lane L;
      L.live = false;
      L.best = MISS_WORD;
      L.path = 0;
      lane_start(L, pb, i);
      while (L.word != CHILD_EMPTY) {
        if (!(L.word & CHILD_LEAF)) {
          lane_node(L, sc, lst, gst);
        } else if (lane_leaf_step(L, sc, any_xform)) {
          lane_pop(L, lst, gst);
        }
      }
      if (MEDIA) lane_media(L, sc, pb.meta[L.path], pb.rng[L.path]);
      pb.hit_t[i] = L.tb;
      pb.hit_p[i] = L.best;
      const uint32_t cls = L.best != MISS_WORD ? sc.mats[sc.info[as_u(sc.prims[L.best + 1u].w)].material].mclass : MC_MISS;
      NextPath nx;
      bool cont;
      switch (cls) {
        case MC_MISS: cont = shade_path<MC_MISS, GUIDE, EXT>(sc, pb, i, ga, nx); break;
        case MC_LIGHT: cont = shade_path<MC_LIGHT, GUIDE, EXT>(sc, pb, i, ga, nx); break;
        case MC_LAMBERTIAN: cont = shade_path<MC_LAMBERTIAN, GUIDE, EXT>(sc, pb, i, ga, nx); break;
        case MC_METAL: cont = shade_path<MC_METAL, GUIDE, EXT>(sc, pb, i, ga, nx); break;
        default: cont = shade_path<MC_GLASS, GUIDE, EXT>(sc, pb, i, ga, nx); break;
      }
      if (!cont) break;
      pb.ray_o[i] = nx.o;
      pb.ray_d[i] = nx.d;
      pb.thr[i] = nx.thr;
      pb.rng[i] = nx.rng;
      pb.meta[i] = nx.meta;
      pb.slot[i] = nx.slot;
    }
  }
  /* one atomic per wave */
  for (int off = 32; off > 0; off >>= 1) rays += __shfl_down(rays, off);
  if ((threadIdx.x & 63u) == 0 && rays) atomicAdd(ta.stats + 2, (unsigned long long)rays);
}

/* Light-traced training records of the guiding network.  A camera path
 * credits a diffuse vertex with light that came through glass only when its
 * own direction happened to hit a lamp's image, so on caustic scenes such
 * records are a few per thousand paths.  A path started at an emitter and
 * aimed at the scene's light-sampling targets (its priority objects, glass
 * included) lands on a diffuse surface after a specular chain far more often
 * -- the photon-based training of directional mixtures of Vorba et al. 2014
 * ("On-line learning of parametric mixture models for light transport
 * simulation").  Lane k serves job k mod n_jobs: an emitter among the job's
 * light-sampling leaves (uniformly, by rejection), a point on it, a direction
 * from the job's light tree (tree_sample / tree_pdf: the mixture the camera
 * paths' light half uses), a hero wavelength; the path follows metal and
 * glass with the camera paths' scatter rules at that wavelength, and its
 * first diffuse hit after at least one specular vertex becomes a record: the
 * direction back along the path, weight = emitted radiance x cos(emitter) x
 * area / pdf(direction) x the chain's attenuation -- the flux it carries up to
 * a constant.  Such hits arrive at a point distributed as L_i(w) cos(theta),
 * the density the lobes are trained towards, so the record's own density and
 * cosine are 1.  Records go to rec/recL[base + k]; recL = 0 where none. */
#define PH_MAX_BOUNCES 16
#define PH_EMITTER_TRIES 16
/* free lanes a wave waits for before it starts new light paths */
#define PH_REFILL 24u
/* whether a light-sampling leaf starts light paths: a plain emitter */
__device__ __forceinline__ bool ph_emitter(const DevScene &sc, uint32_t l) {
  const DevMaterial &m = sc.mats[sc.lights[l].mat];
  return m.mclass == MC_LIGHT && !m.cone && m.emit_spd >= 0;
}
/* A wave works through its own range of light paths: a path's length varies
 * from one bounce to 16, so each turn of the loop is one bounce of every lane,
 * and lanes whose path has ended start the next ones of the range together.
 * Most of a start goes into the light tree's density, and with many
 * light-sampling targets few of them emit: a single job's emitters are looked
 * up once per wave instead of at every try.  2^20 paths on the prism (15
 * targets, 2 of them emitters): 941 us with one path per thread and launch, 903
 * so (1065 refilling every free lane, 891 from 36 on), 503 with the record
 * counts in copies (k_guide_cell_fold). */
__global__ __launch_bounds__(TRACE_BLOCK) void k_guide_photons(DevScene sc, uint32_t n_jobs, GuideRec *rec,
                                                               float *recL, uint32_t n, uint32_t stamp, uint32_t round,
                                                               uint64_t seed, uint32_t *spill, uint32_t *fresh,
                                                               uint32_t copies) {
  __shared__ uint32_t lds_stack[STACK_LDS * TRACE_BLOCK];
  uint32_t *lst = lds_stack + threadIdx.x;
  uint32_t *gst = spill + (size_t)(blockIdx.x * TRACE_BLOCK + threadIdx.x) * STACK_GLOBAL;
  uint32_t *cells = fresh + (size_t)(blockIdx.x % copies) * n_jobs * GD_CELLS; /* this block's copy of the counts */
  const bool any_xform = sc.has_xforms != 0;
  const uint32_t waves = gridDim.x * (TRACE_BLOCK / 64), wave = blockIdx.x * (TRACE_BLOCK / 64) + (threadIdx.x >> 6);
  uint32_t next = (uint32_t)((uint64_t)n * wave / waves);
  const uint32_t end = (uint32_t)((uint64_t)n * (wave + 1u) / waves);
  /* bit l: leaf l of the only job emits */
  const bool masked = n_jobs == 1u && sc.jobs[0].n_lights <= 64u;
  uint64_t emitters = 0;
  if (masked) emitters = __ballot(__lane_id() < sc.jobs[0].n_lights && ph_emitter(sc, sc.jobs[0].light_base + __lane_id()));
  bool alive = false, specular = false;
  uint32_t k = 0, job = 0, hero = 0, bounce = 0;
  uint64_t s = 0;
  float T = 0.0f, time = 0.0f;
  V o = mk(0.0f, 0.0f, 0.0f), d = o;
  for (;;) {
    const uint64_t idle = __ballot(!alive);
    if (next < end && (uint32_t)__popcll(idle) >= PH_REFILL) {
      const uint32_t id = next + __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
      next += (uint32_t)__popcll(idle);
      if (!alive && id < end) {
        k = id;
        job = k % n_jobs;
        const DevJob &jb = sc.jobs[job];
        s = pcg_for_path(seed ^ 0xA0761D6478BD642Full, k, round); /* the render's seed and round */
        uint32_t li = 0xFFFFFFFFu;
        if (jb.guiding && jb.n_lights)
          for (int t = 0; t < PH_EMITTER_TRIES; t++) {
            const uint32_t leaf = min((uint32_t)(rnd(s) * (float)jb.n_lights), jb.n_lights - 1u);
            if (masked ? ((emitters >> leaf) & 1u) != 0u : ph_emitter(sc, jb.light_base + leaf)) {
              li = jb.light_base + leaf;
              break;
            }
          }
        T = 0.0f;
        if (li != 0xFFFFFFFFu) {
          const DevLight &E = sc.lights[li];
          V pe, ne;
          float area;
          if (E.type == PT_SPHERE) {
            const float r = E.u[0];
            ne = random_unit_vector(s);
            pe = mk(E.q[0], E.q[1], E.q[2]) + r * ne;
            area = 4.0f * PI_F * r * r;
          } else {
            float a = rnd(s), b = rnd(s);
            if (E.type == PT_TRI && a + b > 1.0f) {
              a = 1.0f - a;
              b = 1.0f - b;
            }
            pe = mk(E.q[0], E.q[1], E.q[2]) + a * mk(E.u[0], E.u[1], E.u[2]) + b * mk(E.v[0], E.v[1], E.v[2]);
            ne = mk(E.n[0], E.n[1], E.n[2]);
            area = E.w[3];
          }
          hero = (uint32_t)(((uint64_t)pcg_next(s) * 400ull) >> 32);
          time = rnd(s);
          d = unit(tree_sample(sc, jb, pe, s));
          const float pd = tree_pdf(sc, jb, pe, d);
          T = sc.spd[sc.mats[E.mat].emit_spd + hero] * dot(d, ne) * area / pd;
          o = pe;
          specular = false;
          bounce = 0;
        }
        alive = T > 0.0f && isfinite(T);
        if (!alive) recL[k] = 0.0f;
      }
      continue; /* until enough lanes have a path, or the range is used up */
    }
    if (!__any(alive)) break;
    if (alive) {
      float carried = 0.0f;
      bool ends = true;
      Lane L;
      lane_start_ray(L, o, d, time, sc.jobs[job].root);
      while (L.word != CHILD_EMPTY) {
        if (!(L.word & CHILD_LEAF)) {
          lane_node(L, sc, lst, gst);
        } else if (lane_leaf_step(L, sc, any_xform)) {
          lane_pop(L, lst, gst);
        }
      }
      if (L.best != MISS_WORD) {
        const Hit h = hit_record<false>(sc, L.best, o, d, time, L.tb);
        const DevMaterial &m = sc.mats[h.material];
        if (m.mclass == MC_METAL || m.mclass == MC_GLASS) {
          const float kk = m.albedo_spd >= 0 ? sc.spd[m.albedo_spd + hero] : 1.0f;
          const float tf = m.thin_film ? interference(m, d, h.n, CLV_LAMBDA_MIN + (int)hero) : 1.0f;
          T *= kk * tf;
          d = m.mclass == MC_METAL ? specular_dir<true>(m, d, h, hero, s) : specular_dir<false>(m, d, h, hero, s);
          o = h.p;
          specular = true;
          bounce++;
          ends = !(bounce < PH_MAX_BOUNCES && T > 0.0f && isfinite(T));
        } else if (m.mclass == MC_LAMBERTIAN && m.kind != CLV_MAT_ISOTROPIC && specular) {
          GuideRec r;
          gd_norm_pos(sc.jobs[job], h.p, r.p);
          r.n[0] = h.n.x;
          r.n[1] = h.n.y;
          r.n[2] = h.n.z;
          const V back = -unit(d);
          r.d[0] = back.x;
          r.d[1] = back.y;
          r.d[2] = back.z;
          r.lam = (float)hero / 400.0f;
          r.pdf = 1.0f;
          r.cosv = 1.0f;
          r.t0 = 1.0f;
          r.src = GD_SRC_LIGHT;
          r.stamp = stamp;
          r.pad = 0u;
          rec[k] = r;
          carried = T;
          if (isfinite(T) && T > 0.0f) /* the gate's evidence: integer counts, so the result is deterministic */
            atomicAdd(cells + (size_t)job * GD_CELLS + gd_cell(r.p), 1u);
        }
      }
      if (ends) {
        recL[k] = isfinite(carried) && carried > 0.0f ? carried : 0.0f;
        alive = false;
      }
    }
  }
}

/* Learned-proposal lobes for every guided path of the Lambertian queue.
 * Resident blocks of 8 waves stage the fp16 weights and the biases in LDS
 * once (one copy serves 8 waves, so 4 waves per SIMD fit), then every wave
 * loops over the queue on its own, 64 paths at a time: one lane per path
 * reconstructs the hit (position normalised to the job's scene box, oriented
 * normal, hero wavelength); the wave runs the MLP on MFMA for its 64 paths,
 * 16 at a time, and 4 lanes per path decode 2 lobes each straight to the
 * lobe buffer.  A wave exchanges data only through its own LDS slices, so
 * the loop has no block barrier: a wave's LDS accesses complete in order, and
 * gi_wave_sync keeps the compiler from moving them across an exchange. */
#define GI_OG 52 /* LDS row stride (floats) of one tile's outputs */
#define GI_WAVES 8
#define GI_BLOCK (64 * GI_WAVES)
__device__ __forceinline__ void gi_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__global__ __launch_bounds__(GI_BLOCK) void k_guide_infer(DevScene sc, PathBuf pb, GuideArgs ga, const uint32_t *queue,
                                                          const uint32_t *count) {
  /* W1..W4 row-major with rows padded to GD_WLD halfs (bank-conflict-free A operands) */
  __shared__ __attribute__((aligned(16))) _Float16 wl[(3 * GD_HID + GD_OUT_PAD) * GD_WLD];
  __shared__ float bl[GD_HID * 3 + GD_OUT_PAD];
  __shared__ float rin[GI_WAVES][64][8];
  __shared__ float og[GI_WAVES][16 * GI_OG];
  {
    /* 8 uint4 per 64-half row; row i of the stacked W1..W4 goes to LDS row i */
    const uint4 *src = reinterpret_cast<const uint4 *>(ga.Wh);
    for (uint32_t k = threadIdx.x; k < GD_H_WT(0) / 8u; k += GI_BLOCK)
      *reinterpret_cast<uint4 *>(wl + (k >> 3) * GD_WLD + (k & 7u) * 8u) = src[k];
    for (uint32_t k = threadIdx.x; k < GD_HID * 3u + GD_OUT_PAD; k += GI_BLOCK) {
      const uint32_t l = k / GD_HID;
      bl[k] = ga.P[l == 0 ? GD_B1 + k : (l == 1 ? GD_B2 + k - GD_HID : (l == 2 ? GD_B3 + k - 2 * GD_HID
                                                                                 : GD_B4 + k - 3 * GD_HID))];
    }
  }
  __syncthreads(); /* the weights are shared by the block's waves */
  const uint32_t n = *count;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  uint32_t evals = 0;
  for (uint32_t base = blockIdx.x * GI_BLOCK + 64u * (uint32_t)w; base < n; base += gridDim.x * GI_BLOCK) {
    const uint32_t qi = base + lane;
    uint32_t path = 0xFFFFFFFFu;
    float in[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (qi < n) {
      const uint32_t pth = queue[qi];
      const uint32_t meta = pb.meta[pth];
      const DevJob &jb = sc.jobs[meta >> META_JOB_SHIFT];
      const float4 o4 = pb.ray_o[pth], d4 = pb.ray_d[pth];
      const float t = pb.hit_t[pth];
      if (jb.guiding && gd_gate_open(ga, jb, meta >> META_JOB_SHIFT, o4, d4, t)) { /* as the shading kernel decides */
        path = pth;
        const Hit h = hit_record<false>(sc, pb.hit_p[pth], xyz(o4), xyz(d4), d4.w, t);
        gd_norm_pos(jb, h.p, in);
        in[3] = h.n.x;
        in[4] = h.n.y;
        in[5] = h.n.z;
        in[6] = (float)(meta & META_HERO_MASK) / 400.0f;
      }
    }
    /* the vertices to evaluate, compacted to the front of the wave's rows; the
     * tiles past them are skipped */
    const uint64_t am = __ballot(path != 0xFFFFFFFFu);
    const uint32_t cnt = (uint32_t)__popcll(am);
    if (path != 0xFFFFFFFFu) {
      const uint32_t row = (uint32_t)__popcll(am & ((1ull << lane) - 1ull));
#pragma unroll
      for (int k = 0; k < 7; k++) rin[w][row][k] = in[k];
      rin[w][row][7] = __uint_as_float(path);
    }
    if ((uint32_t)lane >= cnt) {
#pragma unroll
      for (int k = 0; k < 7; k++) rin[w][lane][k] = 0.0f;
      rin[w][lane][7] = __uint_as_float(0xFFFFFFFFu);
    }
    evals += cnt;
    gi_wave_sync();
    const int tiles = (int)((cnt + 15u) / 16u);
#pragma unroll 1
    for (int nt = 0; nt < tiles; nt++) {
      const int q = 16 * nt + r;
      {
        const float p[3] = {rin[w][q][0], rin[w][q][1], rin[w][q][2]};
        const float nn[3] = {rin[w][q][3], rin[w][q][4], rin[w][q][5]};
        gh4 x[4];
        gf4 out[3];
        gd_encode(p, nn, rin[w][q][6], x);
        gd_forward_tile_lds(wl, bl, x, out);
#pragma unroll
        for (int mt = 0; mt < 3; mt++)
#pragma unroll
          for (int k = 0; k < 4; k++) og[w][r * GI_OG + 16 * mt + 4 * g + k] = out[mt][k];
      }
      gi_wave_sync();
      const uint32_t pth = __float_as_uint(rin[w][q][7]);
      if (pth != 0xFFFFFFFFu) {
        /* lane g encodes lobes 2g, 2g+1 of path pth.  The softmax's max and sum
         * and the fp16 probabilities' sum come from the path's 4 lanes
         * (r, r + 16, r + 32, r + 48) by exchanges; the last lobe's probability
         * is what the others' (fp16) ones leave */
        const float *o = &og[w][r * GI_OG];
        const float l0 = o[5 * (2 * g) + 4], l1 = o[5 * (2 * g + 1) + 4];
        float mx = fmaxf(l0, l1);
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float e0 = expf(l0 - mx), e1 = expf(l1 - mx);
        float sum = e0 + e1;
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        float wd[2];
        wd[0] = (float)(_Float16)(e0 / sum);
        wd[1] = g == 3 ? 0.0f : (float)(_Float16)(e1 / sum);
        float part = wd[0] + wd[1];
        part += __shfl_xor(part, 16);
        part += __shfl_xor(part, 32);
        if (g == 3) wd[1] = fmaxf(1.0f - part, 0.0f);
        uint32_t v[2 * GD_LSTRIDE];
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int j = 2 * g + h;
          const float a = o[5 * j], b = o[5 * j + 1], c = o[5 * j + 2];
          const bool ok = sqrtf(a * a + b * b + c * c) > 1e-12f;
          const _Float16 kh = (_Float16)expf(gd_clamp_logk(o[5 * j + 3]));
          const _Float16 wh = (_Float16)wd[h];
          v[GD_LSTRIDE * h + 0] = ok ? gd_oct_encode(a, b, c) : gd_oct_encode(0.0f, 0.0f, 1.0f);
          v[GD_LSTRIDE * h + 1] = (uint32_t)__builtin_bit_cast(uint16_t, kh) |
                                  ((uint32_t)__builtin_bit_cast(uint16_t, wh) << 16);
          v[GD_LSTRIDE * h + 2] = __float_as_uint(wd[h] * gd_vmf_norm((float)kh));
        }
        uint2 *dst = reinterpret_cast<uint2 *>(ga.lobes + (size_t)pth * GD_LWORDS + 2 * GD_LSTRIDE * g);
        dst[0] = make_uint2(v[0], v[1]);
        dst[1] = make_uint2(v[2], v[3]);
        dst[2] = make_uint2(v[4], v[5]);
      }
      gi_wave_sync();
    }
  }
  if (lane == 0 && evals && ga.stats) atomicAdd(ga.stats + 3, (unsigned long long)evals);
}

/* ------------------------------------------------------- debug modes --- */
/* One camera ray per pixel through the pixel's corner (x/W, y/H) with no lens
 * offset, as render_pixel_normalmap / _bvhtestcount / _primitivetestcount
 * (draw_cpu.rs:148-207); the pixel's stream draws the wavelength, then the time. */
__global__ __launch_bounds__(256) void k_generate_debug(DevScene sc, PathBuf pb, DebugArgs da) {
  const uint32_t W = da.width, H = da.height, n = W * H;
  const DevJob &jb = sc.jobs[0];
  const DevCamera &c = jb.cam;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const uint32_t r = i / W, x = i - r * W, y = H - 1u - r;
    uint64_t s = pcg_for_path(jb.seed, x + y * W, da.sample);
    const uint32_t wl = (uint32_t)(((uint64_t)pcg_next(s) * 400ull) >> 32);
    const float time = rnd(s);
    const float u = (float)x / (float)W, v = (float)y / (float)H;
    V org = mk(c.origin[0], c.origin[1], c.origin[2]);
    V dir = mk(c.llc[0], c.llc[1], c.llc[2]) + u * mk(c.horizontal[0], c.horizontal[1], c.horizontal[2]) +
            v * mk(c.vertical[0], c.vertical[1], c.vertical[2]) - org;
    dir = unit(dir);
    pb.ray_o[i] = make_float4(org.x, org.y, org.z, __uint_as_float(jb.root));
    pb.ray_d[i] = make_float4(dir.x, dir.y, dir.z, time);
    pb.meta[i] = wl;   /* job 0 */
    pb.rng[i] = s;     /* the stream state a medium's free flight is keyed by */
  }
}

/* normal_to_color (normals.rs:21-33) of the first hit, or the count ramp of
 * bvh_testcount_to_color / primitive_testcount_to_color
 * (debug_visualizations.rs:17-33, 45-61), as linear sRGB -> Xyz<E> */
__global__ __launch_bounds__(256) void k_debug_color(DevScene sc, PathBuf pb, DebugArgs da, const uint32_t *rc,
                                                     float *out) {
  const uint32_t n = da.width * da.height;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    float r, g, b;
    if (da.mode == 1u) {
      const uint32_t off = pb.hit_p[i];
      if (off == MISS_WORD) {
        r = g = b = 0.0f;
      } else {
        const float4 o4 = pb.ray_o[i], d4 = pb.ray_d[i];
        const Hit h = hit_record<false>(sc, off, xyz(o4), xyz(d4), d4.w, pb.hit_t[i]);
        const float nx = -h.n.x, ny = h.n.y, nz = -h.n.z;
        r = 0.5f + 0.5f * nx;
        g = 0.5f + 0.5f * ny;
        b = nz < 0.0f ? 0.0f : nz;
      }
    } else {
      const uint32_t k = rc[2u * i + (da.mode == 3u ? 1u : 0u)];
      if (k <= 255u) r = g = b = (float)k / 255.0f;
      else if (k <= 511u) r = 1.0f, g = 1.0f, b = 0.0f;
      else if (k <= 1023u) r = 1.0f, g = 0.5f, b = 0.0f;
      else r = 1.0f, g = 0.0f, b = 0.0f;
    }
    const float *m = da.lin_to_xyz;
#pragma unroll
    for (int k = 0; k < 3; k++) out[3u * i + k] = m[3 * k] * r + m[3 * k + 1] * g + m[3 * k + 2] * b;
  }
}

/* per-sample estimator (draw_cpu.rs:130-142) and per-pixel sums in sample
 * order; one thread per (pass item, pixel) */
__global__ __launch_bounds__(256) void k_resolve(PathBuf pb, ResolveParams rp, const float4 *cie) {
  const DevJob *jobs = rp.jobs;
  for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < rp.threads; g += gridDim.x * blockDim.x) {
    const DevItem it = rp.items[find_entry(rp.items, rp.n_items, g, &DevItem::res_base)];
    if (it.flags & ITEM_WARMUP) continue; /* training samples only */
    const uint32_t q = g - it.res_base; /* slot within a sample */
    const DevJob &jb = jobs[it.job];
    const uint32_t o = it.order ? tile_pixel(q, jb.width, jb.height) : q;
    const bool fp64 = jb.fp64 != 0;
    const uint32_t a = 3u * (jb.pixel_base + o);
    float a32[3];
    double a64[3], sq[3];
    for (int k = 0; k < 3; k++) {
      sq[k] = rp.acc_sq[a + k];
      if (fp64) a64[k] = rp.acc64[a + k];
      else a32[k] = rp.acc32[a + k];
    }
    auto add = [&](float4 L, uint32_t hero) {
      float c[3];
      sample_xyz(cie, L, hero, c);
      for (int k = 0; k < 3; k++) {
        if (fp64) a64[k] += (double)c[k];
        else a32[k] += c[k];
        sq[k] += (double)c[k] * (double)c[k];
      }
    };
    /* the samples' path states are read 4 at a time before any is added, so
     * that their loads are in flight together */
    uint32_t j = 0;
    for (; j + 4u <= it.samples; j += 4u) {
      float4 Lb[4];
      uint32_t hb[4];
#pragma unroll
      for (uint32_t u = 0; u < 4u; u++) {
        const uint32_t i = it.path_base + (j + u) * it.pixels + q;
        Lb[u] = pb.rad[i];
        hb[u] = pb.hero[i];
      }
#pragma unroll
      for (uint32_t u = 0; u < 4u; u++) add(Lb[u], hb[u]);
    }
    for (; j < it.samples; j++) {
      const uint32_t i = it.path_base + j * it.pixels + q;
      add(pb.rad[i], pb.hero[i]);
    }
    for (int k = 0; k < 3; k++) {
      rp.acc_sq[a + k] = sq[k];
      if (fp64) rp.acc64[a + k] = a64[k];
      else rp.acc32[a + k] = a32[k];
    }
  }
}

/* per-pixel means of every job (pixels of job j start at jobs[j].pixel_base) */
__global__ void k_finalize(ResolveParams rp, float *out, float *out_sq) {
  for (uint32_t o = blockIdx.x * blockDim.x + threadIdx.x; o < rp.pixels * 3u; o += gridDim.x * blockDim.x) {
    const DevJob &jb = rp.jobs[find_entry(rp.jobs, rp.n_jobs, o / 3u, &DevJob::pixel_base)];
    out[o] = jb.fp64 ? (float)(rp.acc64[o] / (double)jb.spp) : rp.acc32[o] / (float)jb.spp;
    if (out_sq) out_sq[o] = (float)(rp.acc_sq[o] / (double)jb.spp);
  }
}

__global__ void k_zero_accum(ResolveParams rp) {
  for (uint32_t o = blockIdx.x * blockDim.x + threadIdx.x; o < rp.pixels * 3u; o += gridDim.x * blockDim.x) {
    rp.acc_sq[o] = 0.0;
    rp.acc64[o] = 0.0;
    rp.acc32[o] = 0.0f;
  }
}

/* ---------------------------------------------------------- launchers --- */
static inline uint32_t grid_for(uint32_t n, uint32_t block, uint32_t cap) {
  uint32_t g = (n + block - 1) / block;
  if (g < 1) g = 1;
  return g < cap ? g : cap;
}

void launch_reset_counts(hipStream_t st, uint32_t *counts, uint32_t in_slot, uint32_t out_slot, uint64_t *stats) {
  hipLaunchKernelGGL(k_reset_counts, dim3(1), dim3(64), 0, st, counts, in_slot, out_slot, (unsigned long long *)stats);
}
void launch_copy_out(hipStream_t st, const void *src, void *dst, size_t bytes, uint32_t *flags, uint32_t stamp,
                     const uint64_t *stats, uint64_t *stats_out) {
  hipLaunchKernelGGL(k_copy_out, dim3((uint32_t)((bytes + COPY_CHUNK - 1) / COPY_CHUNK)), dim3(CO_THREADS), 0, st,
                     (const uint32_t *)src, (uint32_t *)dst, (uint64_t)(bytes / 4), flags, stamp, stats, stats_out);
}

void launch_zero_u64(hipStream_t st, uint64_t *p, uint32_t n) {
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, st, p, n);
}

void launch_set_count(hipStream_t st, uint32_t *counts, uint32_t slot, uint32_t value) {
  hipLaunchKernelGGL(k_set_count, dim3(1), dim3(64), 0, st, counts, slot, value);
}
void launch_generate(hipStream_t st, const DevScene &sc, const PathBuf &pb, const GenParams &gp) {
  hipLaunchKernelGGL(k_generate, dim3(grid_for(gp.paths, 256, 65535)), dim3(256), 0, st, sc, pb, gp);
}
static uint32_t g_trace_blocks = 0;

uint32_t trace_grid_blocks() {
  if (g_trace_blocks) return g_trace_blocks;
  int dev = 0, cus = 0, per_cu = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(k_trace_simple<false, MODE_EXTEND, ORDER_BOTH>),
                                                      TRACE_BLOCK, 0);
  if (cus < 1) cus = 1;
  if (per_cu < 1) per_cu = 1;
  g_trace_blocks = (uint32_t)(cus * per_cu);
  return g_trace_blocks;
}

size_t trace_spill_words(uint32_t blocks) { return (size_t)blocks * TRACE_BLOCK * STACK_GLOBAL; }

size_t lds_trace_bytes(uint32_t nodes, uint32_t units) {
  return (size_t)nodes * sizeof(Bvh4Node) + (size_t)units * 16u + (size_t)LT_STACK_LDS * LT_BLOCK * 4u;
}
uint32_t lds_trace_stack_bytes() { return LT_STACK_LDS * LT_BLOCK * 4u; }
size_t lds_trace_spill_words(uint32_t blocks) { return (size_t)blocks * LT_BLOCK * LT_STACK_GLOBAL; }

uint32_t lds_trace_grid_blocks(size_t lds_bytes) {
  int dev = 0, cus = 0, per_cu = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(k_trace_lds<false, 0>),
                                                      LT_BLOCK, lds_bytes);
  if (cus < 1) cus = 1;
  if (per_cu < 1) per_cu = 1;
  return (uint32_t)(cus * per_cu);
}

void launch_trace_lds(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta, uint32_t blocks,
                      size_t lds_bytes, bool counting, int mode) {
  if (sc.has_media) { /* the host plans media batches with the plain traversal; this only keeps them correct */
    if (mode == 1)
      hipLaunchKernelGGL((k_trace_simple<false, MODE_PRIMARY, ORDER_BOTH, true>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc,
                         pb, ta);
    else if (counting)
      hipLaunchKernelGGL((k_trace_simple<true, MODE_EXTEND, ORDER_BOTH, true>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb,
                         ta);
    else
      hipLaunchKernelGGL((k_trace_simple<false, MODE_EXTEND, ORDER_BOTH, true>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc,
                         pb, ta);
    return;
  }
  if (mode == 1)
    hipLaunchKernelGGL((k_trace_lds<false, 1>), dim3(blocks), dim3(LT_BLOCK), lds_bytes, st, sc, pb, ta);
  else if (counting)
    hipLaunchKernelGGL((k_trace_lds<true, 0>), dim3(blocks), dim3(LT_BLOCK), lds_bytes, st, sc, pb, ta);
  else
    hipLaunchKernelGGL((k_trace_lds<false, 0>), dim3(blocks), dim3(LT_BLOCK), lds_bytes, st, sc, pb, ta);
}

void launch_extend(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta, uint32_t blocks,
                   bool counting, int variant) {
  if (sc.has_media) {
    if (counting)
      hipLaunchKernelGGL((k_trace_simple<true, MODE_EXTEND, ORDER_BOTH, true>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb,
                         ta);
    else
      hipLaunchKernelGGL((k_trace_simple<false, MODE_EXTEND, ORDER_BOTH, true>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc,
                         pb, ta);
  } else if (variant == TRACE_PERSISTENT) {
    if (counting)
      hipLaunchKernelGGL((k_trace<true, MODE_EXTEND>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
    else
      hipLaunchKernelGGL((k_trace<false, MODE_EXTEND>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
  } else if (variant == TRACE_MAJORITY && !counting) {
    hipLaunchKernelGGL((k_trace_simple<false, MODE_EXTEND, ORDER_MAJORITY>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
  } else if (variant == TRACE_WW) {
    if (counting)
      hipLaunchKernelGGL((k_trace_simple<true, MODE_EXTEND, ORDER_WW>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
    else
      hipLaunchKernelGGL((k_trace_simple<false, MODE_EXTEND, ORDER_WW>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
  } else {
    if (counting)
      hipLaunchKernelGGL((k_trace_simple<true, MODE_EXTEND, ORDER_BOTH>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
    else
      hipLaunchKernelGGL((k_trace_simple<false, MODE_EXTEND, ORDER_BOTH>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
  }
}

void launch_primary(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta, uint32_t blocks,
                    int variant) {
  if (sc.has_media)
    hipLaunchKernelGGL((k_trace_simple<false, MODE_PRIMARY, ORDER_BOTH, true>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb,
                       ta);
  else if (variant == TRACE_PERSISTENT)
    hipLaunchKernelGGL((k_trace<false, MODE_PRIMARY>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
  else
    hipLaunchKernelGGL((k_trace_simple<false, MODE_PRIMARY, ORDER_BOTH>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
}
void launch_generate_debug(hipStream_t st, const DevScene &sc, const PathBuf &pb, const DebugArgs &da) {
  hipLaunchKernelGGL(k_generate_debug, dim3(grid_for(da.width * da.height, 256, 8192)), dim3(256), 0, st, sc, pb, da);
}
void launch_primary_counting(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta,
                             uint32_t blocks) {
  if (sc.has_media)
    hipLaunchKernelGGL((k_trace_simple<true, MODE_PRIMARY, ORDER_BOTH, true>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb,
                       ta);
  else
    hipLaunchKernelGGL((k_trace_simple<true, MODE_PRIMARY, ORDER_BOTH>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta);
}
void launch_debug_color(hipStream_t st, const DevScene &sc, const PathBuf &pb, const DebugArgs &da,
                        const uint32_t *ray_counts, float *out) {
  hipLaunchKernelGGL(k_debug_color, dim3(grid_for(da.width * da.height, 256, 8192)), dim3(256), 0, st, sc, pb, da,
                     ray_counts, out);
}
/* The shading kernel's blocks walk the bounce's chunks in a grid-stride loop
 * with the same number of steps each, so a grid larger than what fits on the
 * device at once runs a second, partly empty round; the grid is capped at the
 * resident blocks of the instance launched (queried at context creation). */
void shade_grid_blocks(uint32_t out[4]) {
  int dev = 0, cus = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const void *fn[4] = {reinterpret_cast<const void *>(k_shade<false, false>),
                       reinterpret_cast<const void *>(k_shade<false, true>),
                       reinterpret_cast<const void *>(k_shade<true, false>),
                       reinterpret_cast<const void *>(k_shade<true, true>)};
  for (int k = 0; k < 4; k++) {
    int per_cu = 0;
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn[k], 256, 0);
    out[k] = (uint32_t)std::max(1, per_cu) * (uint32_t)std::max(1, cus);
  }
}

void launch_shade(hipStream_t st, const DevScene &sc, const PathBuf &pb, const ShadeQueues &sq, uint32_t *counts,
                  uint32_t out_slot, uint32_t max_paths, uint32_t grid_cap, const uint32_t resident[4],
                  const GuideArgs &ga) {
  const uint32_t inst = (ga.on ? 2u : 0u) + (sc.has_ext ? 1u : 0u);
  uint32_t g = grid_for(max_paths + 64u * MC_COUNT, 256, std::min(grid_cap, resident[inst]));
  if (ga.on && sc.has_ext)
    hipLaunchKernelGGL((k_shade<true, true>), dim3(g), dim3(256), 0, st, sc, pb, sq, counts, out_slot, ga);
  else if (ga.on)
    hipLaunchKernelGGL((k_shade<true, false>), dim3(g), dim3(256), 0, st, sc, pb, sq, counts, out_slot, ga);
  else if (sc.has_ext)
    hipLaunchKernelGGL((k_shade<false, true>), dim3(g), dim3(256), 0, st, sc, pb, sq, counts, out_slot, ga);
  else
    hipLaunchKernelGGL((k_shade<false, false>), dim3(g), dim3(256), 0, st, sc, pb, sq, counts, out_slot, ga);
}
void launch_tail(hipStream_t st, const DevScene &sc, const PathBuf &pb, const TraceArgs &ta, uint32_t blocks,
                 const GuideArgs &ga) {
#define CLV_TAIL(G, E, M) hipLaunchKernelGGL((k_tail<G, E, M>), dim3(blocks), dim3(TRACE_BLOCK), 0, st, sc, pb, ta, ga)
  const bool g = ga.on != 0, e = sc.has_ext != 0, m = sc.has_media != 0;
  if (g) {
    if (e) { if (m) CLV_TAIL(true, true, true); else CLV_TAIL(true, true, false); }
    else { if (m) CLV_TAIL(true, false, true); else CLV_TAIL(true, false, false); }
  } else {
    if (e) { if (m) CLV_TAIL(false, true, true); else CLV_TAIL(false, true, false); }
    else { if (m) CLV_TAIL(false, false, true); else CLV_TAIL(false, false, false); }
  }
#undef CLV_TAIL
}

/* resident blocks of the light-traced records' kernel on the current device */
uint32_t guide_photon_grid_blocks() {
  int per_cu = 0, dev = 0, cus = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_guide_photons, TRACE_BLOCK, 0);
  return (uint32_t)std::max(1, per_cu) * (uint32_t)std::max(1, cus);
}
void launch_guide_photons(hipStream_t st, const DevScene &sc, uint32_t n_jobs, GuideRec *rec, float *recL, uint32_t n,
                          uint32_t stamp, uint32_t round, uint64_t seed, uint32_t *spill, uint32_t blocks,
                          uint32_t *fresh, uint32_t copies) {
  if (n == 0 || n_jobs == 0) return;
  hipLaunchKernelGGL(k_guide_photons, dim3(std::min(blocks, grid_for(n, TRACE_BLOCK, 1u << 30))), dim3(TRACE_BLOCK), 0,
                     st, sc, n_jobs, rec, recL, n, stamp, round, seed, spill, fresh, copies);
}

/* A round's record counts come in `copies` copies (launch_guide_photons):
 * caustics put most of a round's records in a few cells, and adds to one
 * address from all over the device wait for each other (half of the
 * light-traced round with one copy, 2^20 paths on the prism).  Here the copies
 * are added to the counts so far and to the job totals, and cleared.  A block
 * covers GF_PER cells of one job. */
#define GF_PER 4096u
__global__ __launch_bounds__(256) void k_guide_cell_fold(uint32_t *fresh, uint32_t copies, uint32_t n_jobs, uint32_t *cells,
                                                         uint32_t *cell_tot) {
  __shared__ uint32_t part[4];
  const size_t first = (size_t)blockIdx.x * GF_PER, stride = (size_t)n_jobs * GD_CELLS;
  uint32_t acc = 0;
  for (uint32_t c = threadIdx.x * 4u; c < GF_PER; c += 1024u) {
    uint4 sum = make_uint4(0u, 0u, 0u, 0u);
    for (uint32_t r = 0; r < copies; r++) {
      uint4 *p = reinterpret_cast<uint4 *>(fresh + r * stride + first + c);
      const uint4 v = *p;
      if (v.x | v.y | v.z | v.w) *p = make_uint4(0u, 0u, 0u, 0u);
      sum.x += v.x;
      sum.y += v.y;
      sum.z += v.z;
      sum.w += v.w;
    }
    if (sum.x | sum.y | sum.z | sum.w) {
      uint4 *q = reinterpret_cast<uint4 *>(cells + first + c);
      const uint4 v = *q;
      *q = make_uint4(v.x + sum.x, v.y + sum.y, v.z + sum.z, v.w + sum.w);
      acc += sum.x + sum.y + sum.z + sum.w;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
  if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t t = part[0] + part[1] + part[2] + part[3];
    if (t) atomicAdd(cell_tot + first / GD_CELLS, t);
  }
}

/* the gate: a cell is open if the records in it and its 26 neighbours, per
 * cell, reach `density` times what its job's records would leave per cell
 * spread evenly over one GD_GRID x GD_GRID plane of the grid -- where
 * light arrives through glass concentrated, not the thin spread of glass
 * reflections -- or if the job received no records at all */
__global__ __launch_bounds__(256) void k_guide_gate(const uint32_t *cells, const uint32_t *cell_tot, uint8_t *gate,
                                                    uint32_t n_jobs, float density) {
  const size_t n = (size_t)n_jobs * GD_CELLS;
  for (size_t i = (size_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (size_t)gridDim.x * 256u) {
    const uint32_t job = (uint32_t)(i / GD_CELLS), c = (uint32_t)(i % GD_CELLS);
    const uint32_t x = c % GD_GRID, y = (c / GD_GRID) % GD_GRID, z = c / (GD_GRID * GD_GRID);
    const uint32_t *jc = cells + (size_t)job * GD_CELLS;
    const uint32_t tot = cell_tot[job];
    uint32_t sum = 0;
    for (int dz = -1; dz <= 1; dz++)
      for (int dy = -1; dy <= 1; dy++)
        for (int dx = -1; dx <= 1; dx++) {
          const int xx = (int)x + dx, yy = (int)y + dy, zz = (int)z + dz;
          if (xx < 0 || yy < 0 || zz < 0 || xx >= (int)GD_GRID || yy >= (int)GD_GRID || zz >= (int)GD_GRID) continue;
          sum += jc[((uint32_t)zz * GD_GRID + (uint32_t)yy) * GD_GRID + (uint32_t)xx];
        }
    const bool open = tot == 0u || (sum > 0u && (float)sum / 27.0f >= density * (float)tot / (float)(GD_GRID * GD_GRID));
    gate[i] = open ? 1u : 0u;
  }
}
void launch_guide_gate(hipStream_t st, uint32_t *fresh, uint32_t copies, uint32_t *cells, uint32_t *cell_tot,
                       uint8_t *gate, uint32_t n_jobs, float density) {
  const size_t n = (size_t)n_jobs * GD_CELLS;
  hipLaunchKernelGGL(k_guide_cell_fold, dim3((uint32_t)(n / GF_PER)), dim3(256), 0, st, fresh, copies, n_jobs, cells, cell_tot);
  hipLaunchKernelGGL(k_guide_gate, dim3((uint32_t)std::min<size_t>((n + 255u) / 256u, 16384u)), dim3(256), 0, st, cells,
                     cell_tot, gate, n_jobs, density);
}

/* resident blocks of the inference kernel on the current device (each block
 * stages the weights once); queried at context creation, so that a launch
 * sequence under stream capture makes no device queries */
uint32_t guide_infer_grid_blocks() {
  int per_cu = 0, dev = 0, cus = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_guide_infer, GI_BLOCK, 0);
  return (uint32_t)std::max(1, per_cu) * (uint32_t)std::max(1, cus);
}

void launch_guide_infer(hipStream_t st, const DevScene &sc, const PathBuf &pb, const GuideArgs &ga,
                        const uint32_t *queue, const uint32_t *count, uint32_t max_paths, uint32_t resident) {
  hipLaunchKernelGGL(k_guide_infer, dim3(std::min(resident, grid_for(max_paths, GI_BLOCK, 1u << 30))), dim3(GI_BLOCK), 0,
                     st, sc, pb, ga, queue, count);
}

/* k_paths: blocks of 8 waves that share a scene in LDS, or of 2 that read it from memory */
#define PS_BLOCK_LDS 512
#define PS_BLOCK_GLOBAL 128
uint32_t paths_block(bool full) { return full ? PS_BLOCK_LDS : PS_BLOCK_GLOBAL; }
size_t paths_lds_bytes(bool full, uint32_t nodes, uint32_t units) {
  return (size_t)nodes * sizeof(Bvh4Node) + (size_t)units * 16u + (size_t)PS_WORDS * paths_block(full) * 4u;
}
size_t paths_spill_words(bool full, uint32_t blocks) {
  return (size_t)blocks * paths_block(full) * (TRAV_TOTAL - PS_WORDS);
}

typedef void (*paths_fn)(DevScene, GenParams, PathsArgs);
template <int BLOCK, bool FULL, bool XF>
static paths_fn paths_instance_of(bool ext, bool media) {
  if (media) return k_paths<BLOCK, true, true, FULL, XF>; /* a medium's phase function is an extended material */
  return ext ? k_paths<BLOCK, true, false, FULL, XF> : k_paths<BLOCK, false, false, FULL, XF>;
}
static paths_fn paths_instance(const DevScene &sc, bool full) {
  const bool ext = sc.has_ext != 0, media = sc.has_media != 0, xf = sc.has_xforms != 0;
  if (full)
    return xf ? paths_instance_of<PS_BLOCK_LDS, true, true>(ext, media) : paths_instance_of<PS_BLOCK_LDS, true, false>(ext, media);
  return xf ? paths_instance_of<PS_BLOCK_GLOBAL, false, true>(ext, media)
            : paths_instance_of<PS_BLOCK_GLOBAL, false, false>(ext, media);
}
uint32_t paths_grid_blocks(size_t lds_bytes, const DevScene &sc, bool full) {
  int dev = 0, cus = 0, per_cu = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(paths_instance(sc, full)),
                                                     (int)paths_block(full), lds_bytes);
  return (uint32_t)std::max(1, per_cu) * (uint32_t)std::max(1, cus);
}
void launch_paths(hipStream_t st, const DevScene &sc, const GenParams &gp, const PathsArgs &pa, uint32_t blocks,
                  size_t lds_bytes, bool begin) {
  hipLaunchKernelGGL(k_paths_begin, dim3(1), dim3(64), 0, st, pa.next, blocks * pa.first, begin ? pa.stats : nullptr);
  hipLaunchKernelGGL(paths_instance(sc, pa.full != 0), dim3(blocks),
                     dim3(paths_block(pa.full != 0)), lds_bytes, st, sc, gp, pa);
}
void launch_resolve_xyz(hipStream_t st, const ResolveParams &rp, const F3 *res, float *out, float *out_sq) {
  hipLaunchKernelGGL(k_resolve_xyz, dim3(grid_for(rp.threads, 256, 65535)), dim3(256), 0, st, rp, res, out, out_sq);
}

void launch_resolve(hipStream_t st, const PathBuf &pb, const ResolveParams &rp, const float4 *cie) {
  hipLaunchKernelGGL(k_resolve, dim3(grid_for(rp.threads, 256, 65535)), dim3(256), 0, st, pb, rp, cie);
}
void launch_finalize(hipStream_t st, const ResolveParams &rp, float *out, float *out_sq) {
  hipLaunchKernelGGL(k_finalize, dim3(grid_for(rp.pixels * 3u, 256, 65535)), dim3(256), 0, st, rp, out, out_sq);
}
void launch_zero_accum(hipStream_t st, const ResolveParams &rp) {
  hipLaunchKernelGGL(k_zero_accum, dim3(grid_for(rp.pixels * 3u, 256, 65535)), dim3(256), 0, st, rp);
}

/* ------------------------------------------ allocation-free hit probe --- */
/* The device memory of clv_primary_hits_noalloc: one array per GPU, held
 * until the process ends.  It carries the job and pass-item tables, the
 * counters, the path state of NA_CHUNK camera rays, a distance buffer for
 * callers that want no distances, and the traversal stack overflow of an
 * NA_BLOCKS-block grid.  Host code never takes the array's name as an
 * address: na_scratch_address() asks the runtime for the current device's
 * copy (once per context, at clv_create), and every kernel and copy uses
 * that pointer. */
constexpr size_t na_round(size_t x) { return (x + 255u) & ~(size_t)255u; }
constexpr size_t NA_OFF_JOB = 0;
constexpr size_t NA_OFF_ITEM = NA_OFF_JOB + na_round(sizeof(DevJob));
constexpr size_t NA_OFF_COUNTS = NA_OFF_ITEM + na_round(sizeof(DevItem));
constexpr size_t NA_OFF_RAY_O = NA_OFF_COUNTS + na_round(CNT_TOTAL * 4u);
constexpr size_t NA_OFF_RAY_D = NA_OFF_RAY_O + 16u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_THR = NA_OFF_RAY_D + 16u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_RAD = NA_OFF_THR + 16u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_RNG = NA_OFF_RAD + 16u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_META = NA_OFF_RNG + 8u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_SLOT = NA_OFF_META + 4u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_HERO = NA_OFF_SLOT + 4u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_HIT_T = NA_OFF_HERO + 4u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_HIT_P = NA_OFF_HIT_T + 4u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_TS = NA_OFF_HIT_P + 4u * (size_t)NA_CHUNK;
constexpr size_t NA_OFF_SPILL = NA_OFF_TS + 4u * (size_t)NA_CHUNK;
constexpr size_t NA_BYTES = NA_OFF_SPILL + 4u * (size_t)NA_BLOCKS * TRACE_BLOCK * STACK_GLOBAL;
static_assert(NA_BYTES == NA_SCRATCH_BYTES, "NA_SCRATCH_BYTES in kernels.h must match the scratch layout");

static __device__ __align__(256) unsigned char scratch[NA_SCRATCH_BYTES];

int na_scratch_address(void **out) {
  *out = nullptr;
  return hipGetSymbolAddress(out, HIP_SYMBOL(scratch)) == hipSuccess && *out ? 0 : -1;
}

NaView na_view(void *base) {
  char *b = static_cast<char *>(base);
  NaView v = NaView();
  v.job = reinterpret_cast<DevJob *>(b + NA_OFF_JOB);
  v.item = reinterpret_cast<DevItem *>(b + NA_OFF_ITEM);
  v.counts = reinterpret_cast<uint32_t *>(b + NA_OFF_COUNTS);
  v.ts = reinterpret_cast<float *>(b + NA_OFF_TS);
  v.spill = reinterpret_cast<uint32_t *>(b + NA_OFF_SPILL);
  PathBuf &pb = v.pb;
  pb.ray_o = pb.n_ray_o = reinterpret_cast<float4 *>(b + NA_OFF_RAY_O);
  pb.ray_d = pb.n_ray_d = reinterpret_cast<float4 *>(b + NA_OFF_RAY_D);
  pb.thr = pb.n_thr = reinterpret_cast<float4 *>(b + NA_OFF_THR);
  pb.rad = reinterpret_cast<float4 *>(b + NA_OFF_RAD);
  pb.rng = pb.n_rng = reinterpret_cast<uint64_t *>(b + NA_OFF_RNG);
  pb.meta = pb.n_meta = reinterpret_cast<uint32_t *>(b + NA_OFF_META);
  pb.slot = pb.n_slot = reinterpret_cast<uint32_t *>(b + NA_OFF_SLOT);
  pb.hero = reinterpret_cast<uint32_t *>(b + NA_OFF_HERO);
  pb.hit_t = reinterpret_cast<float *>(b + NA_OFF_HIT_T);
  pb.hit_p = reinterpret_cast<uint32_t *>(b + NA_OFF_HIT_P);
  return v;
}

/* the job and the chunk's pass item come in as kernel arguments (no copy
 * from host memory), the counters start at zero */
__global__ void k_na_setup(DevJob jb, DevItem it, DevJob *job, DevItem *item, uint32_t *counts) {
  if (threadIdx.x == 0) {
    *job = jb;
    *item = it;
  }
  if (threadIdx.x < CNT_TOTAL) counts[threadIdx.x] = 0u;
}

void launch_na_setup(hipStream_t st, const DevJob &jb, const DevItem &it, const NaView &v) {
  hipLaunchKernelGGL(k_na_setup, dim3(1), dim3(64), 0, st, jb, it, v.job, v.item, v.counts);
}

}  // namespace clv
