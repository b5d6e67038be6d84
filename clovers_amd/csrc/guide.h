/*
 * guide.h -- the learned proposal of the guided sampler (device side).
 *
 * At a diffuse (Lambertian) vertex the plain method samples the reference's
 * ½ light-tree + ½ cosine mixture (clovers-cli/src/trace.rs:80-120,
 * clovers/src/pdf.rs:106-141).  The guided method keeps the light-tree half
 * and splits the cosine half: with probability alpha the direction is drawn
 * from a learned density q, otherwise from the cosine lobe, and the sample is
 * weighted by the one-sample MIS mixture pdf
 *     p(w) = ½ p_light(w) + ½ (alpha q(w) + (1 - alpha) p_cos(w)),
 * so the estimator stays unbiased whatever q is, and direct light from small
 * emitters keeps its exact area sampling.
 *
 * q is a mixture of GD_LOBES von Mises-Fisher lobes on the sphere,
 *     q(w) = sum_j pi_j * kappa_j / (2 pi (1 - exp(-2 kappa_j))) * exp(kappa_j (mu_j . w - 1)),
 * whose parameters come from a small MLP (3 hidden layers of 64, ReLU) of the
 * vertex position (normalised to the scene box, frequency-encoded), the
 * oriented normal and the hero wavelength.  The network runs on MFMA in fp16
 * with fp32 accumulation; it is trained online on the tracer's own radiance
 * samples by minimising the KL divergence from the target density
 * proportional to L_i(w) * cos(theta) (Mueller et al. 2019, "Neural Importance
 * Sampling"; vMF-mixture outputs as in Dong et al. 2023, "Neural Parametric
 * Mixtures for Path Guiding"):
 *     loss = - sum_s  (F_s / p_s) * log q(w_s),   F_s = L_s cos(theta_s).
 *
 * Matrix layout: every layer is computed transposed, out^T = W . in^T, so
 * that the MFMA result of one layer (lane l holds rows 4*(l/16)+i of column
 * l%16) is exactly the B operand of the next (lane l supplies k = 4*(l/16)+i
 * of column l%16): columns are queries, activations never leave registers in
 * the forward pass.
 */
#ifndef CLV_GUIDE_H
#define CLV_GUIDE_H
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace clv {

#define GD_IN 64        /* encoded input features */
#define GD_HID 64       /* hidden width */
#define GD_LOBES 8
#define GD_OUT 40       /* per lobe: mu (3, unnormalised), log kappa, mixture logit */
#define GD_OUT_PAD 48   /* output rows padded to whole 16-row tiles */
#define GD_PAIRS 4      /* per position axis: sin/cos of pi 2^k x for k = 2m and 2m + 1, m < 4 */

/* fp32 master parameter vector: W1 b1 W2 b2 W3 b3 W4 b4, W row-major [out][in] */
#define GD_W1 0
#define GD_B1 (GD_W1 + GD_HID * GD_IN)
#define GD_W2 (GD_B1 + GD_HID)
#define GD_B2 (GD_W2 + GD_HID * GD_HID)
#define GD_W3 (GD_B2 + GD_HID)
#define GD_B3 (GD_W3 + GD_HID * GD_HID)
#define GD_W4 (GD_B3 + GD_HID)
#define GD_B4 (GD_W4 + GD_OUT_PAD * GD_HID)
#define GD_NPARAM (GD_B4 + GD_OUT_PAD)
/* fp16 copies for the MFMA operands: W1..W4 row-major, then the transposes
 * WT1..WT4 ([in][out], used by the backward pass) */
#define GD_H_W(l) ((l) * GD_HID * GD_IN)                  /* l = 0..3; W4 has 48 rows */
#define GD_H_WT(l) (GD_H_W(3) + GD_OUT_PAD * GD_HID + (l) * GD_HID * GD_IN)
#define GD_NHALF (2 * (3 * GD_HID * GD_IN + GD_OUT_PAD * GD_HID))

#define GD_LOGK_MIN -3.0f /* kappa in [0.05, 4915] */
#define GD_LOGK_MAX 8.5f

/* a training sample: one diffuse vertex of a traced path */
struct GuideRec {
  float p[3];       /* position, normalised to the scene box ([-1, 1]^3) */
  float n[3];       /* oriented normal */
  float d[3];       /* sampled direction */
  float lam;        /* hero wavelength, (lambda - 380) / 400 */
  float pdf;        /* density the direction was drawn with */
  float cosv;       /* cos(theta) of the direction */
  float t0;         /* hero throughput right after this vertex */
  uint32_t src;     /* GD_SRC_*: a camera path's vertex, or a light-traced path's diffuse hit
                       (the radiance that arrives is kept apart, in recL) */
  uint32_t stamp;   /* pass that wrote it */
  uint32_t pad;
};                  /* 64 bytes */

#define GD_SLOTS 3  /* training records kept per path: its last 3 diffuse vertices */
#define GD_SRC_CAMERA 0u
#define GD_SRC_LIGHT 1u

/* Guiding gate: a GD_GRID^3 grid of cells over each guided job's scene box.
 * Light-traced records are counted in the cell where they land; after each
 * training round a cell is open if it or one of its 26 neighbours holds any,
 * or if the job received none at all.  A diffuse vertex in a closed cell
 * samples the plain mixture and the network is not evaluated for it: the
 * guide's share alpha becomes a function of position, fixed before the
 * vertex samples, so the one-sample MIS estimator stays unbiased. */
#define GD_GRID 64u
#define GD_CELLS (GD_GRID * GD_GRID * GD_GRID)

/* cell of a position normalised to the scene box ([-1, 1]^3) */
__device__ __forceinline__ uint32_t gd_cell(const float p[3]) {
  uint32_t c[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const float f = (p[a] + 1.0f) * (0.5f * (float)GD_GRID);
    c[a] = (uint32_t)fminf(fmaxf(f, 0.0f), (float)(GD_GRID - 1u));
  }
  return (c[2] * GD_GRID + c[1]) * GD_GRID + c[0];
}

typedef _Float16 gh4 __attribute__((ext_vector_type(4)));
typedef float gf4 __attribute__((ext_vector_type(4)));

#define GD_PI 3.14159265358979323846f

/* Input features of a query, in 16 cells of 4: feature 4c + i.
 *   c < 12:  axis c % 3, a = pi 2^(2 (c / 3)) x_axis:   sin a, cos a, sin 2a, cos 2a
 *            (8 octaves per position axis)
 *   c = 12:  a = pi lambda:                             sin a, cos a, sin 2a, cos 2a
 *   c = 13:  a = 4 pi lambda:                           the same
 *   c = 14:  p_x, p_y, p_z, 1
 *   c = 15:  n_x, n_y, n_z, lambda
 * (lambda = (wavelength - 380) / 400).  Lane group g of a wave supplies the
 * cells 4 kt + g of its query (k-step kt of the first layer's B operand), so
 * every lane computes one angle per cell with the same instructions: a
 * hardware sine and cosine (which take revolutions and reduce them exactly:
 * |a| / 2 pi <= 32 here) and the double angle from them (one rounding each,
 * below the features' fp16 precision). */
__device__ __forceinline__ void gd_encode(const float p[3], const float n[3], float lam, gh4 x[4],
                                          float *sin2 = nullptr /* sin 2a of the position cells, in fp32 */) {
  const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int kt = 0; kt < 4; kt++) {
    const int c = 4 * kt + g;
    float rev;
    if (kt < 3) {
      const int ax = c % 3;
      const float xa = ax == 0 ? p[0] : (ax == 1 ? p[1] : p[2]);
      rev = xa * (float)(1 << (2 * (c / 3))) * 0.5f;
    } else {
      rev = lam * (g == 0 ? 0.5f : 2.0f);
    }
    const float sn = __builtin_amdgcn_sinf(rev), cs = __builtin_amdgcn_cosf(rev);
    float v0 = sn, v1 = cs, v2 = 2.0f * sn * cs, v3 = 1.0f - 2.0f * sn * sn;
    if (sin2 && kt < 3) sin2[kt] = v2;
    if (kt == 3 && g >= 2) {
      v0 = g == 2 ? p[0] : n[0];
      v1 = g == 2 ? p[1] : n[1];
      v2 = g == 2 ? p[2] : n[2];
      v3 = g == 2 ? 1.0f : lam;
    }
    gh4 v;
    v[0] = (_Float16)v0;
    v[1] = (_Float16)v1;
    v[2] = (_Float16)v2;
    v[3] = (_Float16)v3;
    x[kt] = v;
  }
}

/* out^T[16*MT x 16] = W[16*MT x 64] . in^T[64 x 16] + b: W fp16 row-major with
 * 64 columns, b fp32.  acc[mt] lane l: rows 16 mt + 4 (l/16) + i, column l%16. */
template <int MT>
__device__ __forceinline__ void gd_gemm(const _Float16 *__restrict__ W, const float *__restrict__ b, const gh4 in[4],
                                        gf4 acc[MT]) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    gf4 c;
#pragma unroll
    for (int i = 0; i < 4; i++) c[i] = b[16 * mt + 4 * g + i];
#pragma unroll
    for (int kt = 0; kt < 4; kt++) {
      const gh4 a = *reinterpret_cast<const gh4 *>(W + (16 * mt + r) * 64 + 16 * kt + 4 * g);
      c = __builtin_amdgcn_mfma_f32_16x16x16f16(a, in[kt], c, 0, 0, 0);
    }
    acc[mt] = c;
  }
}

__device__ __forceinline__ gh4 gd_relu_h(gf4 v) {
  gh4 h;
#pragma unroll
  for (int i = 0; i < 4; i++) h[i] = (_Float16)fmaxf(v[i], 0.0f);
  return h;
}

/* forward pass of one 16-query tile: x = encoded inputs (B layout); out = the
 * 48 output rows (rows 40..47 are padding); hidden activations optionally
 * returned (h[layer][kt], fp16, B layout) */
__device__ __forceinline__ void gd_forward_tile(const _Float16 *__restrict__ Wh, const float *__restrict__ P,
                                                const gh4 x[4], gf4 out[3], gh4 (*hid)[4]) {
  gh4 cur[4], nxt[4];
#pragma unroll
  for (int k = 0; k < 4; k++) cur[k] = x[k];
#pragma unroll
  for (int l = 0; l < 3; l++) {
    gf4 acc[4];
    const int boff = l == 0 ? GD_B1 : (l == 1 ? GD_B2 : GD_B3);
    gd_gemm<4>(Wh + GD_H_W(l), P + boff, cur, acc);
#pragma unroll
    for (int k = 0; k < 4; k++) nxt[k] = gd_relu_h(acc[k]);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      cur[k] = nxt[k];
      if (hid) hid[l][k] = nxt[k];
    }
  }
  gd_gemm<3>(Wh + GD_H_W(3), P + GD_B4, cur, out);
}

/* the forward pass with weights (W1..W4 stacked row-major, rows padded to
 * GD_WLD halfs) and biases (b1 b2 b3 b4) staged in LDS */
#define GD_WLD 72
/* The 64-deep contractions run as two 16x16x32 MFMAs.  Within a 32-deep step
 * s, the k positions a lane group supplies are taken as rows
 * {32 s + 4 g + i} and {32 s + 16 + 4 g + i} (i < 4) -- exactly what the lane
 * holds of the previous layer's tiles 2s and 2s+1 -- and the weights are read
 * in the same order, so the activations still never leave registers. */
typedef _Float16 gh8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ gh8 gd_cat(gh4 lo, gh4 hi) {
  gh8 v;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    v[i] = lo[i];
    v[4 + i] = hi[i];
  }
  return v;
}
__device__ __forceinline__ void gd_forward_tile_lds(const _Float16 *W, const float *b, const gh4 x[4], gf4 out[3],
                                                    gh4 (*hid)[4] = nullptr) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  gh4 cur[4];
#pragma unroll
  for (int k = 0; k < 4; k++) cur[k] = x[k];
#pragma unroll
  for (int l = 0; l < 4; l++) {
    const int mts = l == 3 ? 3 : 4;
    gf4 acc[4];
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
      if (mt >= mts) break;
      gf4 c;
#pragma unroll
      for (int i = 0; i < 4; i++) c[i] = b[GD_HID * l + 16 * mt + 4 * g + i];
      const _Float16 *wrow = W + (GD_HID * l + 16 * mt + r) * GD_WLD + 4 * g;
#pragma unroll
      for (int st = 0; st < 2; st++) {
        const gh8 a = gd_cat(*reinterpret_cast<const gh4 *>(wrow + 32 * st), *reinterpret_cast<const gh4 *>(wrow + 32 * st + 16));
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, gd_cat(cur[2 * st], cur[2 * st + 1]), c, 0, 0, 0);
      }
      acc[mt] = c;
    }
    if (l < 3) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        cur[k] = gd_relu_h(acc[k]);
        if (hid) hid[l][k] = cur[k];
      }
    } else {
#pragma unroll
      for (int k = 0; k < 3; k++) out[k] = acc[k];
    }
  }
}

/* decoded lobe parameters of one query: mu (unit), kappa, mixture weight */
struct GdLobes {
  float mu[GD_LOBES][3];
  float kappa[GD_LOBES];
  float w[GD_LOBES];
};

__device__ __forceinline__ float gd_clamp_logk(float s) { return fminf(fmaxf(s, GD_LOGK_MIN), GD_LOGK_MAX); }

__device__ __forceinline__ void gd_decode(const float o[GD_OUT], GdLobes &L) {
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < GD_LOBES; j++) mx = fmaxf(mx, o[5 * j + 4]);
  float sum = 0.0f;
#pragma unroll
  for (int j = 0; j < GD_LOBES; j++) {
    const float a = o[5 * j], b = o[5 * j + 1], c = o[5 * j + 2];
    const float len = sqrtf(a * a + b * b + c * c);
    if (len > 1e-12f) {
      L.mu[j][0] = a / len;
      L.mu[j][1] = b / len;
      L.mu[j][2] = c / len;
    } else {
      L.mu[j][0] = 0.0f;
      L.mu[j][1] = 0.0f;
      L.mu[j][2] = 1.0f;
    }
    L.kappa[j] = expf(gd_clamp_logk(o[5 * j + 3]));
    L.w[j] = expf(o[5 * j + 4] - mx);
    sum += L.w[j];
  }
#pragma unroll
  for (int j = 0; j < GD_LOBES; j++) L.w[j] /= sum;
}

/* normalisation of a vMF lobe on S^2: kappa / (2 pi (1 - exp(-2 kappa))) */
__device__ __forceinline__ float gd_vmf_norm(float k) { return k / (2.0f * GD_PI * -expm1f(-2.0f * k)); }

/* stored lobes of a query, GD_LSTRIDE 32-bit words per lobe (96 bytes a
 * query): the mean direction on an octahedral map in two 16-bit fixed-point
 * coordinates (Cigolle et al. 2014, "A Survey of Efficient Representations
 * for Independent Unit Vectors"), kappa and the probability of choosing the
 * lobe as fp16, and that probability x the lobe's normalisation in fp32.
 * Sampling and the density both use the decoded values, so they describe
 * one distribution exactly. */
#define GD_LSTRIDE 3
#define GD_LWORDS (GD_LOBES * GD_LSTRIDE)

__device__ __forceinline__ uint32_t gd_oct_encode(float x, float y, float z) {
  const float s = fabsf(x) + fabsf(y) + fabsf(z);
  float u = x / s, v = y / s;
  if (z < 0.0f) {
    const float uu = (1.0f - fabsf(v)) * copysignf(1.0f, u);
    v = (1.0f - fabsf(u)) * copysignf(1.0f, v);
    u = uu;
  }
  const uint32_t qu = (uint32_t)rintf(fminf(fmaxf(u * 0.5f + 0.5f, 0.0f), 1.0f) * 65535.0f);
  const uint32_t qv = (uint32_t)rintf(fminf(fmaxf(v * 0.5f + 0.5f, 0.0f), 1.0f) * 65535.0f);
  return qu | (qv << 16);
}

__device__ __forceinline__ void gd_oct_decode(uint32_t w, float &x, float &y, float &z) {
  float u = (float)(w & 0xFFFFu) * (2.0f / 65535.0f) - 1.0f;
  float v = (float)(w >> 16) * (2.0f / 65535.0f) - 1.0f;
  const float zz = 1.0f - fabsf(u) - fabsf(v);
  const float t = fmaxf(-zz, 0.0f);
  u += u >= 0.0f ? -t : t;
  v += v >= 0.0f ? -t : t;
  const float inv = 1.0f / sqrtf(u * u + v * v + zz * zz);
  x = u * inv;
  y = v * inv;
  z = zz * inv;
}

__device__ __forceinline__ float gd_half_lo(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu)); }
__device__ __forceinline__ float gd_half_hi(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)); }

/* q(w) of stored lobes */
__device__ __forceinline__ float gd_pdf(const uint32_t *lob, float dx, float dy, float dz) {
  float q = 0.0f;
#pragma unroll
  for (int j = 0; j < GD_LOBES; j++) {
    const uint32_t *l = lob + GD_LSTRIDE * j;
    float mx, my, mz;
    gd_oct_decode(l[0], mx, my, mz);
    const float c = mx * dx + my * dy + mz * dz;
    q += __uint_as_float(l[2]) * expf(gd_half_lo(l[1]) * (c - 1.0f));
  }
  return q;
}

/* draw a direction from the stored lobes with three uniforms: lobe choice,
 * then Jakob 2012 ("Numerically stable sampling of the von Mises Fisher
 * distribution on S^2"): cos = 1 + log(u1 + (1 - u1) exp(-2 kappa)) / kappa */
__device__ __forceinline__ void gd_sample(const uint32_t *lob, float u0, float u1, float u2, float &dx, float &dy,
                                          float &dz) {
  int j = GD_LOBES - 1;
  float acc = 0.0f;
#pragma unroll
  for (int k = 0; k < GD_LOBES - 1; k++) {
    acc += gd_half_hi(lob[GD_LSTRIDE * k + 1]);
    if (u0 < acc) { j = k; break; }
  }
  const uint32_t *l = lob + GD_LSTRIDE * j;
  const float k = gd_half_lo(l[1]);
  float w = 1.0f + logf(u1 + (1.0f - u1) * expf(-2.0f * k)) / k;
  w = fminf(fmaxf(w, -1.0f), 1.0f);
  const float s = sqrtf(fmaxf(0.0f, 1.0f - w * w));
  const float phi = 2.0f * GD_PI * u2;
  const float vx = s * cosf(phi), vy = s * sinf(phi);
  /* frame around mu (Duff et al. 2017 branchless orthonormal basis) */
  float mx, my, mz;
  gd_oct_decode(l[0], mx, my, mz);
  const float sg = copysignf(1.0f, mz);
  const float a = -1.0f / (sg + mz);
  const float bb = mx * my * a;
  const float t1x = 1.0f + sg * mx * mx * a, t1y = sg * bb, t1z = -sg * mx;
  const float t2x = bb, t2y = sg + my * my * a, t2z = -my;
  dx = vx * t1x + vy * t2x + w * mx;
  dy = vx * t1y + vy * t2y + w * my;
  dz = vx * t1z + vy * t2z + w * mz;
  const float len = sqrtf(dx * dx + dy * dy + dz * dz);
  dx /= len;
  dy /= len;
  dz /= len;
}

}  // namespace clv
#endif
