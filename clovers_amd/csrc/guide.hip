/*
 * guide.hip -- online training of the guiding network (see guide.h).
 *
 * After every wavefront pass of a guided render:
 *   k_guide_count / k_guide_scan / k_guide_scatter
 *       compact the pass' training records with a radiance sample (L > 0)
 *       into a list, in slot order (deterministic), and compute their mean
 *       MC weight F/p;
 *   k_guide_train (per step)
 *       four waves per group of 64 records: forward on MFMA, d(loss)/d(outputs)
 *       per record, backward on MFMA; every group writes its summed parameter
 *       gradient to its own slice of a partial buffer (no atomics);
 *   k_guide_adam (per step)
 *       sums the slices in group order, Adam update of the fp32 master
 *       parameters, refresh of the fp16 operand copies.
 * k_guide_eval and the gradient mode of k_guide_adam serve the C ABI's
 * network probes (clv_guide_eval, clv_guide_grad).
 */
#include <hip/hip_runtime.h>
#include <math.h>

#include "guide.h"
#include "kernels.h"

namespace clv {

#define GT_LD 72     /* LDS row stride (halfs) of activation tiles: 64 + 8 against bank conflicts */
#define GT_OG 49     /* LDS row stride (floats) of output / gradient rows */

/* The back-propagated gradients go through fp16 (MFMA operands), whose
 * largest finite value is 65504: a record with a large weight F/p and a
 * sharp lobe (the gradient grows with kappa, up to ~5000) overflows it, and
 * one inf turns the whole network into NaN.  So each group of 64 records holds its fp16
 * gradients in units of 2^se, a power of two chosen per layer from the
 * group's largest magnitude so that it lands in [2^(GT_TOP-1), 2^GT_TOP);
 * partial sums leave it multiplied by 2^-se, which is exact. */
#define GT_TOP 12
#define GT_EMAX 100

__device__ __forceinline__ float gt_wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}

/* the exponent for values whose largest magnitude is m, held in units 2^se */
__device__ __forceinline__ int gt_exponent(float m, int se) {
  if (!(m > 0.0f) || !isfinite(m)) return se;
  int e;
  frexpf(m, &e); /* m in [2^(e-1), 2^e) */
  return min(max(se + GT_TOP - e, -GT_EMAX), GT_EMAX);
}

/* a record of this pass with radiance (recL is zeroed when the pass starts
 * and when a record is written); the record itself is read only then.
 * *light: the record comes from a light-traced path */
__device__ __forceinline__ bool rec_valid(const GuideRec *rec, const float *recL, uint32_t i, float *w, bool *light) {
  const float L = recL[i];
  if (!(L > 0.0f && isfinite(L))) return false;
  const GuideRec &r = rec[i];
  if (!(r.pdf > 0.0f && isfinite(r.pdf) && r.t0 > 0.0f)) return false;
  *w = L * r.cosv / r.pdf;
  *light = r.src == GD_SRC_LIGHT;
  return true;
}

/* ---------------------------------------------------------- compaction --- */
/* each block covers GC_PER consecutive records, 256 at a time, so the scan
 * has few block counts to add up */
#define GC_PER 4096u
/* per block of GC_PER records: valid records (bcount[b]), of them from
 * light-traced paths (bcount[nb + b]), and the weight sums of the camera and
 * the light-traced ones (bweight[2b], bweight[2b + 1]) */
__global__ __launch_bounds__(256) void k_guide_count(const GuideRec *rec, const float *recL, uint32_t n,
                                                     uint32_t *bcount, float *bweight) {
  __shared__ uint32_t sc[2][256];
  __shared__ float sw[2][256];
  uint32_t c = 0, cl = 0;
  float w = 0.0f, wl = 0.0f;
  for (uint32_t k = 0; k < GC_PER; k += 256u) {
    const uint32_t i = blockIdx.x * GC_PER + k + threadIdx.x;
    float wt;
    bool light;
    if (i < n && rec_valid(rec, recL, i, &wt, &light)) {
      c++;
      if (light) {
        cl++;
        wl += wt;
      } else {
        w += wt;
      }
    }
  }
  sc[0][threadIdx.x] = c;
  sc[1][threadIdx.x] = cl;
  sw[0][threadIdx.x] = w;
  sw[1][threadIdx.x] = wl;
  __syncthreads();
  for (uint32_t s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      for (int q = 0; q < 2; q++) {
        sc[q][threadIdx.x] += sc[q][threadIdx.x + s];
        sw[q][threadIdx.x] += sw[q][threadIdx.x + s];
      }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    bcount[blockIdx.x] = sc[0][0];
    bcount[gridDim.x + blockIdx.x] = sc[1][0];
    bweight[2 * blockIdx.x] = sw[0][0];
    bweight[2 * blockIdx.x + 1] = sw[1][0];
  }
}

/* one block: exclusive scan of the block counts; totals[0] = valid records,
 * totals[1] / totals[2] = the mean weight of the camera / light-traced ones
 * (as float bits): each source's weights are used relative to their own mean */
__global__ __launch_bounds__(1024) void k_guide_scan(uint32_t *bcount, const float *bweight, uint32_t nb,
                                                     uint32_t *totals, uint32_t cap, unsigned long long *used) {
  __shared__ uint32_t part[1024];
  __shared__ double wpart[1024], wlpart[1024];
  const uint32_t per = (nb + 1023u) / 1024u;
  const uint32_t b0 = threadIdx.x * per, b1 = min(nb, b0 + per);
  uint32_t s = 0, sl = 0;
  double w = 0.0, wl = 0.0;
  for (uint32_t b = b0; b < b1; b++) {
    s += bcount[b];
    sl += bcount[nb + b];
    w += (double)bweight[2 * b];
    wl += (double)bweight[2 * b + 1];
  }
  wpart[threadIdx.x] = w;
  wlpart[threadIdx.x] = wl;
  /* the counts' exclusive prefix by waves; the weights are added one after
   * the other (their order is part of the result), each source by a thread of
   * its own beside that: 23 -> 9 us, most of it that chain of additions */
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t pre = s, lpre = sl;
#pragma unroll
  for (uint32_t k = 1; k < 64u; k <<= 1) {
    const uint32_t u = __shfl_up(pre, k), lu = __shfl_up(lpre, k);
    if (lane >= k) {
      pre += u;
      lpre += lu;
    }
  }
  __shared__ uint32_t wsum[16], lwsum[16];
  if (lane == 63u) {
    wsum[wave] = pre;
    lwsum[wave] = lpre;
  }
  __syncthreads();
  uint32_t base = 0, all = 0, lall = 0;
  for (uint32_t k = 0; k < 16u; k++) {
    if (k < wave) base += wsum[k];
    all += wsum[k];
    lall += lwsum[k];
  }
  part[threadIdx.x] = base + pre - s;
  if (threadIdx.x == 0 || threadIdx.x == 64) {
    const double *src = threadIdx.x == 0 ? wpart : wlpart;
    const uint32_t cnt = threadIdx.x == 0 ? all - lall : lall;
    double acc = 0.0;
#pragma unroll 16
    for (uint32_t t = 0; t < 1024u; t++) acc += src[t];
    totals[threadIdx.x == 0 ? 1 : 2] = __float_as_uint(cnt ? (float)(acc / (double)cnt) : 0.0f);
  }
  if (threadIdx.x == 128) {
    totals[0] = all;
    if (used) *used += (unsigned long long)min(all, cap);
  }
  __syncthreads();
  uint32_t run = part[threadIdx.x];
  for (uint32_t b = b0; b < b1; b++) {
    uint32_t v = bcount[b];
    bcount[b] = run;
    run += v;
  }
}

__global__ __launch_bounds__(256) void k_guide_scatter(const GuideRec *rec, const float *recL, uint32_t n,
                                                       const uint32_t *boffset, uint32_t *list) {
  __shared__ uint32_t wcount[4];
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  uint32_t off = boffset[blockIdx.x];
  for (uint32_t k = 0; k < GC_PER; k += 256u) {  /* block-uniform: chunks in record order */
    const uint32_t i = blockIdx.x * GC_PER + k + threadIdx.x;
    float wt;
    bool light;
    const bool v = i < n && rec_valid(rec, recL, i, &wt, &light);
    const uint64_t m = __ballot(v);
    if (lane == 0) wcount[w] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t o = off;
    for (uint32_t q = 0; q < w; q++) o += wcount[q];
    if (v) list[o + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = i;
    off += wcount[0] + wcount[1] + wcount[2] + wcount[3];
    __syncthreads();
  }
}

/* ------------------------------------------------------------ training --- */
/* d(-w log q)/d(outputs) of a record by the 4 lanes that share it (lane group g
 * of 16 records: lobes g and g + 4): o = the record's raw outputs, gr = the
 * gradients of the lane's two lobes, 5 each.  Sums over the lobes run in lobe
 * order on every lane. */
__device__ __forceinline__ float gd_lobe_sum(const float v[2], int r) {
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < GD_LOBES; j++) s += __shfl(v[j >> 2], r + 16 * (j & 3));
  return s;
}
__device__ void gd_loss_grad(const float *o, const float d[3], float w, int r, int g, float gr[2][5]) {
  float mx = fmaxf(o[5 * g + 4], o[5 * (g + 4) + 4]);
  mx = fmaxf(mx, __shfl_xor(mx, 16));
  mx = fmaxf(mx, __shfl_xor(mx, 32));
  float mu[2][3], kappa[2], wt[2], f[2], c[2], wf[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int j = g + 4 * h;
    const float a = o[5 * j], b = o[5 * j + 1], cc = o[5 * j + 2];
    const float len = sqrtf(a * a + b * b + cc * cc);
    const bool ok = len > 1e-12f;
    mu[h][0] = ok ? a / len : 0.0f;
    mu[h][1] = ok ? b / len : 0.0f;
    mu[h][2] = ok ? cc / len : 1.0f;
    kappa[h] = expf(gd_clamp_logk(o[5 * j + 3]));
    wt[h] = expf(o[5 * j + 4] - mx);
  }
  const float sum = gd_lobe_sum(wt, r);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    wt[h] /= sum;
    c[h] = mu[h][0] * d[0] + mu[h][1] * d[1] + mu[h][2] * d[2];
    f[h] = gd_vmf_norm(kappa[h]) * expf(kappa[h] * (c[h] - 1.0f));
    wf[h] = wt[h] * f[h];
  }
  float q = gd_lobe_sum(wf, r);
  if (!(q > 1e-30f)) q = 1e-30f;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int j = g + 4 * h;
#pragma unroll
    for (int t = 0; t < 5; t++) gr[h][t] = 0.0f;
    if (!(w > 0.0f)) continue;
    const float rr = wf[h] / q;
    const float k = kappa[h];
    gr[h][4] = -w * (rr - wt[h]);
    const float s = o[5 * j + 3];
    if (s > GD_LOGK_MIN && s < GD_LOGK_MAX) {
      const float dlogf = 1.0f / k - 2.0f / expm1f(2.0f * k) + (c[h] - 1.0f);
      gr[h][3] = -w * rr * k * dlogf;
    }
    const float a = o[5 * j], b = o[5 * j + 1], cc = o[5 * j + 2];
    const float len = sqrtf(a * a + b * b + cc * cc);
    if (len > 1e-12f) {
      const float gm[3] = {-w * rr * k * d[0], -w * rr * k * d[1], -w * rr * k * d[2]};
      const float mg = mu[h][0] * gm[0] + mu[h][1] * gm[1] + mu[h][2] * gm[2];
#pragma unroll
      for (int t = 0; t < 3; t++) gr[h][t] = (gm[t] - mu[h][t] * mg) / len;
    }
  }
}

struct GuideTrainArgs {
  const GuideRec *rec;
  const float *recL;
  const uint32_t *list;    /* compacted record slots */
  const uint32_t *totals;  /* [0] valid records, [1] mean weight (float bits) */
  uint32_t cap;            /* records used per round */
  uint32_t step_base;      /* first used record of this step */
  uint32_t step_len;       /* records per step (grid = step_len / 64) */
  float wclip;             /* weight cap in units of the mean weight */
  const _Float16 *Wh;
  const float *P;
  float *partial;          /* [group][GD_NPARAM] */
  uint32_t *steps;         /* Adam's step count, one more for a step with records (an empty step changes nothing);
                              NULL in the gradient mode */
};

/* One block = a group of 64 records, 4 waves.  Wave w carries the tile of
 * records 16w .. 16w + 15 through the forward pass, its output gradients and the
 * back-propagated rows, and rows 16w .. of every weight gradient (a contraction
 * over the 64 records of the group, read from LDS).  A step is a chain of
 * short dependent phases and 256 groups, one to a CU, so its time is the
 * latency of one group: with the group on one wave 34.1 us a step of 16,384
 * records, 27.5 on four (12 of them up to the end of the forward pass, 2 the
 * output gradients, 14 the backward pass and the 16 MB of slices).  Asking for
 * the weights' cache lines ahead changed nothing. */
__global__ __launch_bounds__(256) void k_guide_train(GuideTrainArgs a) {
  __shared__ float rin[64][12];           /* inputs (7), direction (3), weight */
  __shared__ __attribute__((aligned(16))) _Float16 H[4][64 * GT_LD]; /* activations A0..A3, [feature][record] */
  __shared__ __attribute__((aligned(16))) _Float16 DZ[64 * GT_LD];   /* back-propagated rows, [neuron][record] */
  __shared__ float OG[64 * GT_OG];        /* outputs, then their gradients, [record][48] */
  __shared__ float wmax[4];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, g = lane >> 4, q = 16 * w + r;
  const uint32_t nvalid = a.totals[0];
  const uint32_t nuse = min(nvalid, a.cap);
  if (a.steps && blockIdx.x == 0 && tid == 0 && a.step_base < nuse) *a.steps += 1u;
  if (tid < 64) {
    const uint32_t u = a.step_base + blockIdx.x * 64u + (uint32_t)tid;
    float in[7] = {0, 0, 0, 0, 0, 0, 0}, wgt = 0.0f, dir[3] = {0.0f, 0.0f, 1.0f};
    if (u < nuse) {
      const uint32_t slot = a.list[(uint32_t)(((uint64_t)u * nvalid) / nuse)];
      const GuideRec R = a.rec[slot];
      const float wmean = __uint_as_float(a.totals[R.src == GD_SRC_LIGHT ? 2 : 1]);
      wgt = wmean > 0.0f ? fminf(a.recL[slot] * R.cosv / R.pdf / wmean, a.wclip) : 0.0f;
      for (int k = 0; k < 3; k++) {
        in[k] = R.p[k];
        in[3 + k] = R.n[k];
        dir[k] = R.d[k];
      }
      in[6] = R.lam;
    }
    for (int k = 0; k < 7; k++) rin[tid][k] = in[k];
    for (int k = 0; k < 3; k++) rin[tid][7 + k] = dir[k];
    rin[tid][10] = wgt;
  }
  __syncthreads();
  /* forward; every activation to LDS */
  {
    gh4 cur[4];
    const float p[3] = {rin[q][0], rin[q][1], rin[q][2]}, n[3] = {rin[q][3], rin[q][4], rin[q][5]};
    float sin2[3];
    gd_encode(p, n, rin[q][6], cur, sin2);
    /* sin 2a = 2 sin a cos a goes to fp16 in one rounding (v_fma_mixlo), except
     * in the first layer's operands of the group's last tile, where the product
     * is rounded to fp32 before: the last bit of a feature decides a seed's
     * network and image, so each use keeps the rounding it has always had */
#pragma unroll
    for (int kt = 0; kt < 4; kt++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        _Float16 f = cur[kt][i];
        asm volatile("" : "+v"(f));
        cur[kt][i] = f;
        H[0][(16 * kt + 4 * g + i) * GT_LD + q] = f;
      }
    if (w == 3)
#pragma unroll
      for (int kt = 0; kt < 3; kt++) {
        asm volatile("" : "+v"(sin2[kt]));
        cur[kt][2] = (_Float16)sin2[kt];
      }
#pragma unroll
    for (int l = 0; l < 4; l++) {
      const int mts = l == 3 ? 3 : 4;
      const _Float16 *W = a.Wh + GD_H_W(l);
      const float *bias = a.P + (l == 0 ? GD_B1 : (l == 1 ? GD_B2 : (l == 2 ? GD_B3 : GD_B4)));
      gf4 acc[4];
#pragma unroll
      for (int mt = 0; mt < 4; mt++) {
        if (mt >= mts) break;
        gf4 c;
#pragma unroll
        for (int i = 0; i < 4; i++) c[i] = bias[16 * mt + 4 * g + i];
#pragma unroll
        for (int kt = 0; kt < 4; kt++) {
          const gh4 wa = *reinterpret_cast<const gh4 *>(W + (16 * mt + r) * 64 + 16 * kt + 4 * g);
          c = __builtin_amdgcn_mfma_f32_16x16x16f16(wa, cur[kt], c, 0, 0, 0);
        }
        acc[mt] = c;
      }
      if (l < 3) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
          cur[k] = gd_relu_h(acc[k]);
#pragma unroll
          for (int i = 0; i < 4; i++) H[l + 1][(16 * k + 4 * g + i) * GT_LD + q] = cur[k][i];
        }
      } else {
#pragma unroll
        for (int mt = 0; mt < 3; mt++)
#pragma unroll
          for (int i = 0; i < 4; i++) OG[q * GT_OG + 16 * mt + 4 * g + i] = acc[mt][i];
      }
    }
  }
  __syncthreads();
  /* output gradients of the wave's records */
  {
    float gr[2][5];
    const float dir[3] = {rin[q][7], rin[q][8], rin[q][9]};
    gd_loss_grad(&OG[q * GT_OG], dir, rin[q][10], r, g, gr);
    bool fin = true;
    float gmax = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int t = 0; t < 5; t++) {
        fin = fin && isfinite(gr[h][t]);
        gmax = fmaxf(gmax, fabsf(gr[h][t]));
      }
    /* a record whose gradient is not finite is left out */
    const uint64_t bad = __ballot(!fin);
    fin = ((bad >> r) & 0x0001000100010001ull) == 0ull;
    if (!fin) gmax = 0.0f;
    __syncthreads(); /* the outputs are read */
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int t = 0; t < 5; t++) OG[q * GT_OG + 5 * (g + 4 * h) + t] = fin ? gr[h][t] : 0.0f;
    OG[q * GT_OG + GD_OUT + 2 * g] = 0.0f; /* the padding rows */
    OG[q * GT_OG + GD_OUT + 2 * g + 1] = 0.0f;
    gmax = gt_wave_max(gmax);
    if (lane == 0) wmax[w] = gmax;
  }
  __syncthreads();
  int se = gt_exponent(fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3])), 0);
  float *part = a.partial + (size_t)blockIdx.x * GD_NPARAM;
  /* layer 4: D = output gradients (48 rows), fp16 in units of 2^se */
  gh4 din[4]; /* [k-step]: B operands of the current layer's D for the wave's records */
#pragma unroll
  for (int kt = 0; kt < 3; kt++) {
    gh4 v;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const _Float16 gv = (_Float16)ldexpf(OG[q * GT_OG + 16 * kt + 4 * g + i], se);
      v[i] = gv;
      DZ[(16 * kt + 4 * g + i) * GT_LD + q] = gv;
    }
    din[kt] = v;
  }
  if (w == 3 && lane < GD_OUT_PAD) {
    /* four independent sums, so the LDS reads are not one dependent chain */
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
#pragma unroll
    for (int k = 0; k < 64; k += 4) {
      s0 += OG[k * GT_OG + lane];
      s1 += OG[(k + 1) * GT_OG + lane];
      s2 += OG[(k + 2) * GT_OG + lane];
      s3 += OG[(k + 3) * GT_OG + lane];
    }
    part[GD_B4 + lane] = (s0 + s1) + (s2 + s3);
  }
  __syncthreads();
#pragma unroll
  for (int layer = 4; layer >= 1; layer--) {
    const int rows = layer == 4 ? GD_OUT_PAD : GD_HID;
    const int wofs = layer == 1 ? GD_W1 : (layer == 2 ? GD_W2 : (layer == 3 ? GD_W3 : GD_W4));
    /* W^T's operands for D_{layer-1}, on their way while dW is computed */
    const int kts = rows / 16, lda = rows;
    gh4 wt[4][4];
    if (layer > 1) {
      const _Float16 *WT = a.Wh + GD_H_WT(layer - 1);
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int kt = 0; kt < 4; kt++)
          if (kt < kts) wt[mt][kt] = *reinterpret_cast<const gh4 *>(WT + (16 * mt + r) * lda + 16 * kt + 4 * g);
    }
    /* dW = D . A_{layer-1}^T : M = rows (16 a wave), N = 64 features, K = 64 records */
    if (16 * w < rows) {
      gh4 av[4];
#pragma unroll
      for (int kt = 0; kt < 4; kt++) av[kt] = *reinterpret_cast<const gh4 *>(&DZ[(16 * w + r) * GT_LD + 16 * kt + 4 * g]);
#pragma unroll
      for (int nt = 0; nt < 4; nt++) {
        gf4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kt = 0; kt < 4; kt++) {
          const gh4 bv = *reinterpret_cast<const gh4 *>(&H[layer - 1][(16 * nt + r) * GT_LD + 16 * kt + 4 * g]);
          c = __builtin_amdgcn_mfma_f32_16x16x16f16(av[kt], bv, c, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) part[wofs + (16 * w + 4 * g + i) * 64 + 16 * nt + r] = ldexpf(c[i], -se);
      }
    }
    if (layer == 1) break;
    /* D_{layer-1} = (W^T . D) masked by A_{layer-1} > 0, in fp32 until the
     * group has picked its new scale */
    gf4 acc[4];
    float amax = 0.0f;
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
      gf4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kt = 0; kt < 4; kt++)
        if (kt < kts) c = __builtin_amdgcn_mfma_f32_16x16x16f16(wt[mt][kt], din[kt], c, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const bool on = (float)H[layer - 1][(16 * mt + 4 * g + i) * GT_LD + q] > 0.0f;
        const float x = on ? c[i] : 0.0f;
        c[i] = x;
        amax = fmaxf(amax, fabsf(x));
      }
      acc[mt] = c;
    }
    amax = gt_wave_max(amax);
    if (lane == 0) wmax[w] = amax;
    __syncthreads(); /* every wave is done reading DZ */
    const int se_new = gt_exponent(fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3])), se);
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
      gh4 v;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        v[i] = (_Float16)ldexpf(acc[mt][i], se_new - se);
        DZ[(16 * mt + 4 * g + i) * GT_LD + q] = v[i];
      }
      din[mt] = v;
    }
    se = se_new;
    __syncthreads();
    if (w == layer - 2) {
      const int bofs = layer == 2 ? GD_B1 : (layer == 3 ? GD_B2 : GD_B3);
      /* this lane's row of 64 records, 8 halfs per LDS read, four independent sums */
      const gh8 *row = reinterpret_cast<const gh8 *>(&DZ[lane * GT_LD]);
      float sv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < 8; c++) {
        const gh8 v = row[c];
        sv[c & 3] += (((float)v[0] + (float)v[1]) + ((float)v[2] + (float)v[3])) +
                     (((float)v[4] + (float)v[5]) + ((float)v[6] + (float)v[7]));
      }
      part[bofs + lane] = ldexpf((sv[0] + sv[1]) + (sv[2] + sv[3]), -se);
    }
  }
}

/* the gradient's sum runs over chunks of GD_RCHUNK groups, each in group
 * order, then over the chunks in order */
#define GD_RCHUNK 16u
struct GuideAdamArgs {
  float *P;
  float *m;
  float *v;
  _Float16 *Wh;
  const float *partial;     /* [group][GD_NPARAM] */
  const uint32_t *totals;
  uint32_t cap, step_base, step_len;
  float lr, beta1, beta2, eps;
  const uint32_t *steps;    /* Adam steps taken so far, this one included (bias corrections 1 - beta^t) */
  float *grad_out;          /* gradient mode: write the mean gradient here, no update */
};

__device__ __forceinline__ void refresh_half(_Float16 *Wh, uint32_t p, float val) {
  int layer, row, col, rows;
  uint32_t base;
  if (p < GD_B1) { layer = 0; base = GD_W1; rows = GD_HID; }
  else if (p >= GD_W2 && p < GD_B2) { layer = 1; base = GD_W2; rows = GD_HID; }
  else if (p >= GD_W3 && p < GD_B3) { layer = 2; base = GD_W3; rows = GD_HID; }
  else if (p >= GD_W4 && p < GD_B4) { layer = 3; base = GD_W4; rows = GD_OUT_PAD; }
  else return;
  row = (int)((p - base) / 64u);
  col = (int)((p - base) % 64u);
  Wh[GD_H_W(layer) + row * 64 + col] = (_Float16)val;
  Wh[GD_H_WT(layer) + col * rows + row] = (_Float16)val;
}

/* One step's gradient sum and Adam update: a block takes 64 parameters, wave
 * c of it the chunks c, c + 16, .. of their group slices; wave 0 adds the chunks and
 * updates.  (As two launches, with the chunk sums through memory, the pair took
 * 13.4 us a step; together 6.0.) */
__global__ __launch_bounds__(1024) void k_guide_adam(GuideAdamArgs a) {
  __shared__ float sums[16][64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, p = blockIdx.x * 64u + lane;
  const uint32_t nuse = min(a.totals[0], a.cap);
  if (a.step_base >= nuse) return; /* an empty step: no update */
  const uint32_t len = min(a.step_len, nuse - a.step_base);
  const uint32_t groups = (len + 63u) / 64u, nchunk = (groups + GD_RCHUNK - 1u) / GD_RCHUNK;
  float gsum = 0.0f;
  for (uint32_t c0 = 0; c0 < nchunk; c0 += 16u) { /* block-uniform */
    const uint32_t w0 = (c0 + wave) * GD_RCHUNK, w1 = min(groups, w0 + GD_RCHUNK);
    float s = 0.0f;
    if (p < GD_NPARAM) {
      const float *src = a.partial + (size_t)w0 * GD_NPARAM + p;
      if (w0 + GD_RCHUNK <= groups) {
        float v[GD_RCHUNK];
#pragma unroll
        for (uint32_t k = 0; k < GD_RCHUNK; k++) v[k] = src[(size_t)k * GD_NPARAM];
#pragma unroll
        for (uint32_t k = 0; k < GD_RCHUNK; k++) s += v[k];
      } else {
        for (uint32_t k = w0; k < w1; k++) s += a.partial[(size_t)k * GD_NPARAM + p];
      }
    }
    sums[wave][lane] = s;
    __syncthreads();
    if (wave == 0)
      for (uint32_t k = 0; k < min(16u, nchunk - c0); k++) gsum += sums[k][lane];
    __syncthreads();
  }
  if (wave != 0 || p >= GD_NPARAM) return;
  const float gr = gsum / (float)len;
  if (a.grad_out) {
    a.grad_out[p] = gr;
    return;
  }
  if (!isfinite(gr)) return; /* keep the parameter and its moments finite */
  const float t = (float)max(*a.steps, 1u);
  const float bc1 = 1.0f - powf(a.beta1, t), bc2 = 1.0f - powf(a.beta2, t);
  const float m = a.beta1 * a.m[p] + (1.0f - a.beta1) * gr;
  const float v = a.beta2 * a.v[p] + (1.0f - a.beta2) * gr * gr;
  a.m[p] = m;
  a.v[p] = v;
  const float val = a.P[p] - a.lr * (m / bc1) / (sqrtf(v / bc2) + a.eps);
  a.P[p] = val;
  refresh_half(a.Wh, p, val);
}

/* fp16 operand copies from the master parameters */
__global__ __launch_bounds__(256) void k_guide_halves(const float *P, _Float16 *Wh) {
  const uint32_t p = blockIdx.x * 256u + threadIdx.x;
  if (p < GD_NPARAM) refresh_half(Wh, p, P[p]);
}

/* network probe: raw outputs (40) and decoded lobes (40) of n inputs
 * (p xyz, n xyz, lambda; 7 floats each), through the rendering path's forward
 * pass (weights staged in LDS, 16x16x32 MFMAs) */
__global__ __launch_bounds__(64) void k_guide_eval(const float *in, uint32_t n, const _Float16 *Wh, const float *P,
                                                   float *raw, float *lobes) {
  __shared__ __attribute__((aligned(16))) _Float16 wl[(3 * GD_HID + GD_OUT_PAD) * GD_WLD];
  __shared__ float bl[GD_HID * 3 + GD_OUT_PAD];
  __shared__ float rin[64][8];
  __shared__ float OG[64 * GT_OG];
  const int lane = threadIdx.x, r = lane & 15, g = lane >> 4;
  {
    const uint4 *src = reinterpret_cast<const uint4 *>(Wh);
    for (uint32_t k = threadIdx.x; k < GD_H_WT(0) / 8u; k += 64u)
      *reinterpret_cast<uint4 *>(wl + (k >> 3) * GD_WLD + (k & 7u) * 8u) = src[k];
    for (uint32_t k = threadIdx.x; k < GD_HID * 3u + GD_OUT_PAD; k += 64u) {
      const uint32_t l = k / GD_HID;
      bl[k] = P[l == 0 ? GD_B1 + k : (l == 1 ? GD_B2 + k - GD_HID : (l == 2 ? GD_B3 + k - 2 * GD_HID
                                                                               : GD_B4 + k - 3 * GD_HID))];
    }
  }
  const uint32_t i = blockIdx.x * 64u + (uint32_t)lane;
  for (int k = 0; k < 7; k++) rin[lane][k] = i < n ? in[7 * (size_t)i + k] : 0.0f;
  __syncthreads();
  for (int nt = 0; nt < 4; nt++) {
    const int q = 16 * nt + r;
    const float p[3] = {rin[q][0], rin[q][1], rin[q][2]}, nn[3] = {rin[q][3], rin[q][4], rin[q][5]};
    gh4 x[4];
    gf4 out[3];
    gd_encode(p, nn, rin[q][6], x);
    gd_forward_tile_lds(wl, bl, x, out);
#pragma unroll
    for (int mt = 0; mt < 3; mt++)
#pragma unroll
      for (int k = 0; k < 4; k++) OG[q * GT_OG + 16 * mt + 4 * g + k] = out[mt][k];
  }
  __syncthreads();
  if (i >= n) return;
  float o[GD_OUT];
  for (int k = 0; k < GD_OUT; k++) {
    o[k] = OG[lane * GT_OG + k];
    raw[GD_OUT * (size_t)i + k] = o[k];
  }
  GdLobes L;
  gd_decode(o, L);
  for (int j = 0; j < GD_LOBES; j++) {
    float *d = lobes + GD_OUT * (size_t)i + 5 * j;
    d[0] = L.mu[j][0];
    d[1] = L.mu[j][1];
    d[2] = L.mu[j][2];
    d[3] = L.kappa[j];
    d[4] = L.w[j];
  }
}

/* ---------------------------------------------------------- launchers --- */
void launch_guide_collect(hipStream_t st, const GuideRec *rec, const float *recL, uint32_t n, uint32_t *bcount,
                          float *bweight, uint32_t *totals, uint32_t *list, uint32_t cap, unsigned long long *used) {
  const uint32_t nb = (n + GC_PER - 1u) / GC_PER;
  hipLaunchKernelGGL(k_guide_count, dim3(nb), dim3(256), 0, st, rec, recL, n, bcount, bweight);
  hipLaunchKernelGGL(k_guide_scan, dim3(1), dim3(1024), 0, st, bcount, bweight, nb, totals, cap, used);
  hipLaunchKernelGGL(k_guide_scatter, dim3(nb), dim3(256), 0, st, rec, recL, n, bcount, list);
}

void launch_guide_step(hipStream_t st, const GuideRec *rec, const float *recL, const uint32_t *list,
                       uint32_t *totals, uint32_t cap, uint32_t step_base, uint32_t step_len, float wclip,
                       float *P, float *m, float *v, _Float16 *Wh, float *partial, float lr, float *grad_out) {
  GuideTrainArgs ta;
  ta.rec = rec;
  ta.recL = recL;
  ta.list = list;
  ta.totals = totals;
  ta.cap = cap;
  ta.step_base = step_base;
  ta.step_len = step_len;
  ta.wclip = wclip;
  ta.Wh = Wh;
  ta.P = P;
  ta.partial = partial;
  ta.steps = grad_out ? nullptr : totals + 3;
  hipLaunchKernelGGL(k_guide_train, dim3((step_len + 63u) / 64u), dim3(256), 0, st, ta);
  GuideAdamArgs aa;
  aa.P = P;
  aa.m = m;
  aa.v = v;
  aa.Wh = Wh;
  aa.partial = partial;
  aa.totals = totals;
  aa.cap = cap;
  aa.step_base = step_base;
  aa.step_len = step_len;
  aa.lr = lr;
  aa.beta1 = 0.9f;
  aa.beta2 = 0.99f;
  aa.eps = 1e-8f;
  aa.steps = totals + 3;
  aa.grad_out = grad_out;
  hipLaunchKernelGGL(k_guide_adam, dim3((GD_NPARAM + 63u) / 64u), dim3(1024), 0, st, aa);
}

void launch_guide_halves(hipStream_t st, const float *P, _Float16 *Wh) {
  hipLaunchKernelGGL(k_guide_halves, dim3((GD_NPARAM + 255u) / 256u), dim3(256), 0, st, P, Wh);
}

void launch_guide_eval(hipStream_t st, const float *in, uint32_t n, const _Float16 *Wh, const float *P, float *raw,
                       float *lobes) {
  hipLaunchKernelGGL(k_guide_eval, dim3((n + 63u) / 64u), dim3(64), 0, st, in, n, Wh, P, raw, lobes);
}

}  // namespace clv
