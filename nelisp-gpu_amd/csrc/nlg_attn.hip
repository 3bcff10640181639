// nlg_attn.hip -- attention on the reference's f32 layouts.
//
//   decode-attn / decode-attn-b (kernels.el:315-390): single-query causal GQA
//     over cached K/V.  The reference spends one invocation per output
//     element and recomputes every q.k product hd times; here a workgroup
//     owns one (sequence, head): each wave takes every 4th position, its 64
//     lanes split the head dimension (coalesced 512-byte K/V rows at hd=128),
//     the q.k product is one DPP reduction, and the four waves' running
//     (z, ctx) are merged through LDS.
//   attn-causal-gqa (kernels.el:934-990): 32-query tiles on the f32 matrix
//     cores; one wave per (head, query) for the forms those do not take.
//   attn-scores / attn-context (kernels.el:205-235): per element, serial in
//     the reference's order (bit-identical up to the 1/sqrt(hd) scale).
// Every access is bounds-checked (reads past a buffer give 0, writes are
// dropped) because POS comes from device memory.
#include <math.h>

#include "nlg_internal.h"

#define NEG_BIG (-1.0e30f)

struct AB {
  const float *p;
  uint32_t n;
};
__device__ __forceinline__ float ald(const AB &b, uint32_t i) { return i < b.n ? b.p[i] : 0.0f; }

struct DecArgs {
  AB q, ck, cv, pos;
  float *c;
  uint32_t nc;
  uint32_t B, dim, heads, kvheads, maxseq, hd, grp, kvdim;
  uint32_t hslots;  // head slots per sequence = ceil(dim / hd)
  uint32_t domain;  // output elements that are written: min(B*dim, 64*groups)
};

// EPL: head elements per lane (hd <= 64*EPL).
template <int EPL>
__global__ __launch_bounds__(256) void k_decode_attn(DecArgs a) {
  __shared__ float s_ctx[4][64 * EPL];
  __shared__ float s_z[4], s_mx[4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t bb = blockIdx.x / a.hslots, h = blockIdx.x % a.hslots;
  const uint32_t kvh = a.grp ? h / a.grp : 0u;
  const uint32_t pos = nlg_f2u(ald(a.pos, 0)), len = pos + 1u;
  const uint32_t cbase = (bb * a.maxseq) * a.kvdim, c0q = bb * a.dim + h * a.hd;
  const float coef = 1.0f / sqrtf((float)a.hd);
  float q[EPL];
#pragma unroll
  for (int e = 0; e < EPL; e++) {
    const uint32_t t = lane + 64 * e;
    q[e] = t < a.hd ? ald(a.q, c0q + t) : 0.0f;
  }
  // Positions whose K row starts past both cache buffers read as all-zero
  // rows: score exactly 0 and a zero V row.  They are folded in analytically
  // so a wild POS cannot make the loop run for billions of trips.
  const uint32_t kvoff = kvh * a.hd;
  uint64_t lim = a.ck.n > a.cv.n ? a.ck.n : a.cv.n;
  uint64_t jloop64 = len;
  if (a.kvdim) {
    uint64_t base0 = (uint64_t)cbase + kvoff;
    uint64_t jmax = base0 >= lim ? 0 : (lim - base0 + a.kvdim - 1) / a.kvdim;
    if (jloop64 > jmax) jloop64 = jmax;
  }
  const uint32_t jloop = (uint32_t)jloop64;
  // pass 1: the maximum score (seeded -1e30 as the reference)
  float mx = NEG_BIG;
  for (uint32_t j = w; j < jloop; j += 4) {
    const uint32_t kb = cbase + (j * a.kvdim + kvoff);
    float d = 0.0f;
#pragma unroll
    for (int e = 0; e < EPL; e++) {
      const uint32_t t = lane + 64 * e;
      if (t < a.hd) d = __fadd_rn(d, __fmul_rn(q[e], ald(a.ck, kb + t)));
    }
    const float s = __fmul_rn(nlg_wave_sum_f32(d), coef);
    if (s > mx) mx = s;
  }
  if (jloop < len && 0.0f > mx) mx = 0.0f;
  if (lane == 0) s_mx[w] = mx;
  __syncthreads();
  mx = s_mx[0];
  for (int i = 1; i < 4; i++) mx = s_mx[i] > mx ? s_mx[i] : mx;
  // pass 2: z and ctx
  float z = 0.0f, ctx[EPL];
#pragma unroll
  for (int e = 0; e < EPL; e++) ctx[e] = 0.0f;
  for (uint32_t j = w; j < jloop; j += 4) {
    const uint32_t kb = cbase + (j * a.kvdim + kvoff);
    float d = 0.0f;
#pragma unroll
    for (int e = 0; e < EPL; e++) {
      const uint32_t t = lane + 64 * e;
      if (t < a.hd) d = __fadd_rn(d, __fmul_rn(q[e], ald(a.ck, kb + t)));
    }
    const float ee = expf(__fsub_rn(__fmul_rn(nlg_wave_sum_f32(d), coef), mx));
    z = __fadd_rn(z, ee);
#pragma unroll
    for (int e = 0; e < EPL; e++) {
      const uint32_t t = lane + 64 * e;
      if (t < a.hd) ctx[e] = __fadd_rn(ctx[e], __fmul_rn(ee, ald(a.cv, kb + t)));
    }
  }
#pragma unroll
  for (int e = 0; e < EPL; e++) s_ctx[w][lane + 64 * e] = ctx[e];
  if (lane == 0) s_z[w] = z;
  __syncthreads();
  if (w == 0) {
    float zt = __fadd_rn(__fadd_rn(s_z[0], s_z[1]), __fadd_rn(s_z[2], s_z[3]));
    if (jloop < len) zt = __fadd_rn(zt, __fmul_rn((float)(len - jloop), expf(__fsub_rn(0.0f, mx))));
#pragma unroll
    for (int e = 0; e < EPL; e++) {
      const uint32_t t = lane + 64 * e;
      const float ct = __fadd_rn(__fadd_rn(s_ctx[0][t], s_ctx[1][t]), __fadd_rn(s_ctx[2][t], s_ctx[3][t]));
      const uint32_t oc = h * a.hd + t;  // output column within the sequence
      const uint32_t idx = bb * a.dim + oc;
      if (t < a.hd && oc < a.dim && idx < a.domain && idx < a.nc) a.c[idx] = ct / zt;
    }
  }
}

static int decode_attn_common(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st,
                              bool batched) {
  DecArgs a;
  a.B = batched ? p[0] : 1u;
  a.dim = p[batched ? 1 : 0];
  a.heads = p[batched ? 2 : 1];
  a.kvheads = p[batched ? 3 : 2];
  a.maxseq = batched ? p[4] : 0u;
  const char *k = batched ? "decode-attn-b" : "decode-attn";
  if (!a.heads || !a.kvheads) return nlg_fail("%s: heads and kvheads must be nonzero", k);
  a.hd = a.dim / a.heads;
  a.grp = a.heads / a.kvheads;
  a.kvdim = a.kvheads * a.hd;
  if (!a.hd) return NLG_OK;  // the reference divides by zero only inside an empty domain
  if (a.hd > 512) return nlg_fail("%s: head dim %u > 512", k, a.hd);
  a.hslots = (a.dim + a.hd - 1) / a.hd;
  const uint64_t dom = nlg_domain((uint32_t)(a.B * a.dim), groups);
  if (!dom) return NLG_OK;
  a.domain = (uint32_t)dom;
  a.q = AB{(const float *)b[0].ptr, b[0].nfloats};
  a.ck = AB{(const float *)b[1].ptr, b[1].nfloats};
  a.cv = AB{(const float *)b[2].ptr, b[2].nfloats};
  a.pos = AB{(const float *)b[3].ptr, b[3].nfloats};
  a.c = (float *)b[4].ptr;
  a.nc = b[4].nfloats;
  const uint32_t seqs = (uint32_t)((dom + a.dim - 1) / a.dim);
  dim3 g(seqs * a.hslots), blk(256);
  if (a.hd <= 64) hipLaunchKernelGGL(k_decode_attn<1>, g, blk, 0, st, a);
  else if (a.hd <= 128) hipLaunchKernelGGL(k_decode_attn<2>, g, blk, 0, st, a);
  else if (a.hd <= 256) hipLaunchKernelGGL(k_decode_attn<4>, g, blk, 0, st, a);
  else hipLaunchKernelGGL(k_decode_attn<8>, g, blk, 0, st, a);
  NLG_LAUNCHED(k);
  return NLG_OK;
}
int L_decode_attn(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  return decode_attn_common(b, p, groups, st, false);
}
int L_decode_attn_b(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  return decode_attn_common(b, p, groups, st, true);
}

// attn-causal-gqa: one wave per (head, query i), lanes over the head dim.
struct GqaArgs {
  AB q, k, v;
  float *ctx;
  uint32_t nctx;
  uint32_t seq, heads, kvheads, hd, n;  // n = rows handled: min(heads*seq, 64*groups)
};
template <int EPL>
__global__ __launch_bounds__(256) void k_attn_gqa(GqaArgs a) {
  const int lane = threadIdx.x & 63;
  const uint64_t r = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= a.n) return;
  const uint32_t idx = (uint32_t)r, h = idx / a.seq, i = idx % a.seq;
  const uint32_t qdim = a.heads * a.hd, kvdim = a.kvheads * a.hd, grp = a.heads / a.kvheads;
  const uint32_t qb = i * qdim + h * a.hd, kc = (grp ? h / grp : 0u) * a.hd;
  const float scale = 1.0f / sqrtf((float)a.hd);
  float q[EPL];
#pragma unroll
  for (int e = 0; e < EPL; e++) {
    const uint32_t t = lane + 64 * e;
    q[e] = t < a.hd ? ald(a.q, qb + t) : 0.0f;
  }
  const uint32_t n = i + 1;
  float mx = NEG_BIG;
  for (uint32_t j = 0; j < n; j++) {
    const uint32_t kb = j * kvdim + kc;
    float d = 0.0f;
#pragma unroll
    for (int e = 0; e < EPL; e++) {
      const uint32_t t = lane + 64 * e;
      if (t < a.hd) d = __fadd_rn(d, __fmul_rn(q[e], ald(a.k, kb + t)));
    }
    const float s = __fmul_rn(nlg_wave_sum_f32(d), scale);
    if (s > mx) mx = s;
  }
  float sm = 0.0f, ctx[EPL];
#pragma unroll
  for (int e = 0; e < EPL; e++) ctx[e] = 0.0f;
  for (uint32_t j = 0; j < n; j++) {
    const uint32_t kb = j * kvdim + kc;
    float d = 0.0f;
#pragma unroll
    for (int e = 0; e < EPL; e++) {
      const uint32_t t = lane + 64 * e;
      if (t < a.hd) d = __fadd_rn(d, __fmul_rn(q[e], ald(a.k, kb + t)));
    }
    const float ee = expf(__fsub_rn(__fmul_rn(nlg_wave_sum_f32(d), scale), mx));
    sm = __fadd_rn(sm, ee);
#pragma unroll
    for (int e = 0; e < EPL; e++) {
      const uint32_t t = lane + 64 * e;
      if (t < a.hd) ctx[e] = __fadd_rn(ctx[e], __fmul_rn(ee, ald(a.v, kb + t)));
    }
  }
#pragma unroll
  for (int e = 0; e < EPL; e++) {
    const uint32_t t = lane + 64 * e;
    if (t < a.hd && qb + t < a.nctx) a.ctx[qb + t] = ctx[e] / sm;
  }
}


// attn-causal-gqa on the f32 matrix cores (v_mfma_f32_32x32x2_f32: f32 inputs,
// products and sums; lane 32g + i holds A[i][g] and B[g][i], result r of lane
// 32g + i is C[(r % 4) + 8 (r / 4) + 4 g][i]) for the head dims instantiated
// below.  A workgroup owns 32 queries of one head; its eight waves take every
// eighth 32-key block, newest first, each with its own running maximum, sum
// and context, and meet in LDS.
//  * S^T = K Q^T: lane (g, i) holds key i's and query i's float4s 2t + g, so
//    lane (g, q) receives query q's scores of keys (r % 4) + 8 (r / 4) + 4 g.
//  * O^T += V^T P^T: step t contracts exactly keys (t % 4) + 8 (t / 4) + 4 g,
//    so the probabilities go in from the registers the scores came out in,
//    and V is read in whole 128-byte runs.
// Waves split a tile's keys rather than a kv head's query heads: causality
// makes the last query block seq / 32 key blocks long, and the longest
// workgroup sets the time of a short prompt.  Bound by the matrix cores
// (8,192 cycles a key block and wave at head dim 128): 20 heads over 5 of 128,
// 1,024 positions 2,283 -> 82 us (65 TFLOP/s; 75 us with the loads taken out of
// the loop, the rest is 2.5 rounds of workgroups), 4,096 positions 957 us (90
// TFLOP/s of the 157 the f32 cores reach), 128 positions 10.6 us.  Four waves
// in two workgroups per CU measured the same; queries held in registers (one
// wave per SIMD) 79 us at 1,024.
// Keys past a query are masked in the scores; in the diagonal block their
// probability of zero meets V rows the query does not attend, so there
// infinities and NaNs of V are left out of the product and added for the
// queries that attend them (0 x Inf would reach the others).
#define GQA_NW 8  // waves per workgroup
template <int HD>
__global__ __launch_bounds__(64 * GQA_NW) void k_gqa_mfma(GqaArgs a) {
  typedef float v16f __attribute__((ext_vector_type(16)));
  constexpr int KT = HD / 8, NT = (HD + 31) / 32, PITCH = 32 * NT + 4;
  __shared__ __align__(16) float s_o[GQA_NW][32][PITCH];
  __shared__ float s_m[GQA_NW][32], s_z[GQA_NW][32];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 5, i = lane & 31;
  const uint32_t nqb = (a.seq + 31) / 32;
  const uint32_t qb = nqb - 1 - blockIdx.x / a.heads, h = blockIdx.x % a.heads;  // longest first
  if (h * a.seq + qb * 32 >= a.n) return;  // a partial grid does not reach this tile
  const uint32_t qdim = a.heads * HD, kvdim = a.kvheads * HD, kc = h / (a.heads / a.kvheads) * HD;
  const uint32_t last = a.seq - 1;
  const float coef = NLG_LOG2E / sqrtf((float)HD);  // scores in base 2
  // the tile's queries, in wave 1's part of s_o until the waves meet
  float(*s_q)[PITCH] = s_o[1];
  for (uint32_t e = threadIdx.x; e < 32 * (HD / 4); e += 64 * GQA_NW) {
    const uint32_t q = e / (HD / 4), d = 4 * (e % (HD / 4)), row = qb * 32 + q < last ? qb * 32 + q : last;
    *(float4 *)&s_q[q][d] = *(const float4 *)(a.q.p + (size_t)row * qdim + h * HD + d);
  }
  float4 kv[KT];
  auto load_k = [&](uint32_t kb) {
    const uint32_t row = kb * 32 + i < last ? kb * 32 + i : last;
    const float *kp = a.k.p + (size_t)row * kvdim + kc + 4 * g;
#pragma unroll
    for (int t = 0; t < KT; t++) kv[t] = *(const float4 *)(kp + 8 * t);
  };
  v16f o[NT];
#pragma unroll
  for (int n = 0; n < NT; n++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[n][r] = 0.0f;
  float m = NEG_BIG * NLG_LOG2E, z = 0.0f;  // z: this lane's half of the keys
  if (qb >= (uint32_t)w) load_k(qb - w);
  __syncthreads();
  for (int64_t kb = (int64_t)qb - w; kb >= 0; kb -= GQA_NW) {
    const bool diag = kb == qb;
    float v[16][NT];
#pragma unroll
    for (int t = 0; t < 16; t++) {
      const uint32_t key = (uint32_t)kb * 32 + (t % 4) + 8 * (t / 4) + 4 * g;
      const float *vp = a.v.p + (size_t)(key < last ? key : last) * kvdim + kc;
#pragma unroll
      for (int n = 0; n < NT; n++) v[t][n] = vp[HD % 32 && 32 * n + i >= HD ? HD - 1 : 32 * n + i];
    }
    __builtin_amdgcn_sched_barrier(0);  // V on its way before the scores
    asm volatile("" ::: "memory");      // the queries stay in LDS (not hoisted into registers)
    v16f s;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = 0.0f;
#pragma unroll
    for (int t = 0; t < KT; t++) {
      const float4 q = *(const float4 *)&s_q[i][8 * t + 4 * g];
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[t].x, q.x, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[t].y, q.y, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[t].z, q.z, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[t].w, q.w, s, 0, 0, 0);
    }
    if (kb >= GQA_NW) load_k((uint32_t)kb - GQA_NW);
    __builtin_amdgcn_sched_barrier(0);  // the next K before this block's softmax
    float bm = m;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      float x = s[r] * coef;
      if (diag && (r % 4) + 8 * (r / 4) + 4 * g > i) x = -INFINITY;
      s[r] = x;
      bm = x > bm ? x : bm;  // NaN never becomes the maximum
    }
    const float ob = __shfl_xor(bm, 32);
    bm = ob > bm ? ob : bm;
    if (__any(bm > m)) {
      const float al = nlg_exp2(m - bm);
      z *= al;
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[n][r] *= al;
      m = bm;
    }
    float p[16];
#pragma unroll
    for (int r = 0; r < 16; r++) {
      p[r] = nlg_exp2(s[r] - m);
      z += p[r];
    }
    bool fix = false;
    if (diag) {
      uint32_t top = 0;  // the largest exponent
#pragma unroll
      for (int t = 0; t < 16; t++)
#pragma unroll
        for (int n = 0; n < NT; n++) {
          const uint32_t e = __float_as_uint(v[t][n]) & 0x7f800000u;
          top = e > top ? e : top;
        }
      fix = __any(top == 0x7f800000u);
      if (fix) {
#pragma unroll
        for (int t = 0; t < 16; t++)
#pragma unroll
          for (int n = 0; n < NT; n++)
            if ((__float_as_uint(v[t][n]) & 0x7f800000u) == 0x7f800000u) v[t][n] = 0.0f;
      }
    }
#pragma unroll
    for (int t = 0; t < 16; t++)
#pragma unroll
      for (int n = 0; n < NT; n++) o[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[t][n], p[t], o[n], 0, 0, 0);
    if (fix) {  // wave 0 only: its part of s_o hands the probabilities round
      float *sp = &s_o[0][0][0];
#pragma unroll
      for (int r = 0; r < 16; r++) sp[((r % 4) + 8 * (r / 4) + 4 * g) * 33 + i] = p[r];
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      for (uint32_t k = 0; k < 32 && (uint32_t)kb * 32 + k <= last; k++) {
        const float pk = sp[k * 33 + i];
        const float *vp = a.v.p + (size_t)((uint32_t)kb * 32 + k) * kvdim + kc;
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int d = 32 * n + (r % 4) + 8 * (r / 4) + 4 * g;
            const float x = d < HD ? vp[d] : 0.0f;
            if ((__float_as_uint(x) & 0x7f800000u) == 0x7f800000u && (int)k <= i) o[n][r] = fmaf(pk, x, o[n][r]);
          }
      }
    }
  }
  z += __shfl_xor(z, 32);
  if (g == 0) {
    s_m[w][i] = m;
    s_z[w][i] = z;
  }
  __syncthreads();
  float mm = s_m[0][i];
#pragma unroll
  for (int k = 1; k < GQA_NW; k++) mm = s_m[k][i] > mm ? s_m[k][i] : mm;
  const float sc = nlg_exp2(m - mm);
#pragma unroll
  for (int n = 0; n < NT; n++)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *(float4 *)&s_o[w][i][32 * n + 2 * r + 4 * g] =
          make_float4(o[n][r] * sc, o[n][r + 1] * sc, o[n][r + 2] * sc, o[n][r + 3] * sc);
  __syncthreads();
  for (uint32_t e = threadIdx.x; e < 32 * (HD / 4); e += 64 * GQA_NW) {
    const uint32_t q = e / (HD / 4), d = 4 * (e % (HD / 4)), row = qb * 32 + q;
    float qm = s_m[0][q], zz = 0.0f;
#pragma unroll
    for (int k = 1; k < GQA_NW; k++) qm = s_m[k][q] > qm ? s_m[k][q] : qm;
    float4 c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < GQA_NW; k++) {
      zz = fmaf(s_z[k][q], nlg_exp2(s_m[k][q] - qm), zz);
      const float4 x = *(const float4 *)&s_o[k][q][d];
      c.x += x.x; c.y += x.y; c.z += x.z; c.w += x.w;
    }
    if (row <= last && h * a.seq + row < a.n)
      *(float4 *)(a.ctx + (size_t)row * qdim + h * HD + d) = make_float4(c.x / zz, c.y / zz, c.z / zz, c.w / zz);
  }
}

// The matrix-core form reads whole float4 rows without bounds checks: every
// buffer must hold its full extent, 16-byte aligned (V is read by elements),
// and each kv head must serve the same number of query heads.  Taken at every
// length: one query block already beats the per-query walk (2 x 128-lane
// reductions per key) at 16 positions.
static bool gqa_mfma_ok(const GqaArgs &a) {
  const uint64_t rows = (uint64_t)a.heads * a.seq, qn = rows * a.hd, kn = (uint64_t)a.seq * a.kvheads * a.hd;
  const uintptr_t at = (uintptr_t)a.q.p | (uintptr_t)a.k.p | (uintptr_t)a.ctx;
  return a.heads && a.heads % a.kvheads == 0 && rows < (1u << 31) && a.q.n >= qn && a.nctx >= qn &&
         a.k.n >= kn && a.v.n >= kn && a.q.p && a.k.p && a.v.p && a.ctx && (at & 15) == 0;
}

int L_attn_causal_gqa(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  GqaArgs a;
  a.seq = p[0];
  a.heads = p[1];
  a.kvheads = p[2];
  a.hd = p[3];
  if (!a.kvheads || !a.seq) return a.seq ? nlg_fail("attn-causal-gqa: kvheads must be nonzero") : NLG_OK;
  if (a.hd > 512) return nlg_fail("attn-causal-gqa: head dim %u > 512", a.hd);
  const uint64_t n = nlg_domain((uint32_t)(a.heads * a.seq), groups);
  if (!n || !a.hd) return NLG_OK;
  a.n = (uint32_t)n;
  a.q = AB{(const float *)b[0].ptr, b[0].nfloats};
  a.k = AB{(const float *)b[1].ptr, b[1].nfloats};
  a.v = AB{(const float *)b[2].ptr, b[2].nfloats};
  a.ctx = (float *)b[3].ptr;
  a.nctx = b[3].nfloats;
  const dim3 blk(256);
  if (gqa_mfma_ok(a)) {
    const dim3 t((a.seq + 31) / 32 * a.heads);
    bool took = true;
    const dim3 blk(64 * GQA_NW);
    if (a.hd == 128) hipLaunchKernelGGL(k_gqa_mfma<128>, t, blk, 0, st, a);
    else if (a.hd == 96) hipLaunchKernelGGL(k_gqa_mfma<96>, t, blk, 0, st, a);
    else if (a.hd == 80) hipLaunchKernelGGL(k_gqa_mfma<80>, t, blk, 0, st, a);
    else if (a.hd == 64) hipLaunchKernelGGL(k_gqa_mfma<64>, t, blk, 0, st, a);
    else if (a.hd == 32) hipLaunchKernelGGL(k_gqa_mfma<32>, t, blk, 0, st, a);
    else took = false;
    if (took) {
      NLG_LAUNCHED("attn-causal-gqa");
      return NLG_OK;
    }
  }
  const dim3 g(nlg_blocks(n, 4));
  if (a.hd <= 64) hipLaunchKernelGGL(k_attn_gqa<1>, g, blk, 0, st, a);
  else if (a.hd <= 128) hipLaunchKernelGGL(k_attn_gqa<2>, g, blk, 0, st, a);
  else if (a.hd <= 256) hipLaunchKernelGGL(k_attn_gqa<4>, g, blk, 0, st, a);
  else hipLaunchKernelGGL(k_attn_gqa<8>, g, blk, 0, st, a);
  NLG_LAUNCHED("attn-causal-gqa");
  return NLG_OK;
}

// attn-scores (kernels.el:205-222), per element, serial dot in reference order.
__global__ __launch_bounds__(256) void k_attn_scores(AB q, AB k, float *s, uint32_t ns, uint32_t n,
                                                     uint32_t seq, uint32_t dim, uint32_t heads,
                                                     uint32_t kvheads) {
  const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const uint32_t hd = dim / heads, grp = heads / kvheads, kvdim = kvheads * hd;
  const uint32_t h = idx / (seq * seq), rem = idx % (seq * seq), i = rem / seq, j = rem % seq;
  if (j > i && idx < ns) s[idx] = NEG_BIG;
  if (j < i + 1) {
    const uint32_t kvh = grp ? h / grp : 0u, qb = i * dim + h * hd, kb = j * kvdim + kvh * hd;
    float acc = 0.0f;
    for (uint32_t t = 0; t < hd; t++) acc = __fadd_rn(acc, __fmul_rn(ald(q, qb + t), ald(k, kb + t)));
    if (idx < ns) s[idx] = __fmul_rn(acc, 1.0f / sqrtf((float)hd));
  }
}
int L_attn_scores(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  const uint32_t seq = p[0], dim = p[1], heads = p[2], kvheads = p[3];
  if (!heads || !kvheads) return nlg_fail("attn-scores: heads and kvheads must be nonzero");
  const uint64_t n = nlg_domain((uint32_t)((heads * seq) * seq), groups);
  if (!n || !seq) return NLG_OK;
  hipLaunchKernelGGL(k_attn_scores, dim3(nlg_blocks(n, 256)), dim3(256), 0, st,
                     AB{(const float *)b[0].ptr, b[0].nfloats}, AB{(const float *)b[1].ptr, b[1].nfloats},
                     (float *)b[2].ptr, b[2].nfloats, (uint32_t)n, seq, dim, heads, kvheads);
  NLG_LAUNCHED("attn-scores");
  return NLG_OK;
}

// attn-context (kernels.el:223-235), per element, serial in reference order.
__global__ __launch_bounds__(256) void k_attn_context(AB pm, AB v, float *c, uint32_t nc, uint32_t n,
                                                      uint32_t seq, uint32_t dim, uint32_t heads,
                                                      uint32_t kvheads) {
  const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const uint32_t hd = dim / heads, grp = heads / kvheads, kvdim = kvheads * hd;
  const uint32_t i = idx / dim, cc = idx % dim;
  const uint32_t h = hd ? cc / hd : 0u, t = hd ? cc % hd : 0u, kvh = grp ? h / grp : 0u;
  const uint32_t pb = h * (seq * seq) + i * seq;
  float acc = 0.0f;
  for (uint32_t j = 0; j < seq; j++)
    acc = __fadd_rn(acc, __fmul_rn(ald(pm, pb + j), ald(v, j * kvdim + (kvh * hd + t))));
  if (idx < nc) c[idx] = acc;
}
int L_attn_context(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  const uint32_t seq = p[0], dim = p[1], heads = p[2], kvheads = p[3];
  if (!heads || !kvheads) return nlg_fail("attn-context: heads and kvheads must be nonzero");
  const uint64_t n = nlg_domain((uint32_t)(seq * dim), groups);
  if (!n) return NLG_OK;
  hipLaunchKernelGGL(k_attn_context, dim3(nlg_blocks(n, 256)), dim3(256), 0, st,
                     AB{(const float *)b[0].ptr, b[0].nfloats}, AB{(const float *)b[1].ptr, b[1].nfloats},
                     (float *)b[2].ptr, b[2].nfloats, (uint32_t)n, seq, dim, heads, kvheads);
  NLG_LAUNCHED("attn-context");
  return NLG_OK;
}
