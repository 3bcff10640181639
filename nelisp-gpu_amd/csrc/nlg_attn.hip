// nlg_attn.hip -- attention on the reference's f32 layouts.
//
//   decode-attn / decode-attn-b (kernels.el:315-390): single-query causal GQA
//     over cached K/V.  The reference spends one invocation per output
//     element and recomputes every q.k product hd times; here the positions
//     are split over workgroups that each serve the query heads of one kv head
//     (k_decode_split).  Forms that is not made for: a workgroup owns one
//     (sequence, head), each wave takes every 4th position, its 64 lanes split
//     the head dimension, the q.k product is one DPP reduction, and the four
//     waves' running (z, ctx) are merged through LDS (k_decode_attn).
//   attn-causal-gqa (kernels.el:934-990): 32-query tiles on the f32 matrix
//     cores; one wave per (head, query) for the forms those do not take.
//   attn-scores / attn-context (kernels.el:205-235): per element, serial in
//     the reference's order (bit-identical up to the 1/sqrt(hd) scale).
// Every access is bounds-checked (reads past a buffer give 0, writes are
// dropped) because POS comes from device memory.
#include <math.h>

#include <mutex>

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


// decode-attn(-b) with the positions split: a workgroup takes G query heads of
// one kv head of one sequence, so a K or V row is read once for them, and its
// eight waves walk blocks of DS_NI x PPI positions (float4 pieces, L lanes a
// row, PPI = 64 / L rows an instruction) dealt round-robin over all waves of
// all `nsplit` workgroups of the unit.  One pass: each block moves the wave's
// running maximum, sum and context, the next block's rows already on their way.
// Maxima are kept as raw q.k and a difference is scaled where it is
// exponentiated (dec_exp): it is exact near the maximum, so the largest element
// weighs exactly 1 at any finite score (a maximum rounded after the scaling is off
// by half its ulp, an exponent past 127 from scores of 1e10 on), and smaller
// scores are rounded at their distance to the maximum.  With nsplit > 1 the workgroup leaves its partial
// context and (maximum, sum) for k_decode_merge; with 1 it writes C.
// Bound by the K/V stream and, below a few MB, by the launches and the chain
// position -> rows -> partials: 4 sequences of 2,048 positions, 20 heads over 5
// of 128 (42 MB) 927 -> 20.0 us; one of 701 positions 159 -> 9.4; one of 8,001,
// 32 heads over 8 (66 MB) 3,794 -> 27.3 (2.4 TB/s); one of 32 9.4 -> 5.5.  k_decode_attn,
// two passes of one position a wave at a time, stays for buffers that hold no
// whole float4 rows.
#define DS_WAVES 8
#define DS_NI 8
#define DS_MAX_SPLIT 64  // a merge workgroup's first wave holds one partial a lane
struct SplitArgs {
  DecArgs d;
  uint32_t nsplit, hgroups;  // workgroups per (sequence, kv head, head group); head groups per kv head
  float *pctx, *pmz;         // [B][heads][nsplit][hd], [B][heads][nsplit][2]
};

// exp((s - m) / sqrt(hd)) of raw dot products, coef = log2(e) / sqrt(hd)
__device__ __forceinline__ float dec_exp(float s, float m, float coef) { return nlg_exp2((s - m) * coef); }

// Sum over aligned groups of L lanes (16, 32 or 64), in every lane.
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
  v = v + __int_as_float(nlg_dpp<0xB1>(__float_as_int(v)));   // quad_perm [1,0,3,2]
  v = v + __int_as_float(nlg_dpp<0x4E>(__float_as_int(v)));   // quad_perm [2,3,0,1]
  v = v + __int_as_float(nlg_dpp<0x141>(__float_as_int(v)));  // row_half_mirror
  v = v + __int_as_float(nlg_dpp<0x140>(__float_as_int(v)));  // row_mirror
  if (L >= 32) v = nlg_halve_f32<16>(v, v);
  if (L >= 64) v = nlg_halve_f32<32>(v, v);
  return v;
}

template <int L, int G, bool SPLIT>
__global__ __launch_bounds__(64 * DS_WAVES) void k_decode_split(SplitArgs sa) {
  constexpr int PPI = 64 / L, PB = DS_NI * PPI;
  const DecArgs &a = sa.d;
  __shared__ __align__(16) float s_ctx[DS_WAVES][G][4 * L];
  __shared__ float s_m[DS_WAVES][G], s_z[DS_WAVES][G];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, sub = lane / L, dl = lane % L;
  const uint32_t split = SPLIT ? blockIdx.x % sa.nsplit : 0u, unit = SPLIT ? blockIdx.x / sa.nsplit : blockIdx.x;
  const uint32_t hg = unit % sa.hgroups, kvh = unit / sa.hgroups % a.kvheads, bb = unit / sa.hgroups / a.kvheads;
  const uint32_t h0 = kvh * a.grp + hg * G, nh = a.grp - hg * G < (uint32_t)G ? a.grp - hg * G : (uint32_t)G;
  const uint32_t pos = nlg_f2u(ald(a.pos, 0)), len = pos + 1u;
  const uint64_t base0 = (uint64_t)bb * a.maxseq * a.kvdim;
  // rows past the caches score 0 with a zero V row: counted at the end
  const uint64_t rows = base0 < a.ck.n ? (a.ck.n - base0) / a.kvdim : 0;
  const uint32_t jl = len < rows ? len : (uint32_t)rows;
  const bool on = 4u * dl < a.hd;
  const float coef = NLG_LOG2E / sqrtf((float)a.hd), least = NEG_BIG * sqrtf((float)a.hd);
  const float4 zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float4 q[G], cx[G];
  float m[G], z[G];
#pragma unroll
  for (int h = 0; h < G; h++) {
    const uint32_t hh = (uint32_t)h < nh ? h0 + h : h0;
    q[h] = *(const float4 *)(a.q.p + (size_t)bb * a.dim + (size_t)hh * a.hd + (on ? 4 * dl : 0));
    if (!on) q[h] = zero4;
    cx[h] = zero4;
    m[h] = least;
    z[h] = 0.0f;
  }
  const size_t rb = base0 + kvh * a.hd + (on ? 4 * dl : 0);
  const float *kp = a.ck.p + rb, *vp = a.cv.p + rb;
  const uint32_t stride = DS_WAVES * sa.nsplit * PB;
  uint32_t j0 = (w * sa.nsplit + split) * PB;
  float4 kn[DS_NI], vn[DS_NI];
  // rows past the last position fetch the last one again (one cached row)
  auto load = [&](uint32_t j) {
#pragma unroll
    for (int i = 0; i < DS_NI; i++) {
      const uint32_t r = j + i * PPI + sub, rc = r < jl ? r : jl - 1;
      kn[i] = *(const float4 *)(kp + (size_t)rc * a.kvdim);
    }
#pragma unroll
    for (int i = 0; i < DS_NI; i++) {
      const uint32_t r = j + i * PPI + sub, rc = r < jl ? r : jl - 1;
      vn[i] = *(const float4 *)(vp + (size_t)rc * a.kvdim);
    }
  };
  if (j0 < jl) load(j0);
  for (; j0 < jl; j0 += stride) {
    float4 k[DS_NI], v[DS_NI];
#pragma unroll
    for (int i = 0; i < DS_NI; i++) {
      const bool ok = j0 + i * PPI + sub < jl;  // a row not attended may hold anything: its V counts as zeros
      k[i] = kn[i];
      v[i] = make_float4(ok ? vn[i].x : 0.0f, ok ? vn[i].y : 0.0f, ok ? vn[i].z : 0.0f, ok ? vn[i].w : 0.0f);
    }
    const uint32_t nx = jl - j0 > stride ? j0 + stride : jl - 1;
    load(nx);
    float s[DS_NI][G];
#pragma unroll
    for (int i = 0; i < DS_NI; i++)
#pragma unroll
      for (int h = 0; h < G; h++) {
        float d = q[h].x * k[i].x;
        d = fmaf(q[h].y, k[i].y, d);
        d = fmaf(q[h].z, k[i].z, d);
        d = fmaf(q[h].w, k[i].w, d);
        if (!on) d = 0.0f;
        d = lanes_sum<L>(d);
        s[i][h] = j0 + i * PPI + sub < jl ? d : -INFINITY;
      }
#pragma unroll
    for (int h = 0; h < G; h++) {
      float bm = s[0][h] > m[h] ? s[0][h] : m[h];  // NaN never becomes the maximum
#pragma unroll
      for (int i = 1; i < DS_NI; i++) bm = s[i][h] > bm ? s[i][h] : bm;
      const float al = dec_exp(m[h], bm, coef);
      m[h] = bm;
      z[h] *= al;
      cx[h].x *= al; cx[h].y *= al; cx[h].z *= al; cx[h].w *= al;
#pragma unroll
      for (int i = 0; i < DS_NI; i++) {
        const float e = dec_exp(s[i][h], bm, coef);
        z[h] += e;
        cx[h].x = fmaf(e, v[i].x, cx[h].x);
        cx[h].y = fmaf(e, v[i].y, cx[h].y);
        cx[h].z = fmaf(e, v[i].z, cx[h].z);
        cx[h].w = fmaf(e, v[i].w, cx[h].w);
      }
    }
  }
  // the wave's row slots meet, then the waves
#pragma unroll
  for (int h = 0; h < G; h++) {
#pragma unroll
    for (int off = L; off < 64; off <<= 1) {
      const float om = __shfl_xor(m[h], off), mm = om > m[h] ? om : m[h];
      const float al = dec_exp(m[h], mm, coef), ol = dec_exp(om, mm, coef);
      z[h] = fmaf(z[h], al, __shfl_xor(z[h], off) * ol);
      cx[h].x = fmaf(cx[h].x, al, __shfl_xor(cx[h].x, off) * ol);
      cx[h].y = fmaf(cx[h].y, al, __shfl_xor(cx[h].y, off) * ol);
      cx[h].z = fmaf(cx[h].z, al, __shfl_xor(cx[h].z, off) * ol);
      cx[h].w = fmaf(cx[h].w, al, __shfl_xor(cx[h].w, off) * ol);
      m[h] = mm;
    }
    if (sub == 0) *(float4 *)&s_ctx[w][h][4 * dl] = cx[h];
    if (lane == 0) {
      s_m[w][h] = m[h];
      s_z[w][h] = z[h];
    }
  }
  __syncthreads();
  for (uint32_t e = threadIdx.x; e < nh * a.hd; e += 64 * DS_WAVES) {
    const uint32_t h = e / a.hd, d = e % a.hd;
    float mm = s_m[0][h];
#pragma unroll
    for (int k = 1; k < DS_WAVES; k++) mm = s_m[k][h] > mm ? s_m[k][h] : mm;
    const uint32_t out = split == 0 ? len - jl : 0u;  // positions past the caches: score 0, zero V
    if (out && 0.0f > mm) mm = 0.0f;
    float zz = out ? (float)out * dec_exp(0.0f, mm, coef) : 0.0f, c = 0.0f;
#pragma unroll
    for (int k = 0; k < DS_WAVES; k++) {
      const float sc = dec_exp(s_m[k][h], mm, coef);
      zz = fmaf(s_z[k][h], sc, zz);
      c = fmaf(s_ctx[k][h][d], sc, c);
    }
    const size_t at = (size_t)bb * a.heads + h0 + h;
    if (SPLIT) {
      sa.pctx[(at * sa.nsplit + split) * a.hd + d] = c;
      if (d == 0) {
        sa.pmz[(at * sa.nsplit + split) * 2] = mm;
        sa.pmz[(at * sa.nsplit + split) * 2 + 1] = zz;
      }
    } else {
      const size_t idx = at * a.hd + d;
      if (idx < a.domain && idx < a.nc) a.c[idx] = c / zz;
    }
  }
}

// The workgroups' partials of one (sequence, head), merged and normalised.
__global__ __launch_bounds__(256) void k_decode_merge(SplitArgs sa) {
  const DecArgs &a = sa.d;
  __shared__ float s_w[DS_MAX_SPLIT], s_z;
  const size_t at = blockIdx.x;
  if (threadIdx.x < 64) {
    const uint32_t t = threadIdx.x;
    const float *mz = sa.pmz + at * sa.nsplit * 2;
    const float root = sqrtf((float)a.hd);
    const float m = t < sa.nsplit ? mz[2 * t] : NEG_BIG * root, z = t < sa.nsplit ? mz[2 * t + 1] : 0.0f;
    const float sc = dec_exp(m, nlg_wave_max_f32(m), NLG_LOG2E / root);
    s_w[t] = sc;
    const float zz = nlg_wave_sum_f32(z * sc);
    if (t == 0) s_z = zz;
  }
  __syncthreads();
  const float *pc = sa.pctx + at * sa.nsplit * a.hd;
  for (uint32_t d = threadIdx.x; d < a.hd; d += 256) {
    float c = 0.0f;
#pragma unroll 8
    for (uint32_t k = 0; k < sa.nsplit; k++) c = fmaf(pc[(size_t)k * a.hd + d], s_w[k], c);
    const size_t idx = at * a.hd + d;
    if (idx < a.domain && idx < a.nc) a.c[idx] = c / s_z;
  }
}

template <int L, bool SPLIT>
static void decode_split_go(const SplitArgs &sa, uint32_t g, hipStream_t st) {
  const dim3 grid(sa.d.B * sa.d.kvheads * sa.hgroups * sa.nsplit), blk(64 * DS_WAVES);
  if (g == 4) hipLaunchKernelGGL((k_decode_split<L, 4, SPLIT>), grid, blk, 0, st, sa);
  else if (g == 2) hipLaunchKernelGGL((k_decode_split<L, 2, SPLIT>), grid, blk, 0, st, sa);
  else hipLaunchKernelGGL((k_decode_split<L, 1, SPLIT>), grid, blk, 0, st, sa);
}
template <bool SPLIT>
static void decode_split_hd(const SplitArgs &sa, uint32_t g, hipStream_t st) {
  if (sa.d.hd <= 64) decode_split_go<16, SPLIT>(sa, g, st);
  else if (sa.d.hd <= 128) decode_split_go<32, SPLIT>(sa, g, st);
  else decode_split_go<64, SPLIT>(sa, g, st);
}

// Whether k_decode_split takes this call (whole float4 rows, unchecked: the
// caches hold whole rows, as many of K as of V; q and every head's output
// columns exist), and its launches.  The partials live in a scratch of the
// stream; the mutex keeps two threads' launch pairs on one stream apart.  A
// call that is being captured, or whose scratch cannot be had, runs with one
// workgroup per unit, in one launch and without scratch: a graph may be
// replayed beside other calls.
static bool decode_split(const DecArgs &a, hipStream_t st) {
  const uintptr_t at = (uintptr_t)a.q.p | (uintptr_t)a.ck.p | (uintptr_t)a.cv.p;
  if (a.hd % 4 || a.hd > 256 || a.dim != a.heads * a.hd || a.heads % a.kvheads || !a.q.p || !a.ck.p || !a.cv.p ||
      (at & 15) || a.ck.n != a.cv.n || a.ck.n % a.kvdim || a.q.n < (uint64_t)a.B * a.dim ||
      (uint64_t)a.B * a.dim >= (1u << 31) || (uint64_t)a.B * a.maxseq * a.kvdim > 0xffffffffull)
    return false;
  SplitArgs sa{};
  sa.d = a;
  // four heads a workgroup, unless that leaves half of its registers idle
  const uint32_t g = a.grp >= 3 ? 4u : a.grp;
  sa.hgroups = (a.grp + g - 1) / g;
  sa.nsplit = 1;
  // two workgroups per CU (for two and four heads of up to 128 the registers hold one at a
  // time: two rounds), none with less than a block for each wave of the cache's room
  const uint64_t units = (uint64_t)a.B * a.kvheads * sa.hgroups;
  if (!nlg_fits(units, 64 * DS_WAVES)) return false;  // (k_decode_attn's workgroups are half as large)
  const uint64_t rows = a.maxseq ? a.maxseq : a.ck.n / a.kvdim;
  const uint32_t pb = DS_NI * (a.hd <= 64 ? 4u : a.hd <= 128 ? 2u : 1u);
  uint64_t want = 2ull * nlg_num_cu() / units, most = (rows + DS_WAVES * pb - 1) / (DS_WAVES * pb);
  if (want > DS_MAX_SPLIT) want = DS_MAX_SPLIT;
  if (want > most) want = most;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (want > 1 && hipStreamIsCapturing(st, &cs) == hipSuccess && cs == hipStreamCaptureStatusNone) {
    const size_t n = (size_t)a.B * a.heads * want;
    static std::mutex mu;
    std::lock_guard<std::mutex> lk(mu);
    if (float *ws = (float *)nlg_scratch_try((n * a.hd + 2 * n) * 4, st, 3)) {
      sa.nsplit = (uint32_t)want;
      sa.pctx = ws;
      sa.pmz = ws + n * a.hd;
      decode_split_hd<true>(sa, g, st);
      hipLaunchKernelGGL(k_decode_merge, dim3(a.B * a.heads), dim3(256), 0, st, sa);
      return true;
    }
  }
  decode_split_hd<false>(sa, g, st);
  return true;
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
  if (decode_split(a, st)) {
    NLG_LAUNCHED(k);
    return NLG_OK;
  }
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
// 1,024 positions 2,283 -> 82 us (65 TFLOP/s of the 153 a large f32 product reaches;
// 2.5 rounds of workgroups), 300 positions 22.5 us, 128 12.3, 16 9.8 (14.9 before).  Four waves
// in two workgroups per CU measured the same; queries held in registers (one
// wave per SIMD) 79 us at 1,024.
// Keys past a query are masked in the scores; in the diagonal block their
// probability of zero meets V rows the query does not attend, so there
// infinities and NaNs of V are left out of the product and added for the
// queries that attend them (0 x Inf would reach the others).
// A score is summed in chains of 8 dimensions that meet in pairs.  One chain over
// the head dimension rounds after each of them: 2-norm error against 64 bits at head
// dim 128, 16 / 40 / 100 / 300 / 700 positions, the per-query kernel 0.89 / 1.13 /
// 1.47 / 2.09 / 2.82e-7, one chain 1.62 / 2.13 / 2.52 / 2.90 / 3.15e-7, chains of 16
// 0.88 / 1.10 / 1.27 / 1.42 / 1.57e-7, of 8 0.84 / 1.06 / 1.22 / 1.37 / 1.51e-7 at the same
// time.  The pairs' sums need the registers that held the next block's K: a block
// loads its own, and the other wave of the SIMD covers it (with both, 160 registers
// spilled and 1,024 positions took 352 us, not 82).
#define GQA_NW 8  // waves per workgroup
typedef float gqa_v16f __attribute__((ext_vector_type(16)));
template <int T0, int N>
__device__ __forceinline__ gqa_v16f gqa_scores(const float4 *kv, const float *qp) {
  gqa_v16f s;
  if constexpr (N > 1) {
    s = gqa_scores<T0, N / 2>(kv, qp);
    s += gqa_scores<T0 + N / 2, N - N / 2>(kv, qp);
  } else {
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = 0.0f;
    const float4 q = *(const float4 *)(qp + 8 * T0);
    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[T0].x, q.x, s, 0, 0, 0);
    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[T0].y, q.y, s, 0, 0, 0);
    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[T0].z, q.z, s, 0, 0, 0);
    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[T0].w, q.w, s, 0, 0, 0);
  }
  asm volatile("" : "+v"(s)::"memory");  // one chain after the other: K's registers free up as the sums need them
  __builtin_amdgcn_sched_barrier(0);
  return s;
}
template <int HD>
__global__ __launch_bounds__(64 * GQA_NW) void k_gqa_mfma(GqaArgs a) {
  typedef gqa_v16f v16f;
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
  __syncthreads();
  for (int64_t kb = (int64_t)qb - w; kb >= 0; kb -= GQA_NW) {
    const bool diag = kb == qb;
    load_k((uint32_t)kb);
    // V on its way before the scores, half of it once they have freed half of K's registers
    float v[16][NT];
    auto load_v = [&](int t0, int t1) {
#pragma unroll
      for (int t = t0; t < t1; t++) {
        const uint32_t key = (uint32_t)kb * 32 + (t % 4) + 8 * (t / 4) + 4 * g;
        const float *vp = a.v.p + (size_t)(key < last ? key : last) * kvdim + kc;
#pragma unroll
        for (int n = 0; n < NT; n++) v[t][n] = vp[HD % 32 && 32 * n + i >= HD ? HD - 1 : 32 * n + i];
      }
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");  // the queries stay in LDS (not hoisted into registers)
    };
    load_v(0, 8);
    v16f s = gqa_scores<0, KT / 2>(kv, &s_q[i][4 * g]);
    load_v(8, 16);
    s += gqa_scores<KT / 2, KT - KT / 2>(kv, &s_q[i][4 * g]);
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
// and each kv head must serve the same number of query heads.
static bool gqa_mfma_ok(const GqaArgs &a) {
  const uint64_t rows = (uint64_t)a.heads * a.seq, qn = rows * a.hd, kn = (uint64_t)a.seq * a.kvheads * a.hd;
  const uintptr_t at = (uintptr_t)a.q.p | (uintptr_t)a.k.p | (uintptr_t)a.ctx;
  return a.heads && a.heads % a.kvheads == 0 && rows < (1u << 31) &&
         nlg_fits(((uint64_t)a.seq + 31) / 32 * a.heads, 64 * GQA_NW) && a.q.n >= qn && a.nctx >= qn &&
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
  // A few queries: the walk over the keys (k_attn_gqa) is shorter than one key block
  // of the matrix-core tile and the meeting of its waves.  us, walk / tile, 4 and 20
  // heads alike: head dim 128, 1 / 4 / 8 / 9 queries 3.2 / 5.5 / 8.6 / 9.3 against 9.2-9.4;
  // 96, 6 / 7 / 8: 7.1 / 7.8 / 8.7, 7.8; 80, 6 / 7: 7.1 / 7.8, 7.6; 64, 8 / 9: 6.1 / 6.5,
  // 6.3; 32, 5 / 6: 4.6 / 5.0, 4.8.
#define GQA_TILE(HD, WALK)                                                                \
  if (a.hd == HD && a.seq > WALK && gqa_mfma_ok(a)) {                                     \
    const dim3 t((a.seq + 31) / 32 * a.heads);                                            \
    hipLaunchKernelGGL(k_gqa_mfma<HD>, t, dim3(64 * GQA_NW), 0, st, a);                   \
    NLG_LAUNCHED("attn-causal-gqa");                                                      \
    return NLG_OK;                                                                        \
  }
  GQA_TILE(128, 8)
  GQA_TILE(96, 7)
  GQA_TILE(80, 6)
  GQA_TILE(64, 8)
  GQA_TILE(32, 5)
#undef GQA_TILE
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
