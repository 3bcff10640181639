// nlg_gemm.hip -- f32 GEMM behind matmul, matmul-tiled, matmul-reg, linear
// (lisp/nelisp-gpu-kernels.el:17-27, :71-107, :129).
//
// Each output element is one dependent chain of f32 additions in the
// reference, so one kernel serves all four names with the reference's own
// summation order per name (bit-identical results):
//   matmul, matmul-reg, linear  acc = acc + a*b for k = 0..K-1 (acc starts at
//                               0, or at the bias for linear);
//   matmul-tiled                per 16-wide k tile, p0 + (p1 + (... + (p14 +
//                               p15))) added to acc (the tile sum the
//                               reference writes out, zero products past K).
// In small products the chain length bounds the time, not the flops, so the
// work is spread as wide as it goes: one 256-thread workgroup per 16 x 16 output
// tile (a 256^3 product is 256 workgroups, one per CU), one output per thread, the
// tile's A rows and B columns for 256 values of k staged through LDS with
// every global load of a chunk issued before the first is used.  Products of
// more tiles give a thread several outputs (k_mmt).
//
// Partial grids: a dispatch of `groups` workgroups covers only the outputs
// the reference's invocations gid < 64*groups (matmul-tiled: workgroups
// wg < groups) would write; the rest of C is left as it was.
#include "nlg_internal.h"
#include "nlg_mm_tile.h"

#define MM_T 16    // output tile edge
#define MM_KC 256  // k per LDS stage

enum { MM_SERIAL = 0, MM_TILE16 = 1 };
// which outputs a partial grid covers: by row-major index, by 4x4 block
// index (matmul-reg), or by 16x16 tile index (matmul-tiled)
enum { LIM_INDEX = 0, LIM_BLOCK4 = 1, LIM_TILE16 = 2 };

__device__ __forceinline__ bool mm_covered(uint32_t row, uint32_t col, uint32_t N, int lim_mode, uint64_t lim) {
  uint64_t at;
  if (lim_mode == LIM_INDEX) at = (uint64_t)row * N + col;
  else if (lim_mode == LIM_BLOCK4) at = (uint64_t)(row / 4) * ((N + 3) / 4) + col / 4;
  else at = (uint64_t)(row / 16) * ((N + 15) / 16) + col / 16;
  return at < lim;
}

template <int ORDER, bool TRANS_B, bool BIAS>
__global__ __launch_bounds__(256) void k_mm(const float *__restrict__ A, const float *__restrict__ B,
                                            const float *__restrict__ bias, float *__restrict__ C, uint32_t M,
                                            uint32_t N, uint32_t K, int lim_mode, uint64_t lim) {
  __shared__ float As[MM_T][MM_KC + 1];
  __shared__ float Bs[MM_KC][MM_T + 1];
  const uint32_t t = threadIdx.x, tx = t & 15, ty = t >> 4;
  const uint32_t m0 = blockIdx.y * MM_T, n0 = blockIdx.x * MM_T;
  const uint32_t row = m0 + ty, col = n0 + tx;
  float acc = 0.0f;
  if (BIAS) acc = col < N ? bias[col] : 0.0f;
  for (uint32_t k0 = 0; k0 < K; k0 += MM_KC) {
    const uint32_t kc = K - k0 < MM_KC ? K - k0 : MM_KC;
    float ra[MM_T], rb[MM_T];
    // A rows m0..m0+15, k0..k0+255: lane t reads column k0+t of each row
#pragma unroll
    for (int j = 0; j < MM_T; j++) {
      const uint32_t r = m0 + j;
      ra[j] = (r < M && t < kc) ? A[(size_t)r * K + k0 + t] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < MM_T; j++) {
      if (TRANS_B) {  // W [N x K]: lane t reads k0+t of rows n0..n0+15
        const uint32_t c = n0 + j;
        rb[j] = (c < N && t < kc) ? B[(size_t)c * K + k0 + t] : 0.0f;
      } else {  // B [K x N]: lanes read 16 consecutive columns of 16 k rows
        const uint32_t kk = 16 * j + (t >> 4), c = n0 + (t & 15);
        rb[j] = (kk < kc && c < N) ? B[(size_t)(k0 + kk) * N + c] : 0.0f;
      }
    }
    __syncthreads();  // the previous stage has been consumed
#pragma unroll
    for (int j = 0; j < MM_T; j++) {
      As[j][t] = ra[j];
      if (TRANS_B) Bs[t][j] = rb[j];
      else Bs[16 * j + (t >> 4)][t & 15] = rb[j];
    }
    __syncthreads();
    if (ORDER == MM_SERIAL) {
      // acc = acc + a*b, k ascending (kernels.el:24-26, :78-80); unrolled so
      // the LDS reads run well ahead of the dependent adds
#pragma unroll 32
      for (uint32_t k = 0; k < kc; k++) acc = __fadd_rn(acc, __fmul_rn(As[ty][k], Bs[k][tx]));
    } else {
      // kernels.el:99-104: acc + (p0 + (p1 + ... (p14 + p15))) per tile of 16
      for (uint32_t kb = 0; kb < kc; kb += 16) {
        float s = __fmul_rn(As[ty][kb + 15], Bs[kb + 15][tx]);
#pragma unroll
        for (int q = 14; q >= 0; q--) s = __fadd_rn(__fmul_rn(As[ty][kb + q], Bs[kb + q][tx]), s);
        acc = __fadd_rn(acc, s);
      }
    }
  }
  if (row < M && col < N && mm_covered(row, col, N, lim_mode, lim)) C[(size_t)row * N + col] = acc;
}

// The same products and sums with TM x TN outputs a thread, for products large
// enough to fill the chip that way: a 16 TM x 16 TN tile per workgroup, A and B for
// 32 values of k staged in LDS (A transposed, so a thread's rows are one read),
// the next stage's loads in flight, and the LDS reads of four k ahead of the
// arithmetic.  The multiply and the add round apart, so two vector instructions
// per product bound it (79 TFLOP/s with every SIMD issuing from several waves: one
// wave alone issues half as often), and a thread's TM + TN values of a k serve
// TM x TN products.  1,024^3 134 -> 56 us (38 TFLOP/s), 2,048^3 1,024 -> 349 (49).
// 8 x 8 outputs a thread leave one wave per SIMD: 560 us at 2,048^3.
constexpr int MT_KC = 32, MT_KG = 4;  // k per stage; k read ahead

template <int TM, int TN, int ORDER, bool TRANS_B, bool BIAS, bool VEC>
__global__ __launch_bounds__(256) void k_mmt(const float *__restrict__ A, const float *__restrict__ B,
                                             const float *__restrict__ bias, float *__restrict__ C, uint32_t M,
                                             uint32_t N, uint32_t K, int lim_mode, uint64_t lim) {
  constexpr int TA = 16 * TM, TB = 16 * TN, KC = MT_KC, KG = MT_KG;
  constexpr int NA = TA * KC / 1024, NB = TB * KC / 1024;  // float4s of A and of B per thread and stage
  typedef float veca __attribute__((ext_vector_type(TM)));
  typedef float vecb __attribute__((ext_vector_type(TN)));
  __shared__ __align__(16) float As[2][KC][TA + 4], Bs[2][KC][TB + 4];
  const uint32_t t = threadIdx.x, tx = t & 15, ty = t >> 4;
  const uint32_t nt = (N + TB - 1) / TB, m0 = blockIdx.x / nt * TA, n0 = blockIdx.x % nt * TB;
  float4 ra[NA], rb[NB];
  // four k of one row of a [rows x K] matrix (zeros past K, some row's past the last)
  auto row4 = [&](const float *p, uint32_t r, uint32_t rows, uint32_t k) {
    const float *q = p + (size_t)(r < rows ? r : rows - 1) * K;
    float4 v;
    if (VEC) {
      v = *(const float4 *)(q + (k < K ? k : K - 4));
      if (k >= K) v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    } else {
      v.x = k < K ? q[k] : 0.0f;
      v.y = k + 1 < K ? q[k + 1] : 0.0f;
      v.z = k + 2 < K ? q[k + 2] : 0.0f;
      v.w = k + 3 < K ? q[k + 3] : 0.0f;
    }
    return v;
  };
  auto load = [&](uint32_t k0) {
#pragma unroll
    for (int j = 0; j < NA; j++) {
      const uint32_t e = t + 256 * j;
      ra[j] = row4(A, m0 + e % TA, M, k0 + 4 * (e / TA));
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const uint32_t e = t + 256 * j;
      if (TRANS_B) {
        rb[j] = row4(B, n0 + e % TB, N, k0 + 4 * (e / TB));
      } else {
        const uint32_t k = k0 + e / (TB / 4), c = n0 + 4 * (e % (TB / 4));
        const float *q = B + (size_t)(k < K ? k : K - 1) * N;
        float4 v;
        if (VEC) {
          v = *(const float4 *)(q + (c < N ? c : N - 4));
        } else {
          v.x = q[c < N ? c : N - 1];
          v.y = q[c + 1 < N ? c + 1 : N - 1];
          v.z = q[c + 2 < N ? c + 2 : N - 1];
          v.w = q[c + 3 < N ? c + 3 : N - 1];
        }
        rb[j] = k < K ? v : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int j = 0; j < NA; j++) {
      const uint32_t e = t + 256 * j, r = e % TA, k = 4 * (e / TA);
      As[buf][k][r] = ra[j].x; As[buf][k + 1][r] = ra[j].y; As[buf][k + 2][r] = ra[j].z; As[buf][k + 3][r] = ra[j].w;
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const uint32_t e = t + 256 * j, r = e % TB, k = 4 * (e / TB);
      if (TRANS_B) {
        Bs[buf][k][r] = rb[j].x; Bs[buf][k + 1][r] = rb[j].y; Bs[buf][k + 2][r] = rb[j].z; Bs[buf][k + 3][r] = rb[j].w;
      } else {
        *(float4 *)&Bs[buf][e / (TB / 4)][4 * (e % (TB / 4))] = rb[j];
      }
    }
  };
  float acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const uint32_t c = n0 + TN * tx + j;
      acc[i][j] = BIAS ? bias[c < N ? c : N - 1] : 0.0f;
    }
  struct KV {
    veca a;
    vecb b;
  };
  auto get = [&](int buf, int k) {
    return KV{*(const veca *)&As[buf][k][TM * ty], *(const vecb *)&Bs[buf][k][TN * tx]};
  };
  load(0);
  int buf = 0;
  for (uint32_t k0 = 0; k0 < K; k0 += KC, buf ^= 1) {
    const uint32_t kc = K - k0 < (uint32_t)KC ? K - k0 : (uint32_t)KC;
    put(buf);
    __syncthreads();  // the other buffer's readers passed the previous one
    if (k0 + KC < K) load(k0 + KC);
    if (ORDER == MM_SERIAL) {
      if (kc == (uint32_t)KC) {
        KV cur[KG], nxt[KG];
#pragma unroll
        for (int k = 0; k < KG; k++) cur[k] = get(buf, k);
#pragma unroll
        for (int kg = 0; kg < KC; kg += KG) {
          if (kg + KG < KC) {
#pragma unroll
            for (int k = 0; k < KG; k++) nxt[k] = get(buf, kg + KG + k);
          }
          __builtin_amdgcn_sched_barrier(0);  // keep this order: reads, then the arithmetic
#pragma unroll
          for (int k = 0; k < KG; k++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
              for (int j = 0; j < TN; j++) acc[i][j] = __fadd_rn(acc[i][j], __fmul_rn(cur[k].a[i], cur[k].b[j]));
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int k = 0; k < KG; k++) cur[k] = nxt[k];
        }
      } else {
        for (uint32_t k = 0; k < kc; k++) {
          const KV v = get(buf, k);
#pragma unroll
          for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __fadd_rn(acc[i][j], __fmul_rn(v.a[i], v.b[j]));
        }
      }
    } else {
      // kernels.el:99-104: acc + (p0 + (p1 + ... (p14 + p15))) per tile of 16, zero products past K
      for (uint32_t kb = 0; kb < kc; kb += 16) {
        float s[TM][TN];
        KV cur = get(buf, kb + 15);
#pragma unroll
        for (int q = 15; q >= 0; q--) {
          KV nxt;
          if (q) nxt = get(buf, kb + q - 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
              const float p = __fmul_rn(cur.a[i], cur.b[j]);
              s[i][j] = q == 15 ? p : __fadd_rn(p, s[i][j]);
            }
          cur = nxt;
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++) acc[i][j] = __fadd_rn(acc[i][j], s[i][j]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const uint32_t row = m0 + TM * ty + i, col = n0 + TN * tx + j;
      if (row < M && col < N && mm_covered(row, col, N, lim_mode, lim)) C[(size_t)row * N + col] = acc[i][j];
    }
}

template <int ORDER>
static void mm_go(const float *A, const float *B, const float *bias, float *C, uint32_t M, uint32_t N, uint32_t K,
                  bool trans_b, int lim_mode, uint64_t lim, hipStream_t st) {
  const dim3 g(nlg_blocks(N, MM_T), nlg_blocks(M, MM_T)), b(256);
  if (trans_b) {
    if (bias) hipLaunchKernelGGL((k_mm<ORDER, true, true>), g, b, 0, st, A, B, bias, C, M, N, K, lim_mode, lim);
    else hipLaunchKernelGGL((k_mm<ORDER, true, false>), g, b, 0, st, A, B, bias, C, M, N, K, lim_mode, lim);
  } else {
    hipLaunchKernelGGL((k_mm<ORDER, false, false>), g, b, 0, st, A, B, bias, C, M, N, K, lim_mode, lim);
  }
}

template <int TM, int TN, int ORDER, bool VEC>
static void mmt_go(const float *A, const float *B, const float *bias, float *C, uint32_t M, uint32_t N, uint32_t K,
                   bool trans_b, int lim_mode, uint64_t lim, hipStream_t st) {
  constexpr uint32_t TA = 16 * TM, TB = 16 * TN;
  const dim3 g((uint32_t)((uint64_t)((M + TA - 1) / TA) * ((N + TB - 1) / TB))), b(256);
  if (!trans_b) hipLaunchKernelGGL((k_mmt<TM, TN, ORDER, false, false, VEC>), g, b, 0, st, A, B, bias, C, M, N, K, lim_mode, lim);
  else if constexpr (ORDER == MM_SERIAL)
    hipLaunchKernelGGL((k_mmt<TM, TN, ORDER, true, true, VEC>), g, b, 0, st, A, B, bias, C, M, N, K, lim_mode, lim);
}

// whole float4s of A's and B's rows
static bool mm_vec(const float *A, const float *B, uint32_t N, uint32_t K, bool trans_b) {
  return K % 4 == 0 && (trans_b || N % 4 == 0) && (((uintptr_t)A | (uintptr_t)B) & 15) == 0;
}

template <int TM, int TN>
static void mmt(const float *A, const float *B, const float *bias, float *C, uint32_t M, uint32_t N, uint32_t K,
                bool trans_b, int order, int lim_mode, uint64_t lim, hipStream_t st) {
  const bool vec = mm_vec(A, B, N, K, trans_b);
  if (order == MM_TILE16) {
    if (vec) mmt_go<TM, TN, MM_TILE16, true>(A, B, bias, C, M, N, K, trans_b, lim_mode, lim, st);
    else mmt_go<TM, TN, MM_TILE16, false>(A, B, bias, C, M, N, K, trans_b, lim_mode, lim, st);
  } else {
    if (vec) mmt_go<TM, TN, MM_SERIAL, true>(A, B, bias, C, M, N, K, trans_b, lim_mode, lim, st);
    else mmt_go<TM, TN, MM_SERIAL, false>(A, B, bias, C, M, N, K, trans_b, lim_mode, lim, st);
  }
}

static int mm(const float *A, const float *B, const float *bias, float *C, uint32_t M, uint32_t N, uint32_t K,
              bool trans_b, int order, int lim_mode, uint64_t lim, hipStream_t st, const char *name) {
  if (!M || !N || !lim) return NLG_OK;
  if (nlg_blocks(M, MM_T) > 65535) return nlg_fail("%s: M = %u is too large", name, M);
  const bool vec = mm_vec(A, B, N, K, trans_b);
  const int form = K ? mm_tile(M, N, nlg_num_cu(), order == MM_TILE16, vec) : MM_16X16;
  if (form == MM_64X64) mmt<4, 4>(A, B, bias, C, M, N, K, trans_b, order, lim_mode, lim, st);
  else if (form == MM_64X32) mmt<4, 2>(A, B, bias, C, M, N, K, trans_b, order, lim_mode, lim, st);
  else if (form == MM_32X32) mmt<2, 2>(A, B, bias, C, M, N, K, trans_b, order, lim_mode, lim, st);
  else if (order == MM_TILE16) mm_go<MM_TILE16>(A, B, bias, C, M, N, K, trans_b, lim_mode, lim, st);
  else mm_go<MM_SERIAL>(A, B, bias, C, M, N, K, trans_b, lim_mode, lim, st);
  NLG_LAUNCHED(name);
  return NLG_OK;
}

static int mm_check(const nlg_buffer *b, uint32_t M, uint32_t K, uint32_t N, const char *k) {
  if (nlg_need(b, 0, (uint64_t)M * K, k) || nlg_need(b, 1, (uint64_t)K * N, k) ||
      nlg_need(b, 2, (uint64_t)M * N, k))
    return NLG_ERR;
  if ((uint64_t)M * N > 0xffffffffull) return nlg_fail("%s: M*N exceeds 2^32", k);
  return NLG_OK;
}

// matmul (kernels.el:17-27): A B C; push (M K N); invocation idx < M*N
// writes C[idx]
int L_matmul(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  const uint32_t M = p[0], K = p[1], N = p[2];
  if (mm_check(b, M, K, N, "matmul")) return NLG_ERR;
  return mm((const float *)b[0].ptr, (const float *)b[1].ptr, nullptr, (float *)b[2].ptr, M, N, K, false,
            MM_SERIAL, LIM_INDEX, nlg_domain((uint64_t)M * N, groups), st, "matmul");
}
// matmul-tiled (kernels.el:82-107): workgroup wg (of groups) writes C tile wg
int L_matmul_tiled(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  const uint32_t M = p[0], K = p[1], N = p[2];
  if (mm_check(b, M, K, N, "matmul-tiled")) return NLG_ERR;
  return mm((const float *)b[0].ptr, (const float *)b[1].ptr, nullptr, (float *)b[2].ptr, M, N, K, false,
            MM_TILE16, LIM_TILE16, groups, st, "matmul-tiled");
}
// matmul-reg (kernels.el:129): invocation idx writes the 4x4 block idx (row
// block idx / ceil(N/4)); the reference writes past row ends unless M and N
// are multiples of 4, so other shapes are refused.
int L_matmul_reg(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  const uint32_t M = p[0], K = p[1], N = p[2];
  if (M % 4 || N % 4) return nlg_fail("matmul-reg: M and N must be multiples of 4 (got %u, %u)", M, N);
  if (mm_check(b, M, K, N, "matmul-reg")) return NLG_ERR;
  const uint64_t blocks = (uint64_t)(M / 4) * (N / 4);
  return mm((const float *)b[0].ptr, (const float *)b[1].ptr, nullptr, (float *)b[2].ptr, M, N, K, false,
            MM_SERIAL, LIM_BLOCK4, nlg_domain(blocks, groups), st, "matmul-reg");
}
// linear (kernels.el:71-81): X W B C; push (M IN OUT); C = B + X.W^T,
// invocation idx < M*OUT writes C[idx]
int L_linear(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  const uint32_t M = p[0], IN = p[1], OUT = p[2];
  const char *k = "linear";
  if (nlg_need(b, 0, (uint64_t)M * IN, k) || nlg_need(b, 1, (uint64_t)OUT * IN, k) ||
      nlg_need(b, 2, OUT, k) || nlg_need(b, 3, (uint64_t)M * OUT, k))
    return NLG_ERR;
  if ((uint64_t)M * OUT > 0xffffffffull) return nlg_fail("linear: M*OUT exceeds 2^32");
  return mm((const float *)b[0].ptr, (const float *)b[1].ptr, (const float *)b[2].ptr, (float *)b[3].ptr, M,
            OUT, IN, true, MM_SERIAL, LIM_INDEX, nlg_domain((uint64_t)M * OUT, groups), st, k);
}
