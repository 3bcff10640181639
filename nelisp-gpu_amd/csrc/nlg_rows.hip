// nlg_rows.hip -- row reductions: softmax, RMSNorm (istd, per-head).
//
// The reference gives each row to one invocation, which walks it serially
// three times (softmax, kernels.el:28-42).  Here a wave or a workgroup owns a
// row (softmax_threads): it is read from HBM once into registers (16 floats per
// thread at 4096 columns, non-temporal float4 loads), reduced with DPP within
// waves and LDS across them, and written once (non-temporal stores) -- 8 bytes of
// traffic per element, the minimum for an in-place softmax; only rows of more than
// 32,768 columns are read three times.  Reduction order differs from the serial
// reference, so parity is by tolerance (<= 1e-5 relative for softmax, 1e-4 for
// RMSNorm).
#include <math.h>

#include "nlg_internal.h"
#include "nlg_softmax_form.h"

#define EPS6 0.000001f

// Sum over the 16 waves of a workgroup, in every thread.  The waves' sums meet in
// pairs: added one after another, each of 15 sums as large as the result is rounded, and
// rows whose weight lies in a few waves (causal ones) show it.
__device__ __forceinline__ float block_sum16(float v, float *red) {
  v = nlg_wave_sum_f32(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t[16];
#pragma unroll
  for (int i = 0; i < 16; i++) t[i] = red[i];
#pragma unroll
  for (int n = 8; n; n /= 2)
#pragma unroll
    for (int i = 0; i < n; i++) t[i] = t[2 * i] + t[2 * i + 1];
  return t[0];
}

// The reference's max starts from the first element and only moves on a
// strict `>`: NaNs are never selected, except that a NaN first element stays.
// TPR threads take a row and hold EPT of its values each: a wave (no LDS, no
// barrier; four rows a workgroup), a workgroup of 256 or one of 1,024.
template <int TPR, int EPT, bool V4>
__global__ __launch_bounds__(TPR < 256 ? 256 : TPR) void k_softmax_reg(const float *a, float *c, uint32_t rows,
                                                                      uint32_t n) {
  __shared__ float red[TPR < 256 ? 1 : TPR / 64];
  constexpr bool WAVE = TPR == 64;
  constexpr bool PAIRS = WAVE && V4 && EPT == 16;  // a lane's chain as long as with four times the lanes
  const uint32_t tid = threadIdx.x % TPR;
  const uint32_t row = WAVE ? blockIdx.x * 4 + threadIdx.x / 64 : blockIdx.x;
  if (row >= rows) return;
  const float *ar = a + (size_t)row * n;
  float *cr = c + (size_t)row * n;
  const float first = ar[0];
  float v[EPT];
  float mx = -INFINITY;
  if (V4) {
#pragma unroll
    for (int k = 0; k < EPT / 4; k++) {
      const uint32_t i4 = tid + TPR * k;
      float4 q = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
      if (4 * i4 < n) q = nlg_ld_stream_f4((const float4 *)ar + i4);
      v[4 * k] = q.x; v[4 * k + 1] = q.y; v[4 * k + 2] = q.z; v[4 * k + 3] = q.w;
    }
  } else {
#pragma unroll
    for (int k = 0; k < EPT; k++) {
      const uint32_t i = tid + TPR * k;
      v[k] = i < n ? ar[i] : -INFINITY;
    }
  }
#pragma unroll
  for (int k = 0; k < EPT; k++) mx = v[k] > mx ? v[k] : mx;
  mx = WAVE ? nlg_wave_max_f32(mx) : nlg_block_max_f32(mx, red);
  if (first != first) mx = first;
  float s = 0.0f;
#pragma unroll
  for (int k = 0; k < EPT; k++) {
    const uint32_t i = V4 ? 4 * (tid + TPR * (k / 4)) + (k % 4) : tid + TPR * k;
    v[k] = expf(__fsub_rn(v[k], mx));
    if (PAIRS) {
      if (k % 4 == 3 && i < n) s += (v[k - 3] + v[k - 2]) + (v[k - 1] + v[k]);
    } else if (i < n) {
      s = __fadd_rn(s, v[k]);
    }
  }
  s = WAVE ? nlg_wave_sum_f32(s) : TPR == 1024 ? block_sum16(s, red) : nlg_block_sum_f32(s, red);
  if (V4) {
#pragma unroll
    for (int k = 0; k < EPT / 4; k++) {
      const uint32_t i4 = tid + TPR * k;
      if (4 * i4 < n)
        nlg_st_stream_f4((float4 *)cr + i4,
                         make_float4(v[4 * k] / s, v[4 * k + 1] / s, v[4 * k + 2] / s, v[4 * k + 3] / s));
    }
  } else {
#pragma unroll
    for (int k = 0; k < EPT; k++) {
      const uint32_t i = tid + TPR * k;
      if (i < n) cr[i] = v[k] / s;
    }
  }
}

// Rows too long for registers: three streaming passes, same semantics.
__global__ __launch_bounds__(256) void k_softmax_stream(const float *a, float *c, uint32_t rows,
                                                        uint32_t n) {
  __shared__ float red[4];
  const uint32_t row = blockIdx.x;
  if (row >= rows) return;
  const float *ar = a + (size_t)row * n;
  float *cr = c + (size_t)row * n;
  const float first = ar[0];
  float mx = -INFINITY;
  for (uint32_t i = threadIdx.x; i < n; i += 256) mx = ar[i] > mx ? ar[i] : mx;
  mx = nlg_block_max_f32(mx, red);
  if (first != first) mx = first;
  float s = 0.0f;
  for (uint32_t i = threadIdx.x; i < n; i += 256) s = __fadd_rn(s, expf(__fsub_rn(ar[i], mx)));
  s = nlg_block_sum_f32(s, red);
  // each element is read by the thread that then overwrites it: in-place safe
  for (uint32_t i = threadIdx.x; i < n; i += 256) cr[i] = expf(__fsub_rn(ar[i], mx)) / s;
}

static int launch_softmax(const float *a, float *c, uint32_t rows, uint32_t n, hipStream_t st) {
  if (!rows || !n) return NLG_OK;
  const bool v4 = (n % 4 == 0) && ((((uintptr_t)a) | ((uintptr_t)c)) & 15) == 0;
  const uint32_t tpr = softmax_threads(rows, n, v4, nlg_num_cu());
#define SM(TPR, EPT)                                                                                   \
  do {                                                                                                 \
    const dim3 g(TPR == 64 ? (uint32_t)(((uint64_t)rows + 3) / 4) : rows), b(TPR == 64 ? 256 : TPR);   \
    if (v4) hipLaunchKernelGGL((k_softmax_reg<TPR, EPT, true>), g, b, 0, st, a, c, rows, n);           \
    else hipLaunchKernelGGL((k_softmax_reg<TPR, EPT, false>), g, b, 0, st, a, c, rows, n);             \
  } while (0)
  if (tpr == 64) {
    if (n <= 64 * 4) SM(64, 4);
    else SM(64, 16);
  } else if (tpr == 256) {
    if (n <= 256 * 4) SM(256, 4);
    else if (n <= 256 * 8) SM(256, 8);
    else if (n <= 256 * 16) SM(256, 16);
    else SM(256, 32);
  } else if (tpr == 1024) {
    if (n <= 1024 * 16) SM(1024, 16);
    else SM(1024, 32);
  } else {
    hipLaunchKernelGGL(k_softmax_stream, dim3(rows), dim3(256), 0, st, a, c, rows, n);
  }
#undef SM
  NLG_LAUNCHED("softmax");
  return NLG_OK;
}

extern "C" int nlg_softmax_rows(const float *a, float *c, uint32_t rows, uint32_t cols, void *stream) {
  if (nlg_ensure_init()) return NLG_ERR;
  return launch_softmax(a, c, rows, cols, nlg_stream(stream));
}

// softmax by name: A C; push (M N)
int L_softmax(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  const uint32_t M = p[0], N = p[1];
  const uint64_t rows = nlg_domain(M, groups);
  if (nlg_need(b, 0, rows * N, "softmax") || nlg_need(b, 1, rows * N, "softmax")) return NLG_ERR;
  if ((uint64_t)M * N > 0xffffffffull) return nlg_fail("softmax: M*N exceeds 2^32 elements");
  return launch_softmax((const float *)b[0].ptr, (float *)b[1].ptr, (uint32_t)rows, N, st);
}

// rmsnorm-istd (kernels.el:1249-1256): S[r] = 1/sqrt(sum(x^2)/N + 1e-6)
__global__ __launch_bounds__(256) void k_rmsnorm_istd(const float *x, float *s, uint32_t rows,
                                                      uint32_t n) {
  __shared__ float red[4];
  const uint32_t row = blockIdx.x;
  if (row >= rows) return;
  const float *xr = x + (size_t)row * n;
  float ss = 0.0f;
  for (uint32_t i = threadIdx.x; i < n; i += 256) ss = __fadd_rn(ss, __fmul_rn(xr[i], xr[i]));
  ss = nlg_block_sum_f32(ss, red);
  if (threadIdx.x == 0) s[row] = 1.0f / sqrtf(__fadd_rn(ss / (float)n, EPS6));
}

int L_rmsnorm_istd(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  const uint32_t M = p[0], N = p[1];
  const uint64_t rows = nlg_domain(M, groups);
  if (nlg_need(b, 0, rows * N, "rmsnorm-istd") || nlg_need(b, 1, rows, "rmsnorm-istd")) return NLG_ERR;
  if (!rows) return NLG_OK;
  hipLaunchKernelGGL(k_rmsnorm_istd, dim3((uint32_t)rows), dim3(256), 0, st, (const float *)b[0].ptr,
                     (float *)b[1].ptr, (uint32_t)rows, N);
  NLG_LAUNCHED("rmsnorm-istd");
  return NLG_OK;
}

// rmsnorm-heads (kernels.el:823-842): one wave per (position, head) row.
__global__ __launch_bounds__(256) void k_rmsnorm_heads(const float *x, const float *g, float *y,
                                                       uint32_t nrows, uint32_t hd) {
  const int lane = threadIdx.x & 63;
  const uint64_t r = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= nrows) return;
  const float *xr = x + r * hd;
  float ss = 0.0f;
  for (uint32_t i = lane; i < hd; i += 64) ss = __fadd_rn(ss, __fmul_rn(xr[i], xr[i]));
  ss = nlg_wave_sum_f32(ss);
  const float inv = 1.0f / sqrtf(__fadd_rn(ss / (float)hd, EPS6));
  for (uint32_t j = lane; j < hd; j += 64) y[r * hd + j] = __fmul_rn(__fmul_rn(xr[j], inv), g[j]);
}

int L_rmsnorm_heads(const nlg_buffer *b, const uint32_t *p, uint32_t groups, hipStream_t st) {
  const uint32_t seq = p[0], nheads = p[1], hd = p[2];
  const uint64_t rows = nlg_domain((uint32_t)(seq * nheads), groups);
  const char *k = "rmsnorm-heads";
  if (nlg_need(b, 0, rows * hd, k) || nlg_need(b, 1, rows ? hd : 0, k) || nlg_need(b, 2, rows * hd, k))
    return NLG_ERR;
  if (!rows) return NLG_OK;
  hipLaunchKernelGGL(k_rmsnorm_heads, dim3(nlg_blocks(rows, 4)), dim3(256), 0, st,
                     (const float *)b[0].ptr, (const float *)b[1].ptr, (float *)b[2].ptr,
                     (uint32_t)rows, hd);
  NLG_LAUNCHED(k);
  return NLG_OK;
}
