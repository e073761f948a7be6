// Products of one to four rows (float64: one or two) with a row-major matrix: y[m][:] = x[m][:] . B, float32 and float64.
//
// A pass over B and nothing else, so a workgroup takes 16 columns (of float64 the same 16) and all of K: lane (kk, cg)
// of a wavefront reads four neighbouring columns of every 128th row, 4 rows or more in flight, and the 128 partial sums
// of a result meet in the wavefront and then in LDS, in a fixed order.  The MFMA kernels give 32 columns to a workgroup
// and all rows of a 16- or 32-row tile to the matrix cores, of which one to four hold anything; their walk over K is
// eight times as long.  Bound by the latency of its two or three rounds of loads and the launch.
// 1 x 784 . 784 x 300 with x in pinned host memory: 8.6 us (14.2); 1 x 300 . 300 x 100: 3.8 (4.7).
#include <cstdlib>

#include "gh_conv_common.h"
#include "gh_internal.h"

namespace {

constexpr int kWaves = 8, kRows = kWaves * 16;

template <class T, int MT>
__global__ __launch_bounds__(kWaves * 64) void k_gemm_thin(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int M, int N, int K,
                                                           int lda, int ldb, int ldc, const T* __restrict__ bias, int act, float alpha) {
  typedef T V __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  constexpr int U = MT <= 2 && sizeof(T) == 4 ? 8 : 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, cg = lane & 3;
  const int k0 = wave * 16 + (lane >> 2);
  // the last group of four columns is moved left to end with the row
  const T* const b = B + min((int)blockIdx.x * 16 + 4 * cg, N - 4);
  T acc[MT][4];
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int e = 0; e < 4; e++) acc[m][e] = (T)0;
  for (int kb = 0; kb < K; kb += U * kRows) {
    V w[U];
    T x[U][MT];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = min(kb + u * kRows + k0, K - 1);
      w[u] = *(const V*)(b + (int64_t)k * ldb);
#pragma unroll
      for (int m = 0; m < MT; m++) x[u][m] = A[(int64_t)min(m, M - 1) * lda + k];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool in = kb + u * kRows + k0 < K;
#pragma unroll
      for (int m = 0; m < MT; m++) {
        const T xv = in ? x[u][m] : (T)0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const T wv = in ? w[u][e] : (T)0;
          if constexpr (sizeof(T) == 4) acc[m][e] = __builtin_fmaf(xv, wv, acc[m][e]);
          else acc[m][e] = __builtin_fma(xv, wv, acc[m][e]);
        }
      }
    }
  }
  __shared__ T red[kWaves][MT * 16];
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      T v = acc[m][e];
#pragma unroll
      for (int off = 4; off < 64; off <<= 1) v = v + __shfl_xor(v, off, 64);
      if (lane < 4) red[wave][m * 16 + 4 * cg + e] = v;
    }
  __syncthreads();
  const int t = threadIdx.x, m = t >> 4, j = t & 15;
  if (t < MT * 16 && m < M) {
    T sum = red[0][t];
#pragma unroll
    for (int w = 1; w < kWaves; w++) sum = sum + red[w][t];
    const int col = min((int)blockIdx.x * 16 + (j & 12), N - 4) + (j & 3);
    if constexpr (sizeof(T) == 4) {
      if (bias) sum = sum + bias[col];
      sum = act_apply(sum, act, alpha);
    }
    C[(int64_t)m * ldc + col] = sum;
  }
}

template <class T>
int launch(gh_ctx* ctx, const gh_cmd& c) {
  const int M = (int)c.dim[0], N = (int)c.dim[1], K = (int)c.dim[2];
  const T* bias = (c.flags & GH_FLAG_GEMM_BIAS) ? (const T*)(uintptr_t)c.ptr[3] : nullptr;
  const int act = (c.flags & GH_FLAG_ACT_RELU) ? 1 : (c.flags & GH_FLAG_ACT_LEAKY) ? 2 : 0;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((N + 15) / 16)), dim3(kWaves * 64), 0, ctx->stream, (const T*)(uintptr_t)c.ptr[0],
                       (const T*)(uintptr_t)c.ptr[1], (T*)(uintptr_t)c.ptr[2], M, N, K, (int)c.dim[3], (int)c.dim[4], (int)c.dim[5], bias, act, c.f[0]);
  };
  if (M == 1) go(k_gemm_thin<T, 1>);
  else if (M == 2) go(k_gemm_thin<T, 2>);
  else if constexpr (sizeof(T) == 4) go(k_gemm_thin<T, 4>);
  return gh_check_hip(ctx, hipGetLastError(), "thin gemm launch");
}

}  // namespace

// One product of up to four rows (two of float64: every row adds its partial sums' way through the wavefront, and at
// eight rows, 8 x 300 x 100, that made 7.3 us of 4.9), operands as they lie, wider than a softmax in a product's epilogue
// (up to 32 columns: the fused and the separate softmax see the same product bits there) and not so wide that 32-column
// tiles fill the device (1 x 1000 x 8000: 14.3 us against 12.3), K long enough for a row per lane, with several rows for
// two (4 x 64 x 100: 4.8 us against 3.9; 4 x 300 x 100 4.8 and 4.9; 4 x 784 x 300 5.4 against 8.4) and, where few
// workgroups share the columns, not so long that cutting it over workgroups pays for a second launch.
bool gh_gemm_thin_takes(const gh_cmd& c) {
  if (c.dim[6] > 1 || (c.flags & (GH_FLAG_TRANS_A | GH_FLAG_TRANS_B | GH_FLAG_GEMM_SOFTMAX))) return false;
  const int64_t rows = gh_dtype_of(c.flags) == GH_F64 ? 2 : 4;
  return c.dim[0] >= 1 && c.dim[0] <= rows && c.dim[1] > 32 && c.dim[1] <= 4096 && c.dim[2] >= (c.dim[0] == 1 ? 64 : 256) && (c.dim[2] <= 4096 || c.dim[1] >= 2048) &&
         !getenv("GORGONIA_HIP_GEMM_PLAN");
}
int gh_launch_gemm_thin(gh_ctx* ctx, const gh_cmd& c) {
  return gh_dtype_of(c.flags) == GH_F64 ? launch<double>(ctx, c) : launch<float>(ctx, c);
}
