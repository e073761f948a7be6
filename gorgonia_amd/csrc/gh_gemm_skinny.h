// The workgroups of the small-output products k_gemm_skinny16 and k_dgemm_skinny (k_gemm.hip), for the kernels that launch them
// alone and beside another product's (k_gemm_gradients.hip).
#pragma once
#include "gh_conv_common.h"
#include "gh_internal.h"

namespace gemm_skinny {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x2_a8 __attribute__((ext_vector_type(2), aligned(8)));

struct Args32 {
  const float* A; const float* B; float* C;
  int M, N, K, lda, ldb, ldc, act;
  float alpha;
  const float* bias;
  int softmax;
};

inline Args32 args32_of(const gh_cmd& c) {
  Args32 g;
  g.A = (const float*)(uintptr_t)c.ptr[0]; g.B = (const float*)(uintptr_t)c.ptr[1]; g.C = (float*)(uintptr_t)c.ptr[2];
  g.M = (int)c.dim[0]; g.N = (int)c.dim[1]; g.K = (int)c.dim[2];
  g.lda = (int)c.dim[3]; g.ldb = (int)c.dim[4]; g.ldc = (int)c.dim[5];
  g.act = (c.flags & GH_FLAG_ACT_RELU) ? 1 : (c.flags & GH_FLAG_ACT_LEAKY) ? 2 : 0;
  g.alpha = c.f[0];
  g.bias = (c.flags & GH_FLAG_GEMM_BIAS) ? (const float*)(uintptr_t)c.ptr[3] : nullptr;
  g.softmax = (c.flags & GH_FLAG_GEMM_SOFTMAX) ? 1 : 0;
  return g;
}

struct Args64 {
  const double* A; const double* B; double* C;
  int M, N, K;
  int64_t sai, sak, sbk, sbj;
  int ldc;
  int64_t sA, sB, sC;
};

inline Args64 args64_of(const gh_cmd& c) {
  const bool ta = c.flags & GH_FLAG_TRANS_A, tb = c.flags & GH_FLAG_TRANS_B, many = c.dim[6] > 1;
  Args64 g;
  g.A = (const double*)(uintptr_t)c.ptr[0]; g.B = (const double*)(uintptr_t)c.ptr[1]; g.C = (double*)(uintptr_t)c.ptr[2];
  g.M = (int)c.dim[0]; g.N = (int)c.dim[1]; g.K = (int)c.dim[2];
  g.sai = ta ? 1 : c.dim[3]; g.sak = ta ? c.dim[3] : 1;
  g.sbk = tb ? 1 : c.dim[4]; g.sbj = tb ? c.dim[4] : 1;
  g.ldc = (int)c.dim[5];
  g.sA = many ? c.dim[7] : 0; g.sB = many ? c.dim[8] : 0; g.sC = many ? c.dim[9] : 0;
  return g;
}

// ---- small-output GEMM on 16-row tiles -----------------------------------------------
// A compute unit keeps only so many cache lines in flight, which holds one
// workgroup to ~40 GB/s of operand fill however its loads are written (measured
// on the 32x32 kernel above), so a product whose 32x32 tiles cover a fraction of
// the chip is bounded by the number of compute units it touches.  This kernel
// cuts the output into tiles of 16 rows by 16*NT columns (two to four times as
// many workgroups) on the 16x16x4 MFMA; the K split over the wavefronts of a
// block and the fixed-order sum of their partial tiles are those of
// k_gemm_skinny.  Lane l = (i = l % 16, q = l / 16) owns k = 16*chunk + 4*q + t
// at MFMA step t: its four A values are one 128-bit load of row i, already in
// MFMA order; of B it takes, per k, the NT adjacent columns n0 + NT*i + c (one
// load of NT floats; with NT = 2 sixteen lanes cover one whole 128-byte line)
// and column set c feeds accumulator c.  The last tile in each direction is
// moved back to end at the matrix edge (M >= 16, N >= 16*NT), so no row or
// column is ever masked; k past K is clamped in the address and zeroed before
// the MFMA.
// TA / TB: the operand is a transposed view (A stored k x m, B stored n x k, as
// for k_sgemm); the lane's four k-values are then four loads for A and one
// 128-bit load for B instead of the other way round.  N < 16 (NT = 1 only;
// transposed views alone reach here with so few columns): one column tile,
// column indices clamped in the loads and masked in the store.
//
// Workgroup id of a grid of gx x gy tiles, slice bz of `slices` of K.  kPlain: no bias and no softmax; kGradient
// (one column tile): a softmax, and `t` behind it.
template <int WV, int NT>
constexpr int lds16() { return WV * 16 * 16 * NT * 4; }

template <int WV, int NT, bool TA, bool TB, bool kPlain, bool kGradient = false, bool kBehind = false>
__device__ __forceinline__ void workgroup16(const Args32& g, int id, int gx, int gy, int bz, int slices, char* lds,
                                            const gh_softmax_gradient<float>& t = {}, const gh_rectify_behind<float>& behind = {}) {
  const int M = g.M, N = g.N, K = g.K, lda = g.lda, ldb = g.ldb, ldc = g.ldc, act = g.act, softmax = kPlain ? 0 : kGradient ? 1 : g.softmax;
  const float alpha = g.alpha;
  const float *__restrict__ const A = g.A, *__restrict__ const B = g.B, *__restrict__ const bias = kPlain ? nullptr : g.bias;
  float* __restrict__ C = g.C;
  constexpr int G = NT == 1 ? 5 : 4;
  constexpr int BN = 16 * NT, TILE = 16 * BN;
  typedef float bvec __attribute__((ext_vector_type(NT), aligned(4)));
  float* const part = (float*)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, q = lane >> 4;
  const bool ragged_n = N < BN;
  // Workgroup ids are dealt round-robin over the 8 XCDs, each with its own L2.
  // Regroup them so that one XCD gets a contiguous run of ids, and walk a run
  // row-tile fastest: every row tile of a column tile then reads that strip of
  // B (the weights, the big operand of a dense layer) through the same L2, once
  // from memory, instead of once per XCD.
  int tile_x, tile_y;
  {
    const int total = gx * gy;
    const int xcd = id & 7, per = total >> 3, extra = total & 7;
    const int nid = xcd * per + min(xcd, extra) + (id >> 3);
    tile_x = nid / gy;
    tile_y = nid - tile_x * gy;
  }
  const int m0 = min(tile_y * 16, M - 16), n0 = ragged_n ? 0 : min(tile_x * BN, N - BN);
  const int all_chunks = (K + 15) / 16, per = (all_chunks + slices - 1) / slices;
  const int chunk0 = bz * per, nchunks = min(all_chunks, chunk0 + per);   // as in k_gemm_skinny
  C += (int64_t)bz * M * N;
  int ncol[NT];   // this lane's columns (clamped when the tile is wider than the matrix)
#pragma unroll
  for (int c = 0; c < NT; c++) ncol[c] = min(n0 + NT * i + c, N - 1);
  // k runs along the row of an untransposed A and of a transposed B
  const float* const a_base = TA ? A + m0 + i : A + (int64_t)(m0 + i) * lda;
  // The lane's quad of chunk `chunk` starts at k0 = 16*chunk + 4*q; a quad that
  // would stick out past K starts at K-4 instead, and its elements below k0
  // (which the quad before it already covers) are zeroed before the MFMA.  So
  // element t always stands for k = kb + t with kb = min(k0, K-4): every load is
  // unconditional, k-contiguous operands are one 128-bit load at any 4-byte
  // aligned address, and no loaded value is touched under a branch (which would
  // make each load wait for the one before it).
  auto load_k4 = [&](const float* row, int kb, float (&dst)[4]) {
    const f32x4 v = *reinterpret_cast<const f32x4_a4*>(row + kb);
#pragma unroll
    for (int t = 0; t < 4; t++) dst[t] = v[t];
  };
  auto load = [&](int chunk, float (&a)[4], float (&b)[4][NT]) {
    const int kb = min(chunk * 16 + 4 * q, K - 4);
    if constexpr (TA) {
#pragma unroll
      for (int t = 0; t < 4; t++) a[t] = a_base[(int64_t)(kb + t) * lda];
    } else {
      load_k4(a_base, kb, a);
    }
    if constexpr (TB) {
#pragma unroll
      for (int c = 0; c < NT; c++) {
        float col[4];
        load_k4(B + (int64_t)ncol[c] * ldb, kb, col);
#pragma unroll
        for (int t = 0; t < 4; t++) b[t][c] = col[t];
      }
    } else {
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const float* src = B + (int64_t)(kb + t) * ldb;
        if constexpr (NT == 1) {
          b[t][0] = src[ncol[0]];
        } else {
          const bvec v = *reinterpret_cast<const bvec*>(src + ncol[0]);
#pragma unroll
          for (int c = 0; c < NT; c++) b[t][c] = v[c];
        }
      }
    }
  };
  auto load_group = [&](int c, float (&a)[G][4], float (&b)[G][4][NT]) {
#pragma unroll
    for (int g = 0; g < G; g++)
      if (c + g * WV < nchunks) load(c + g * WV, a[g], b[g]);
  };
  f32x4 acc[NT];
#pragma unroll
  for (int c = 0; c < NT; c++) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mfma_group = [&](int c, float (&a)[G][4], float (&b)[G][4][NT]) {
#pragma unroll
    for (int g = 0; g < G; g++)
      if (c + g * WV < nchunks) {
        const int k0 = (c + g * WV) * 16 + 4 * q;
        const int first = k0 - min(k0, K - 4);   // elements below this index belong to the quad before
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const float av = t >= first ? a[g][t] : 0.f;
#pragma unroll
          for (int cs = 0; cs < NT; cs++) {
            const float bv = t >= first ? b[g][t][cs] : 0.f;
            acc[cs] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv, acc[cs], 0, 0, 0);
          }
        }
      }
  };
  float a0[G][4], b0[G][4][NT], a1[G][4], b1[G][4][NT];
  int c0 = chunk0 + wave;
  if (c0 < nchunks) load_group(c0, a0, b0);
  while (c0 < nchunks) {
    const int c1 = c0 + G * WV;
    if (c1 < nchunks) load_group(c1, a1, b1);
    mfma_group(c0, a0, b0);
    if (c1 >= nchunks) break;
    c0 = c1 + G * WV;
    if (c0 < nchunks) load_group(c0, a0, b0);
    mfma_group(c1, a1, b1);
  }
  // element v of accumulator c in lane (i, q) is C[m0 + 4*q + v][n0 + NT*i + c]
#pragma unroll
  for (int c = 0; c < NT; c++)
#pragma unroll
    for (int v = 0; v < 4; v++) part[wave * TILE + (4 * q + v) * BN + NT * i + c] = acc[c][v];
  __syncthreads();
  if (NT == 1 && softmax) {
    // Row softmax (N <= 16: the one column tile holds whole rows) with the
    // arithmetic of the softmax kernel: max, exp(x - max) in float64 rounded
    // once, the sum taken in column order, one rounded reciprocal.
    __shared__ float sm_x[16 * 17], sm_e[16 * 17];
    const int e = threadIdx.x, row = (e >> 4) & 15, col = e & 15;
    if (e < TILE) {
      float sum = part[e];
#pragma unroll
      for (int w = 1; w < WV; w++) sum = sum + part[w * TILE + e];
      if (bias && col < N) sum = sum + bias[col];
      sm_x[row * 17 + col] = act_apply(sum, act, alpha);
    }
    __syncthreads();
    if (e < TILE) {
      float mx = -INFINITY;
      for (int j = 0; j < N; j++) mx = fmaxf(mx, sm_x[row * 17 + j]);
      sm_e[row * 17 + col] = col < N ? (float)exp((double)(sm_x[row * 17 + col] - mx)) : 0.f;
    }
    __syncthreads();
    if (e < TILE && col < N) {
      float sum = 0.f;
      for (int j = 0; j < N; j++) sum = sum + sm_e[row * 17 + j];
      const float inv = 1.0f / sum, y = sm_e[row * 17 + col] * inv;
      C[(int64_t)(m0 + row) * ldc + col] = y;
      if constexpr (kGradient) {
        const int64_t at = (int64_t)(m0 + row) * N + col;
        const float v = t.x[at] * *t.s;
        sm_x[row * 17 + col] = v * y;   // (a row's 16 threads are of one wavefront, which is past its reads of sm_x)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        float dot = 0.f;
        for (int j = 0; j < N; j++) dot = dot + sm_x[row * 17 + j];
        const float d = v - dot;
        if (m0 + row >= tile_y * 16) {   // (the last tile's first rows are the one's before it, where x may be g)
          t.g[at] = v;
          t.dx[at] = y * d;
        }
      }
    }
    return;
  }
  constexpr int kRounds = (TILE + WV * 64 - 1) / (WV * 64);
  [[maybe_unused]] float loaded[kRounds];
  if constexpr (kBehind) {
#pragma unroll
    for (int k = 0; k < kRounds; k++) {
      const int e = (int)threadIdx.x + k * WV * 64, col = n0 + e % BN;
      loaded[k] = e < TILE && col < N ? behind.load((int64_t)(m0 + e / BN) * ldc + col) : 0.0f;
    }
  }
#pragma unroll
  for (int k = 0; k < kRounds; k++) {
    const int e = (int)threadIdx.x + k * WV * 64;
    if (e >= TILE) break;
    float sum = part[e];
#pragma unroll
    for (int w = 1; w < WV; w++) sum = sum + part[w * TILE + e];
    const int col = n0 + e % BN;
    if (col >= N) continue;
    if (bias) sum = sum + bias[col];
    const int64_t at = (int64_t)(m0 + e / BN) * ldc + col;
    if constexpr (kBehind) behind.store(C, at, act_apply(sum, act, alpha), loaded[k]);
    else C[at] = act_apply(sum, act, alpha);
  }
}

// Float64 product with a small result (a dense layer on a batch: too few 64x64
// tiles to occupy the device, and a k loop of a thousand steps behind each).
// One workgroup per 16x16 tile of C, its WV wavefronts each summing a slice of
// K straight from global memory into one MFMA accumulator (element (i, k) of
// op(A) at A[i*sai + k*sak], (k, j) of op(B) at B[k*sbk + j*sbj], so every
// transpose is the same code); loads are unconditional at clamped addresses and
// masked afterwards, so they all stay in flight.  The slices are added in LDS in
// wavefront order: the result does not depend on scheduling.
//
// Tile bx, by of product bz of a batch.
template <int WV>
constexpr int lds64() { return WV * 256 * 8; }

template <int WV, bool AV, bool BV, bool kBehind = false>
__device__ __forceinline__ void workgroup64(const Args64& g, int bx, int by, int bz, char* lds, const gh_rectify_behind<double>& behind = {}) {
  const double* __restrict__ const A = g.A + bz * g.sA;
  const double* __restrict__ const B = g.B + bz * g.sB;
  double* __restrict__ const C = g.C + bz * g.sC;
  const int M = g.M, N = g.N, K = g.K, ldc = g.ldc;
  const int64_t sai = g.sai, sak = g.sak, sbk = g.sbk, sbj = g.sbj;
  double (* const part)[256] = (double (*)[256])lds;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int m0 = by * 16, n0 = bx * 16;
  const double* ap = A + (int64_t)min(m0 + lr, M - 1) * sai;
  const double* bp = B + (int64_t)min(n0 + lr, N - 1) * sbj;
  const int kper = (((K + WV - 1) / WV) + 7) & ~7;
  const int k0 = wave * kper, k1 = min(K, k0 + kper);
  f64x4 acc = {0.0, 0.0, 0.0, 0.0};
  if constexpr (AV || BV) {
    // An operand that is k-contiguous: a lane fetches two consecutive k of its row or column in one load (the
    // sixteen k of a step are then two 64-byte pieces instead of sixteen 8-byte ones; 8-byte alignment is all
    // the load needs); which k a lane group multiplies in which MFMA is the same for both operands -
    // k0 + 8 u + 2 lk + e.  The pair that would start at the last k of an odd K starts one earlier and is
    // shifted into place.
    for (int k = k0; k < k1; k += 16) {
      f64x2 a[2], b[2];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int kk = k + 8 * u + 2 * lk;
        const bool last = kk > K - 2;   // kk == K - 1 (its second k does not exist), or past the end (masked below)
        if constexpr (AV) {
          const f64x2 v = *reinterpret_cast<const f64x2_a8*>(ap + min(kk, K - 2));
          a[u] = last ? f64x2{v[1], 0.0} : v;
        }
        if constexpr (BV) {
          const f64x2 v = *reinterpret_cast<const f64x2_a8*>(bp + min(kk, K - 2));
          b[u] = last ? f64x2{v[1], 0.0} : v;
        }
#pragma unroll
        for (int e = 0; e < 2; e++) {
          if constexpr (!AV) a[u][e] = ap[(int64_t)min(kk + e, K - 1) * sak];
          if constexpr (!BV) b[u][e] = bp[(int64_t)min(kk + e, K - 1) * sbk];
        }
      }
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const bool ok = k + 8 * u + 2 * lk + e < k1;
          const double av = ok ? a[u][e] : 0.0, bv = ok ? b[u][e] : 0.0;
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc, 0, 0, 0);
        }
    }
  } else {
    for (int k = k0; k < k1; k += 16) {
      double a[4], b[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int kc = min(k + 4 * u + lk, K - 1);
        a[u] = ap[kc * sak];
        b[u] = bp[kc * sbk];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const bool ok = k + 4 * u + lk < k1;
        a[u] = ok ? a[u] : 0.0;
        b[u] = ok ? b[u] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; u++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[u], acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int v = 0; v < 4; v++) part[wave][v * 64 + lane] = acc[v];
  __syncthreads();
  if (wave == 0) {
    [[maybe_unused]] double loaded[4];
    if constexpr (kBehind) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int i = m0 + 4 * v + lk, j = n0 + lr;
        loaded[v] = i < M && j < N ? behind.load((int64_t)i * ldc + j) : 0.0;
      }
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
      double sum = part[0][v * 64 + lane];
      for (int w = 1; w < WV; w++) sum = sum + part[w][v * 64 + lane];
      const int i = m0 + 4 * v + lk, j = n0 + lr;
      if (i >= M || j >= N) continue;
      if constexpr (kBehind) behind.store(C, (int64_t)i * ldc + j, sum, loaded[v]);
      else C[(int64_t)i * ldc + j] = sum;
    }
  }
}

}  // namespace gemm_skinny
