// The workgroup of k_gemm_direct (k_gemm_direct.hip says how it works), for the kernels that launch it alone and beside another
// product's (k_gemm_gradients.hip).
#pragma once
#include <algorithm>

#include "gh_conv_common.h"
#include "gh_internal.h"
#include "gh_schedule.h"

namespace gemm_direct {

template <class T> struct Unit;
template <> struct Unit<double> {
  typedef double acc __attribute__((ext_vector_type(4)));
  typedef double vec __attribute__((ext_vector_type(2), aligned(8)));
  static constexpr int KQ = 2;
  static __device__ __forceinline__ acc mfma(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int q, int v) { return 4 * v + q; }   // result row of register v in lanes q
};

template <> struct Unit<float> {
  typedef float acc __attribute__((ext_vector_type(4)));
  typedef float vec __attribute__((ext_vector_type(4), aligned(4)));
  static constexpr int KQ = 4;
  static __device__ __forceinline__ acc mfma(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int q, int v) { return 4 * q + v; }
};

template <class T>
struct Gemm {
  const T* A; const T* B; T* C;
  int M, N, K, lda, ldb, ldc;
  int64_t sA, sB, sC;
  const T* bias;   // one value per column, or null
  int act;
  float alpha;
};

template <class T>
inline Gemm<T> gemm_of(const gh_cmd& c, int* batch) {
  Gemm<T> g;
  g.A = (const T*)(uintptr_t)c.ptr[0]; g.B = (const T*)(uintptr_t)c.ptr[1]; g.C = (T*)(uintptr_t)c.ptr[2];
  g.M = (int)c.dim[0]; g.N = (int)c.dim[1]; g.K = (int)c.dim[2];
  g.lda = (int)c.dim[3]; g.ldb = (int)c.dim[4]; g.ldc = (int)c.dim[5];
  *batch = c.dim[6] <= 0 ? 1 : (int)c.dim[6];
  g.sA = *batch > 1 ? c.dim[7] : 0; g.sB = *batch > 1 ? c.dim[8] : 0; g.sC = *batch > 1 ? c.dim[9] : 0;
  g.bias = (c.flags & GH_FLAG_GEMM_BIAS) ? (const T*)(uintptr_t)c.ptr[3] : nullptr;
  g.act = (c.flags & GH_FLAG_ACT_RELU) ? 1 : (c.flags & GH_FLAG_ACT_LEAKY) ? 2 : 0;
  g.alpha = c.f[0];
  return g;
}

// One operand of a tile: TT tiles of 16 rows (of A; of B, columns), rows r0 and up, rmax of them in all.
// KC: k runs along memory.  Rows past the end are the last row again; their results are not stored.
template <class T, int TT, bool kAlongK>
struct Operand {
  static constexpr int KQ = Unit<T>::KQ, V = KQ;
  static constexpr int G = kAlongK ? 0 : TT / V, S = kAlongK ? TT : TT % V;   // groups of V tiles, single tiles
  typedef typename Unit<T>::vec vec;
  static constexpr int kLoads = kAlongK ? TT : KQ * (G + S);
  unsigned off[G + S];   // bytes from the tile's base at k = 0
  int ld;

  // the tile's base is its first row (the last V rows' first, where fewer are left)
  static __device__ __forceinline__ int base_row(int r0, int rmax) { return min(r0, rmax - V); }
  __device__ __forceinline__ const T* init(const T* p, int r0, int rmax, int ld_, int i, int q) {
    ld = ld_;
    const int rb = base_row(r0, rmax);
#pragma unroll
    for (int g = 0; g < G; g++) off[g] = (unsigned)((min(r0 + 16 * V * g + V * i, rmax - V) - rb + KQ * q * ld) * (int)sizeof(T));
#pragma unroll
    for (int s = 0; s < S; s++) {
      const int r = min(r0 + 16 * (V * G + s) + i, rmax - 1) - rb;
      off[G + s] = (unsigned)((kAlongK ? r * ld + KQ * q : r + KQ * q * ld) * (int)sizeof(T));
    }
    return p + (kAlongK ? (int64_t)rb * ld : (int64_t)rb);
  }
  // row of tile t that lane i' holds (the inverse of off, for the stores)
  static __device__ __forceinline__ int row(int t, int i, int r0, int rmax) {
    if (!kAlongK && t < V * G) return min(r0 + 16 * V * (t / V) + V * i, rmax - V) + t % V;
    return r0 + 16 * t + i;
  }
  __device__ __forceinline__ void load(const T* base, int k0, T (&v)[TT][KQ]) const {
    const char* p = (const char*)(base + (kAlongK ? (int64_t)k0 : (int64_t)k0 * ld));
    if constexpr (kAlongK) {
#pragma unroll
      for (int t = 0; t < TT; t++) {
        const vec x = *(const vec*)(p + off[t]);
#pragma unroll
        for (int e = 0; e < KQ; e++) v[t][e] = x[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < KQ; e++) {
        const char* pe = p + (int64_t)e * ld * (int)sizeof(T);
#pragma unroll
        for (int g = 0; g < G; g++) {
          const vec x = *(const vec*)(pe + off[g]);
#pragma unroll
          for (int u = 0; u < V; u++) v[V * g + u][e] = x[u];
        }
#pragma unroll
        for (int s = 0; s < S; s++) v[V * G + s][e] = *(const T*)(pe + off[G + s]);
      }
    }
  }
  // the last, partial chunk: k past K are zero
  __device__ __forceinline__ void load_tail(const T* base, int k0, int K, int q, T (&v)[TT][KQ]) const {
#pragma unroll
    for (int e = 0; e < KQ; e++) {
      const int k = k0 + KQ * q + e, back = max(k - (K - 1), 0);   // k moved back inside
      const char* p = (const char*)(base + (kAlongK ? (int64_t)k0 : (int64_t)k0 * ld)) + (int64_t)(e - back) * (kAlongK ? 1 : ld) * (int)sizeof(T);
#pragma unroll
      for (int t = 0; t < TT; t++) {
        const T x = !kAlongK && t < V * G ? *(const T*)(p + off[t / V] + (t % V) * sizeof(T)) : *(const T*)(p + off[kAlongK ? t : G + t - V * G]);
        v[t][e] = k < K ? x : (T)0;
      }
    }
  }
};

// The memory the wavefronts' sums meet in.
template <class T, int kWaves, int TN, bool kSplitK>
constexpr int lds_of() { return kSplitK ? kWaves * TN * 256 * (int)sizeof(T) : 16; }

// Workgroup id of a grid of gx x gy tiles; bz: which product of a batch.
template <class T, int kWaves, int TM, int TN, bool kSplitK, bool kTA, bool kTB, bool kBehind = false>
__device__ __forceinline__ void workgroup(const Gemm<T>& g, int id, int gx, int gy, int bz, char* lds, const gh_rectify_behind<T>& behind = {}) {
  typedef typename Unit<T>::acc Acc;
  constexpr int KQ = Unit<T>::KQ, KC = 4 * KQ, kThreads = kWaves * 64;
  typedef Operand<T, TM, !kTA> OpA;
  typedef Operand<T, TN, kTB> OpB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, q = lane >> 4;
  // Workgroup ids are dealt round-robin over eight XCDs with an L2 each: give an XCD a contiguous run of tiles, and
  // walk it in groups of eight tile rows so that the tiles under way share rows of A and columns of B.
  int tm, tn;
  {
    const int total = gx * gy;
    const int xcd = id & 7, per = total >> 3, extra = total & 7;
    const int nid = xcd * per + min(xcd, extra) + (id >> 3);
    const int group = 8 * gx, first = nid / group * 8, rows = min(gy - first, 8), in = nid % group;
    tm = first + in % rows;
    tn = in / rows;
  }
  const int m0 = kSplitK ? tm * 16 * TM : (tm * kWaves + wave) * 16 * TM, n0 = tn * 16 * TN;
  if (!kSplitK && m0 >= g.M) return;   // (no barrier in this form)
  T* const C = g.C + bz * g.sC;
  OpA oa;
  OpB ob;
  const T* const A = oa.init(g.A + bz * g.sA, m0, g.M, g.lda, i, q);
  const T* const B = ob.init(g.B + bz * g.sB, n0, g.N, g.ldb, i, q);

  Acc acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++) acc[a][b] = Acc{(T)0, (T)0, (T)0, (T)0};
  struct Frag { T a[TM][KQ]; T b[TN][KQ]; };
  auto multiply = [&](const Frag& f) {
#pragma unroll
    for (int e = 0; e < KQ; e++)
#pragma unroll
      for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) acc[a][b] = Unit<T>::mfma(f.a[a][e], f.b[b][e], acc[a][b]);
  };
  const int full = g.K / KC;   // whole chunks
  Frag even, odd;
  const int first = kSplitK ? 2 * wave : 0;
  if (first < full) {
    // The loads of a chunk are in flight under the MFMAs of the chunk before: two sets of operands taken in turn, each load
    // behind a few MFMAs (gh_schedule.h).  us, before / now: 1226 x 1746, K = 1128 59.1 / 47.0, 1978 x 577, K = 4027 110 / 87, 311 x 993,
    // K = 1190 16.5 / 13.2; float64 113 x 1444, K = 1480 24.3 / 21.1, 291 x 1153, K = 895 19.7 / 17.9; of 150 drawn products of 2e7 multiplications
    // and more, 0.97 of the time together, none slower by more than the launches of one differ.
    // A wavefront has chunks 2 w and 2 w + 1 of every 2 kWaves (all chunks where K is not split).
    constexpr int kPair = kSplitK ? 2 * kWaves : 2, kLoads = OpA::kLoads + OpB::kLoads, kMacs = KQ * TM * TN;
    auto load = [&](int chunk, Frag& f) __attribute__((always_inline)) {
      oa.load(A, chunk * KC, f.a);
      ob.load(B, chunk * KC, f.b);
    };
    auto turn = [&](int ahead, const Frag& now, Frag& next) __attribute__((always_inline)) {
      load(min(ahead, full - 1), next);   // (past the end: no branch around the loads)
      multiply(now);
      gh_spread_loads<kLoads, kMacs>();
      __builtin_amdgcn_sched_barrier(0);
    };
    load(first, even);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // the loop is entered with nothing in flight, so its waits count its own loads only
    int c = first;
    for (; c + 1 < full; c += kPair) {   // (one way out: where paths meet the compiler waits for the worst of them)
      turn(c + 1, even, odd);
      turn(c + kPair, odd, even);
    }
    if (c < full) multiply(even);
  }
  if (g.K % KC && (!kSplitK || wave == full % (2 * kWaves) / 2)) {
    oa.load_tail(A, full * KC, g.K, q, even.a);
    ob.load_tail(B, full * KC, g.K, q, even.b);
    multiply(even);
  }

  auto store = [&](int r, int c, T sum, T loaded) {
    if (r >= g.M || c >= g.N) return;
    if constexpr (sizeof(T) == 4) {
      if (g.bias) sum = sum + g.bias[c];
      sum = act_apply(sum, g.act, g.alpha);
    }
    if constexpr (kBehind) behind.store(C, (int64_t)r * g.ldc + c, sum, loaded);
    else C[(int64_t)r * g.ldc + c] = sum;
  };
  auto load = [&](int r, int c) {
    if constexpr (kBehind) return r < g.M && c < g.N ? behind.load((int64_t)r * g.ldc + c) : (T)0;
    else return (T)0;
  };
  if constexpr (kSplitK) {
    T (* const red)[TN * 256] = (T (*)[TN * 256])lds;
    constexpr int kRounds = (TN * 256 + kThreads - 1) / kThreads;
#pragma unroll
    for (int a = 0; a < TM; a++) {
      if (a) __syncthreads();
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) red[wave][b * 256 + v * 64 + lane] = acc[a][b][v];
      auto row = [&](int e) { return OpA::row(a, Unit<T>::row((e & 63) >> 4, (e >> 6) & 3), m0, g.M); };
      auto col = [&](int e) { return OpB::row(e >> 8, e & 15, n0, g.N); };
      T loaded[kRounds];
#pragma unroll
      for (int k = 0; k < kRounds; k++) {
        const int e = (int)threadIdx.x + k * kThreads;
        loaded[k] = e < TN * 256 ? load(row(e), col(e)) : (T)0;
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < kRounds; k++) {
        const int e = (int)threadIdx.x + k * kThreads;
        if (e >= TN * 256) break;
        T sum = red[0][e];
#pragma unroll
        for (int w = 1; w < kWaves; w++) sum = sum + red[w][e];
        store(row(e), col(e), sum, loaded[k]);
      }
    }
  } else {
    T loaded[TM][TN][4];
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) loaded[a][b][v] = load(OpA::row(a, Unit<T>::row(q, v), m0, g.M), OpB::row(b, i, n0, g.N));
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) store(OpA::row(a, Unit<T>::row(q, v), m0, g.M), OpB::row(b, i, n0, g.N), acc[a][b][v], loaded[a][b][v]);
  }
}

}  // namespace gemm_direct
