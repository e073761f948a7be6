// Matrix products with operands taken from memory straight into the lanes of the 16x16x4 MFMA.
//
// A workgroup owns a tile of 16 TM x 16 TN results and its four wavefronts each sum a quarter of K over the whole
// tile: chunk w, w + 4, ... of KC = 4 KQ consecutive k.  Lane (i, q) holds, of every row of A and column of B it
// feeds, the KQ values k0 + KQ q ... - one 16-byte load where k runs along memory - and MFMA step t takes element
// t of both, so it does not matter that a step's four k are KQ apart.  Where k does not run along memory, a lane
// takes V = KQ neighbouring rows (columns) per k instead, also 16 bytes, and its V tiles are interleaved: tile e
// of a group holds every V-th row.  Nothing is staged and no barrier stands in the loop; the loads of a chunk are
// issued before the MFMAs of the chunk in front of it.  The wavefronts' sums meet in LDS in wavefront order.
//
// Against the LDS-tiled kernels: no tile staging to hide with a second workgroup, so one large tile per compute
// unit runs at the rate of many, any tile height in steps of 16 is to be had, and a product is cut so that its
// tiles come out just under a multiple of the compute units (gemm_direct_tile).
#include <algorithm>

#include "gh_conv_common.h"
#include "gh_internal.h"

namespace {

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

// One operand of a tile: TT tiles of 16 rows (of A; of B, columns), rows r0 and up, rmax of them in all.
// KC: k runs along memory.  Rows past the end are the last row again; their results are not stored.
template <class T, int TT, bool kAlongK>
struct Operand {
  static constexpr int KQ = Unit<T>::KQ, V = KQ;
  static constexpr int G = kAlongK ? 0 : TT / V, S = kAlongK ? TT : TT % V;   // groups of V tiles, single tiles
  typedef typename Unit<T>::vec vec;
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

template <class T, int kWaves, int TM, int TN, bool kSplitK, bool kTA, bool kTB>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(kWaves == 8 || TM * TN * sizeof(T) <= 160 ? 2 : 1))) void k_gemm_direct(const Gemm<T> g) {
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
    const int gx = gridDim.x, gy = gridDim.y, total = gx * gy, id = blockIdx.y * gx + blockIdx.x;
    const int xcd = id & 7, per = total >> 3, extra = total & 7;
    const int nid = xcd * per + min(xcd, extra) + (id >> 3);
    const int group = 8 * gx, first = nid / group * 8, rows = min(gy - first, 8), in = nid % group;
    tm = first + in % rows;
    tn = in / rows;
  }
  const int m0 = kSplitK ? tm * 16 * TM : (tm * kWaves + wave) * 16 * TM, n0 = tn * 16 * TN;
  if (!kSplitK && m0 >= g.M) return;   // (no barrier in this form)
  T* const C = g.C + blockIdx.z * g.sC;
  OpA oa;
  OpB ob;
  const T* const A = oa.init(g.A + blockIdx.z * g.sA, m0, g.M, g.lda, i, q);
  const T* const B = ob.init(g.B + blockIdx.z * g.sB, n0, g.N, g.ldb, i, q);

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
  Frag cur, ahead;
  const int first = kSplitK ? 2 * wave : 0;
  if (first < full) {
    oa.load(A, first * KC, cur.a);
    ob.load(B, first * KC, cur.b);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // the loop is entered with nothing in flight, so its waits count its own loads only
    for (int c = first; c < full;) {
      const int after = c + (kSplitK && (c & 1) ? 2 * kWaves - 1 : 1);
      const int next = min(after, full - 1);   // (past the end: no branch around the loads)
      oa.load(A, next * KC, ahead.a);
      ob.load(B, next * KC, ahead.b);
      multiply(cur);
      cur = ahead;
      c = after;
    }
  }
  if (g.K % KC && (!kSplitK || wave == full % (2 * kWaves) / 2)) {
    oa.load_tail(A, full * KC, g.K, q, cur.a);
    ob.load_tail(B, full * KC, g.K, q, cur.b);
    multiply(cur);
  }

  auto store = [&](int r, int c, T sum) {
    if (r >= g.M || c >= g.N) return;
    if constexpr (sizeof(T) == 4) {
      if (g.bias) sum = sum + g.bias[c];
      sum = act_apply(sum, g.act, g.alpha);
    }
    C[(int64_t)r * g.ldc + c] = sum;
  };
  if constexpr (kSplitK) {
    __shared__ T red[kWaves][TN * 256];
#pragma unroll
    for (int a = 0; a < TM; a++) {
      if (a) __syncthreads();
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) red[wave][b * 256 + v * 64 + lane] = acc[a][b][v];
      __syncthreads();
#pragma unroll
      for (int e = threadIdx.x; e < TN * 256; e += kThreads) {
        T sum = red[0][e];
#pragma unroll
        for (int w = 1; w < kWaves; w++) sum = sum + red[w][e];
        const int l = e & 63, v = (e >> 6) & 3, b = e >> 8;
        store(OpA::row(a, Unit<T>::row(l >> 4, v), m0, g.M), OpB::row(b, l & 15, n0, g.N), sum);
      }
    }
  } else {
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) store(OpA::row(a, Unit<T>::row(q, v), m0, g.M), OpB::row(b, i, n0, g.N), acc[a][b][v]);
  }
}

template <class T, int W, int TM, int TN, bool kSplitK = true>
void launch(gh_ctx* ctx, const Gemm<T>& g, int batch, bool ta, bool tb) {
  constexpr int rows = 16 * TM * (kSplitK ? 1 : W);
  const dim3 grid((unsigned)((g.N + 16 * TN - 1) / (16 * TN)), (unsigned)((g.M + rows - 1) / rows), (unsigned)batch);
  if (ta && tb) hipLaunchKernelGGL((k_gemm_direct<T, W, TM, TN, kSplitK, true, true>), grid, dim3(W * 64), 0, ctx->stream, g);
  else if (ta) hipLaunchKernelGGL((k_gemm_direct<T, W, TM, TN, kSplitK, true, false>), grid, dim3(W * 64), 0, ctx->stream, g);
  else if (tb) hipLaunchKernelGGL((k_gemm_direct<T, W, TM, TN, kSplitK, false, true>), grid, dim3(W * 64), 0, ctx->stream, g);
  else hipLaunchKernelGGL((k_gemm_direct<T, W, TM, TN, kSplitK, false, false>), grid, dim3(W * 64), 0, ctx->stream, g);
}

}  // namespace

// The forms: rows x columns of a workgroup's tile in sixteens, whether its wavefronts split K, and what a multiple of
// the compute units' worth of such tiles takes: us per 16 x 16 results and 1000 of K, and per 16 x 16 results
// (measured over square and ragged products of 100 to 4096; the estimates are within 10 % of the times).
struct Form { int tm, tn; bool split; double per_k, per_tile; };
static const Form kForms32[] = {{2, 4, true, 1.40, 0.12}, {3, 4, true, 1.28, 0.12}, {4, 4, true, 1.25, 0.12},
                                {5, 4, true, 1.22, 0.12}, {4, 4, false, 1.45, 0.06}, {8, 4, false, 1.25, 0.06}};
static const Form kForms64[] = {{2, 2, true, 2.28, 0.17}, {2, 4, true, 2.00, 0.17}, {3, 4, true, 1.92, 0.17}, {4, 4, true, 1.94, 0.17},
                                {5, 4, true, 1.90, 0.17}};

// Whether k_gemm_direct takes a product - at least one whole group of rows and columns, a tile's offsets in 32 bits -
// and the quickest form for it: its number, its time in *us and its rounds of tiles over the compute units.
int gh_gemm_direct_form(const gh_cmd& c, int cus, double* us, int* rounds) {
  const bool f64 = gh_dtype_of(c.flags) == GH_F64;
  const int64_t M = c.dim[0], N = c.dim[1], K = c.dim[2], batch = c.dim[6] <= 0 ? 1 : c.dim[6];
  const int v = f64 ? 2 : 4;
  if (M < v || N < v || batch > 65535 || std::max(c.dim[3], c.dim[4]) * (f64 ? 8 : 4) >= ((int64_t)1 << 31) / 160) return -1;
  const bool along_k = !(c.flags & GH_FLAG_TRANS_A) && (c.flags & GH_FLAG_TRANS_B);   // both operands: half lines per load
  const Form* forms = f64 ? kForms64 : kForms32;
  const int n = f64 ? 5 : 6;
  int best = -1;
  for (int i = 0; i < n; i++) {
    const Form& f = forms[i];
    if (!f64 && f.split && K <= 128) continue;   // four pairs of chunks: half of eight wavefronts would have none
    const int64_t tiles = (M + 16 * f.tm - 1) / (16 * f.tm) * ((N + 16 * f.tn - 1) / (16 * f.tn)) * batch;
    const double per_k = f.per_k * (f64 && along_k && f.tm == 2 ? (f.tn == 2 ? 1.5 : 1.3) : 1.0);
    const double est = 4.0 + (double)((tiles + cus - 1) / cus) * f.tm * f.tn * ((double)K * 1e-3 * per_k + f.per_tile);
    if (best >= 0 && est >= *us) continue;
    *us = est;
    best = i;
    if (rounds) *rounds = (int)((tiles + cus - 1) / cus);
  }
  return best;
}

// K slices of a form: the wavefronts' shares.  One tile per compute unit has eight wavefronts (float32): with four,
// a chunk's MFMAs are over before the next chunk's loads are.
static int waves_of(const gh_cmd& c, const Form& f, int cus) {
  if (!f.split) return 1;
  const int64_t tiles = (c.dim[0] + 16 * f.tm - 1) / (16 * f.tm) * ((c.dim[1] + 16 * f.tn - 1) / (16 * f.tn)) * std::max<int64_t>(1, c.dim[6]);
  return gh_dtype_of(c.flags) != GH_F64 && tiles <= cus ? 8 : 4;
}
int gh_gemm_direct_slices(const gh_cmd& c, int form, int cus) {
  return waves_of(c, (gh_dtype_of(c.flags) == GH_F64 ? kForms64 : kForms32)[form], cus);
}

template <class T>
static Gemm<T> gemm_of(const gh_cmd& c, int* batch) {
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

int gh_launch_gemm_direct(gh_ctx* ctx, const gh_cmd& c, int form) {
  const bool ta = c.flags & GH_FLAG_TRANS_A, tb = c.flags & GH_FLAG_TRANS_B;
  int batch;
  if (gh_dtype_of(c.flags) == GH_F64) {
    const Gemm<double> g = gemm_of<double>(c, &batch);
    switch (form) {
      case 0: launch<double, 4, 2, 2>(ctx, g, batch, ta, tb); break;
      case 1: launch<double, 4, 2, 4>(ctx, g, batch, ta, tb); break;
      case 2: launch<double, 4, 3, 4>(ctx, g, batch, ta, tb); break;
      case 3: launch<double, 4, 4, 4>(ctx, g, batch, ta, tb); break;
      default: launch<double, 4, 5, 4>(ctx, g, batch, ta, tb); break;
    }
  } else {
    const Gemm<float> g = gemm_of<float>(c, &batch);
    const bool eight = waves_of(c, kForms32[form], ctx->cu_count) == 8;
    switch (form) {
      case 0: eight ? launch<float, 8, 2, 4>(ctx, g, batch, ta, tb) : launch<float, 4, 2, 4>(ctx, g, batch, ta, tb); break;
      case 1: eight ? launch<float, 8, 3, 4>(ctx, g, batch, ta, tb) : launch<float, 4, 3, 4>(ctx, g, batch, ta, tb); break;
      case 2: eight ? launch<float, 8, 4, 4>(ctx, g, batch, ta, tb) : launch<float, 4, 4, 4>(ctx, g, batch, ta, tb); break;
      case 3: eight ? launch<float, 8, 5, 4>(ctx, g, batch, ta, tb) : launch<float, 4, 5, 4>(ctx, g, batch, ta, tb); break;
      case 4: launch<float, 4, 1, 4, false>(ctx, g, batch, ta, tb); break;
      default: launch<float, 4, 2, 4, false>(ctx, g, batch, ta, tb); break;
    }
  }
  return gh_check_hip(ctx, hipGetLastError(), "gemm launch");
}
