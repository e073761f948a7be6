// A workgroup of the 3x3 convolution with operands straight from memory (k_conv_lanes.hip has the reasons and the figures;
// k_conv_gradients.hip runs it beside a filter gradient).
#pragma once
#include "gh_conv_common.h"
#include "gh_internal.h"
#include "gh_schedule.h"

namespace conv_lanes {

constexpr int kOutside = 0x7ffffff0;   // past every buffer: a load from there is zero

template <class T> struct Mac;
template <> struct Mac<float> {
  typedef float acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc run(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int q, int v) { return 4 * q + v; }   // result row of register v in lanes q
  static __device__ __forceinline__ float one(__amdgpu_buffer_rsrc_t r, int at, int s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, at, s, 0));
  }
  static constexpr int kNine = 3;   // loads of nine()
  static __device__ __forceinline__ void nine(__amdgpu_buffer_rsrc_t r, int at, int s, float (&v)[9]) {
    typedef float V __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const V x = __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, at + 16 * k, s, 0));
#pragma unroll
      for (int e = 0; e < 4; e++) v[4 * k + e] = x[e];
    }
    v[8] = one(r, at + 32, s);
  }
  template <int V> static __device__ __forceinline__ void run_of(__amdgpu_buffer_rsrc_t r, int at, int s, float* v) {
    typedef float V4 __attribute__((ext_vector_type(4)));
    static_assert(V == 4, "sixteen bytes");
    const V4 x = __builtin_bit_cast(V4, __builtin_amdgcn_raw_buffer_load_b128(r, at, s, 0));
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = x[e];
  }
};
template <> struct Mac<double> {
  typedef double acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc run(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int q, int v) { return 4 * v + q; }
  static __device__ __forceinline__ double one(__amdgpu_buffer_rsrc_t r, int at, int s) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, at, s, 0));
  }
  static constexpr int kNine = 5;
  static __device__ __forceinline__ void nine(__amdgpu_buffer_rsrc_t r, int at, int s, double (&v)[9]) {
    typedef double V __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const V x = __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, at + 16 * k, s, 0));
      v[2 * k] = x[0]; v[2 * k + 1] = x[1];
    }
    v[8] = one(r, at + 64, s);
  }
  template <int V> static __device__ __forceinline__ void run_of(__amdgpu_buffer_rsrc_t r, int at, int s, double* v) {
    typedef double V2 __attribute__((ext_vector_type(2)));
    static_assert(V == 2, "sixteen bytes");
    const V2 x = __builtin_bit_cast(V2, __builtin_amdgcn_raw_buffer_load_b128(r, at, s, 0));
    v[0] = x[0]; v[1] = x[1];
  }
};

template <class T>
struct Lanes {
  const T* x; const T* w; T* y;
  int C, H, W, F, oh, ow, padH;
  int cols, rows;          // columns and rows of the result that groups cover: ow and oh, or the pooled part of them
  int per_row, groups;     // groups of a row, and in all
  int x_bytes, w_bytes;
  int ftiles, ptiles, ft_major;
};

// The 2x2 / 2 pooling's gradient behind an image gradient whose result is the pooled values' (2 oh x 2 ow values each), read
// through a Rectify, and that one's gradient.  float: z; double: a, what was pooled, z in front of its Rectify, and da, the
// pooling's gradient, where it is not dz.
template <class T> struct Unpool { const T* a; const T* z; T* da; T* dz; };

// LDS of a workgroup: the wavefronts' sums of 16 filter rows, the filters' constants
template <class T, int WV, int TM, int V, int G, bool kSplit>
constexpr int lds_of(bool flip) {
  return (kSplit ? WV * V * G * 256 * (int)sizeof(T) : 0) + (sizeof(T) == 4 && !flip ? 4 * 16 * TM * 4 : 0);
}

// Workgroup `block` of `blocks`; lds: lds_of bytes.
template <class T, int WV, int TM, int V, int G, bool kSplit, bool kFlip, bool kPool, bool kUnpool = false>
__device__ __forceinline__ void workgroup(const Lanes<T>& g, const ConvTail& tail, int block, int blocks, char* lds, const Unpool<T>& u = {}) {
  static_assert(!kUnpool || (kSplit && kFlip && !kPool), "behind an image gradient whose wavefronts share the channels");
  typedef Mac<T> U;
  typedef typename U::acc Acc;
  constexpr int S = (int)sizeof(T), TN = V * G;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, q = lane >> 4;
  // Workgroup ids are dealt round-robin over eight XCDs with an L2 each: an XCD gets a contiguous run of tiles, along
  // whichever operand is the larger so that it is read by one XCD only.
  int ft, pt;
  {
    const int total = blocks, id = block, xcd = id & 7, per = total >> 3, extra = total & 7;
    const int nid = xcd * per + min(xcd, extra) + (id >> 3);
    if (g.ft_major) { ft = nid / g.ptiles; pt = nid - ft * g.ptiles; }
    else { pt = nid / g.ftiles; ft = nid - pt * g.ftiles; }
  }
  const int f0 = ft * 16 * TM, g0 = (kSplit ? pt : pt * WV + wave) * 16 * G;
  const int HW = g.H * g.W;
  // a group's image, result row and first column
  auto place = [&](int grp, int* b, int* oy, int* ox) {
    const unsigned line = (unsigned)(kPool ? grp >> 1 : grp) / (unsigned)g.per_row;
    const int lines = kPool ? g.rows >> 1 : g.rows;
    *ox = min(((kPool ? grp >> 1 : grp) - (int)line * g.per_row) * V, g.cols - V);
    *b = (int)(line / (unsigned)lines);
    *oy = (int)line - *b * lines;
    if (kPool) *oy = 2 * *oy + (grp & 1);
  };
  int a_at[TM], b_at[G][3], l_at[G][3], r_at[G][3];
#pragma unroll
  for (int m = 0; m < TM; m++) {
    const int f = min(f0 + 16 * m + i, g.F - 1);   // (rows past the end are not stored)
    a_at[m] = (kFlip ? q * g.F + f : f * g.C + q) * 9 * S;
  }
#pragma unroll
  for (int n = 0; n < G; n++) {
    const int grp = g0 + 16 * n + i;
    int b, oy, ox;
    place(min(grp, g.groups - 1), &b, &oy, &ox);
#pragma unroll
    for (int r = 0; r < 3; r++) {
      const int iy = oy + r - g.padH;
      const bool in = (unsigned)iy < (unsigned)g.H && grp < g.groups;
      const int at = ((b * g.C + q) * HW + iy * g.W + ox) * S;
      b_at[n][r] = in ? at : kOutside;
      l_at[n][r] = in && ox > 0 ? at - S : kOutside;
      r_at[n][r] = in && ox + V < g.W ? at + V * S : kOutside;
    }
  }
  const int a_step = (kFlip ? 4 * g.F : 4) * 9 * S, b_step = 4 * HW * S;
  const int quads = g.C >> 2;
  struct Frag { T a[TM][9]; T b[G][3][V + 2]; };
  // (a quad past the end: from buffers of no bytes, zeros that nothing is read for)
  auto load = [&](int quad, Frag& f) __attribute__((always_inline)) {
    const bool there = quad < quads;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)g.x, 0, there ? g.x_bytes : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)g.w, 0, there ? g.w_bytes : 0, 0x00020000);
#pragma unroll
    for (int m = 0; m < TM; m++) U::nine(rw, a_at[m], quad * a_step, f.a[m]);
#pragma unroll
    for (int n = 0; n < G; n++)
#pragma unroll
      for (int r = 0; r < 3; r++) {
        f.b[n][r][0] = U::one(rx, l_at[n][r], quad * b_step);
        U::template run_of<V>(rx, b_at[n][r], quad * b_step, f.b[n][r] + 1);
        f.b[n][r][V + 1] = U::one(rx, r_at[n][r], quad * b_step);
      }
  };
  Acc acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; m++)
#pragma unroll
    for (int n = 0; n < TN; n++) acc[m][n] = Acc{(T)0, (T)0, (T)0, (T)0};
  auto multiply = [&](const Frag& f) {
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
      for (int m = 0; m < TM; m++)
#pragma unroll
        for (int n = 0; n < TN; n++) acc[m][n] = U::run(f.a[m][kFlip ? 8 - t : t], f.b[n / V][t / 3][n % V + t % 3], acc[m][n]);
  };
  // The filters' BatchNorm constants go into a table, loaded here and worked out behind the channels: 1 / sqrt for each result
  // was up to half of a pooled layer's time (8 x 16 x 112 x 112 -> 32 with all of its channels in a wavefront 24.3 us, with
  // the table filled here 15.3, behind the channels 14.6).
  const int tf = f0 + (int)threadIdx.x;
  const bool fills = sizeof(T) == 4 && !kFlip && tail.mean && (int)threadIdx.x < 16 * TM && tf < g.F;
  float bn_mean = 0.0f, bn_var = 1.0f, bn_gamma = 1.0f, bn_beta = -0.0f;   // (as conv_tail_table has absent ones)
  if (fills) {
    bn_mean = tail.mean[tf];
    bn_var = tail.var[tf];
    if (tail.gamma) bn_gamma = tail.gamma[tf];
    if (tail.beta) bn_beta = tail.beta[tf];
  }
  constexpr int step = kSplit ? WV : 1;
  const int first = kSplit ? wave : 0;
  if (first < quads) {
    // The loads of a quad are in flight under the MFMAs of the quad before: two sets of operands taken in turn, each load
    // behind a few MFMAs (gh_schedule.h).  us, before / now: 8 x 32 x 52 x 52 -> 64 14.5 / 12.7, 8 x 32 x 104 x 104 -> 64 36.7 / 33.0, its gradient
    // 37.0 / 35.0; the gradient of 8 x 128 x 26 x 26 -> 256 31.5 / 28.2, of 8 x 64 x 26 x 26 -> 128 12.9 / 11.9 and beside the filter's 32.6 / 30.7;
    // float64 4 x 256 x 13 x 13 -> 512 42.2 / 37.8, the gradient of 7 x 64 x 24 x 24 -> 128 13.2 / 11.3.
    Frag even, odd;
    int c = first;
    auto turn = [&](const Frag& now, Frag& next) __attribute__((always_inline)) {
      c += step;
      load(c, next);
      multiply(now);
      gh_spread_loads<TM * U::kNine + 9 * G, 9 * TM * TN>();
      __builtin_amdgcn_sched_barrier(0);
    };
    load(first, even);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // the loop is entered with nothing in flight, so its waits count its own loads only
    const int turns = (quads - first + step - 1) / step;
    for (int two = turns >> 1; two > 0; two--) {   // (one way out: where paths meet the compiler waits for the worst of them)
      turn(even, odd);
      turn(odd, even);
    }
    if (turns & 1) multiply(even);
  }

  float* const tab = (float*)(lds + (kSplit ? WV * TN * 256 * S : 0));
  if (fills) {
    const float a = 1.0f / sqrtf(bn_var + tail.eps);
    const int i = threadIdx.x;
    tab[i] = a;
    tab[16 * TM + i] = -bn_mean * a;
    tab[2 * 16 * TM + i] = bn_gamma;
    tab[3 * 16 * TM + i] = bn_beta;
  }
  T (* const red)[TN * 256] = (T (*)[TN * 256])lds;
  auto store = [&](auto epilogue) __attribute__((always_inline)) {
  if constexpr (!kSplit) {
    // A lane holds V neighbours of its group for four filters of each tile and stores them as they are.
    typedef T Row __attribute__((ext_vector_type(V), aligned(sizeof(T))));
    typedef T Half __attribute__((ext_vector_type(V / 2), aligned(sizeof(T))));
#pragma unroll
    for (int n = 0; n < G; n++) {
      const int grp = g0 + 16 * n + i;
      if (grp >= g.groups) continue;   // (the groups of a pair are both inside or both outside)
      int b, oy, ox;
      place(grp, &b, &oy, &ox);
#pragma unroll
      for (int m = 0; m < TM; m++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int f = f0 + 16 * m + U::row(q, v);
          T own[V];
#pragma unroll
          for (int e = 0; e < V; e++) own[e] = epilogue(16 * m + U::row(q, v), acc[m][n * V + e][v]);
          if constexpr (kPool) {
            T best[V / 2];
            T below[V];
#pragma unroll
            for (int e = 0; e < V; e++) below[e] = __shfl_xor(own[e], 1, 64);
#pragma unroll
            for (int k = 0; k < V / 2; k++) {
              best[k] = (T)-3.402823466e+38f;   // scan order and strict > of the pooling kernel
              if (own[2 * k] > best[k]) best[k] = own[2 * k];
              if (own[2 * k + 1] > best[k]) best[k] = own[2 * k + 1];
              if (below[2 * k] > best[k]) best[k] = below[2 * k];
              if (below[2 * k + 1] > best[k]) best[k] = below[2 * k + 1];
            }
            if (f < g.F && !(i & 1)) {
              Half h;
#pragma unroll
              for (int k = 0; k < V / 2; k++) h[k] = best[k];
              *(Half*)(g.y + (((int64_t)b * g.F + f) * (g.rows >> 1) + (oy >> 1)) * (g.cols >> 1) + (ox >> 1)) = h;
            }
          } else if (f < g.F) {
            Row r;
#pragma unroll
            for (int e = 0; e < V; e++) r[e] = own[e];
            *(Row*)(g.y + (((int64_t)b * g.F + f) * g.oh + oy) * g.ow + ox) = r;
          }
        }
    }
  } else {
  // The sums go through LDS, 16 filter rows at a time, and are added in wavefront order.
  const int tid = (int)threadIdx.x;
  constexpr int nthreads = WV * 64;
  auto value = [&](int e) {
    // (eight in the order of k_conv3x3_patch, whose error a sum in one chain is 1 % above)
    constexpr int kHalves = sizeof(T) == 4 && WV == 8 ? 2 : 1, n = WV / kHalves;
    auto part = [&](int v) { return kHalves == 2 ? red[v][e] + red[v + n][e] : red[v][e]; };
    T sum = part(0);
#pragma unroll
    for (int v = 1; v < n; v++) sum = sum + part(v);
    return sum;
  };
#pragma unroll
  for (int m = 0; m < TM; m++) {
    // the windows that this thread's results go back to, loaded under the meeting of the wavefronts
    typedef T Two __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    constexpr int kWindows = kUnpool ? TN * 256 / nthreads : 1;
    static_assert(!kUnpool || TN * 256 % nthreads == 0, "whole rounds of windows");
    [[maybe_unused]] Two z0[kWindows], z1[kWindows], a0[kWindows], a1[kWindows];
    [[maybe_unused]] int64_t pooled[kWindows];
    [[maybe_unused]] int column[kWindows];
    if constexpr (kUnpool) {
#pragma unroll
      for (int k = 0; k < kWindows; k++) {
        const int e = tid + k * nthreads, r = e / (16 * TN), col = e - r * (16 * TN), f = f0 + 16 * m + r, grp = g0 + col / V;
        pooled[k] = -1;
        if (f >= g.F || grp >= g.groups) continue;
        int b, oy, ox;
        place(grp, &b, &oy, &ox);
        column[k] = ox + col % V;
        pooled[k] = (((int64_t)b * g.F + f) * g.oh + oy) * g.ow + column[k];
        const int64_t at = 4 * pooled[k] - 2 * column[k];   // (row r, column c of ow values: row 2 r, column 2 c of 2 ow)
        z0[k] = *(const Two*)(u.z + at);
        z1[k] = *(const Two*)(u.z + at + 2 * g.ow);
        if constexpr (sizeof(T) == 8) {
          a0[k] = *(const Two*)(u.a + at);
          a1[k] = *(const Two*)(u.a + at + 2 * g.ow);
        }
      }
    }
    if (m) __syncthreads();
#pragma unroll
    for (int n = 0; n < G; n++)
#pragma unroll
      for (int v = 0; v < 4; v++)
#pragma unroll
        for (int e = 0; e < V; e++) red[wave][U::row(q, v) * (16 * TN) + (16 * n + i) * V + e] = acc[m][n * V + e][v];
    __syncthreads();
    if constexpr (kPool) {
      for (int e = tid; e < TN * 64; e += nthreads) {   // windows: V / 2 of them in each pair of groups
        const int r = e / (4 * TN), col = e - r * (4 * TN), pair = col / (V / 2), k = col - pair * (V / 2);
        const int f = f0 + 16 * m + r, grp = g0 + 2 * pair;
        if (f >= g.F || grp >= g.groups) continue;
        const int at = r * (16 * TN) + 2 * pair * V + 2 * k;
        T best = (T)-3.402823466e+38f;   // scan order and strict > of the pooling kernel
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const T v = epilogue(16 * m + r, value(at + (u >> 1) * V + (u & 1)));
          if (v > best) best = v;
        }
        int b, oy, ox;
        place(grp, &b, &oy, &ox);
        g.y[(((int64_t)b * g.F + f) * (g.rows >> 1) + (oy >> 1)) * (g.cols >> 1) + (ox >> 1) + k] = best;
      }
    } else if constexpr (kUnpool) {
      // scan order, strict > and "0 + dy" of the pooling's gradient, and the Rectify's behind it, as their kernels have them
#pragma unroll
      for (int k = 0; k < kWindows; k++) {
        if (pooled[k] < 0) continue;
        const int e = tid + k * nthreads;
        const T own = epilogue(16 * m + e / (16 * TN), value(e));
        const int64_t at = 4 * pooled[k] - 2 * column[k], row = 2 * (int64_t)g.ow;
        g.y[pooled[k]] = own;
        T mask[4], v[4] = {z0[k][0], z0[k][1], z1[k][0], z1[k][1]};
#pragma unroll
        for (int j = 0; j < 4; j++) {
          mask[j] = v[j] >= (T)0 ? (T)1 : (T)0;
          v[j] = sizeof(T) == 8 ? (j < 2 ? a0[k][j & 1] : a1[k][j & 1]) : v[j] * mask[j];
        }
        T best = sizeof(T) == 8 ? (T)-1.7976931348623157e+308 : (T)-3.402823466e+38f;
        int arg = -1;
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (v[j] > best) { best = v[j]; arg = j; }
        const T back = (T)0 + own;
        T d[4];
#pragma unroll
        for (int j = 0; j < 4; j++) d[j] = arg == j ? back : (T)0;
        if constexpr (sizeof(T) == 8) {
          if (u.da != u.dz) {
            *(Two*)(u.da + at) = Two{d[0], d[1]};
            *(Two*)(u.da + at + row) = Two{d[2], d[3]};
          }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) d[j] = d[j] * mask[j];
        *(Two*)(u.dz + at) = Two{d[0], d[1]};
        *(Two*)(u.dz + at + row) = Two{d[2], d[3]};
      }
    } else {
      for (int e = tid; e < TN * 256; e += nthreads) {
        const int r = e / (16 * TN), col = e - r * (16 * TN), f = f0 + 16 * m + r, grp = g0 + col / V;
        if (f >= g.F || grp >= g.groups) continue;
        int b, oy, ox;
        place(grp, &b, &oy, &ox);
        g.y[(((int64_t)b * g.F + f) * g.oh + oy) * g.ow + ox + col % V] = epilogue(16 * m + r, value(e));
      }
    }
  }
  }
  };
  if constexpr (sizeof(T) == 8 || kFlip) {
    store([](int, T v) { return v; });
  } else {
    if (!kSplit) __syncthreads();   // the table
    conv_tail_dispatch(tail, [&](auto BN, auto ACT) { store([&](int r, float v) { return tail_apply_fixed<BN(), ACT()>(tab, 16 * TM, r, v, tail.alpha); }); });
  }
}

}  // namespace conv_lanes

// The image gradient g with the filter gradient that ctx holds, in one launch; -1 where no kernel has both (k_conv_gradients.hip).
int gh_try_launch_gradients(gh_ctx* ctx, const conv_lanes::Lanes<float>& g, int waves, int tm, bool split, int blocks);
int gh_try_launch_gradients(gh_ctx* ctx, const conv_lanes::Lanes<double>& g, int waves, int tm, bool split, int blocks);
