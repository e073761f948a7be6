// Conv2d 3x3 / stride 1 and its image gradient, float32 and float64, on the 16x16x4 MFMA with every operand taken
// from memory straight into the lane that feeds it.
//
// GEMM view: M = filters, N = output pixels of the batch, K = channels x nine taps.  The pixels are taken in groups of
// V neighbours of a row, V tiles to sixteen groups: tile e holds pixel e of each.  A step is a quad of channels: lane
// (i, q) holds channel q of the quad, of filter row i its nine taps - contiguous in memory, three wide loads - and of
// group i the V + 2 values under each of the three filter rows - one wide load and the two neighbours, a third of the
// lane addresses that nine taps of V pixels would take one by one.  A row's last group is moved left to end with the
// row (the pixels it shares with the group before come out the same twice), so no wide load leaves a row.  The byte
// offsets do not change from quad to quad (the quad moves a scalar offset), and a value outside the image has an offset
// that the buffer's range check turns into zero, so the loop holds loads and MFMAs and nothing else: no staging, no
// barrier, no edge arithmetic.  The loads of a quad are issued in front of the MFMAs of the quad before it.  The
// wavefronts of a workgroup split the channels of one tile (kSplit), their sums meeting in LDS in wavefront order, or
// own a tile each.  With a pooled result the groups come in pairs, one above the other.
//
// With kFlip the same walk is the image gradient: rows are image channels, K runs over the filters, and a lane's nine
// weights are those of one (filter, channel) pair in reverse.  No mirrored copy of the filters is made.
//
// It is bound by lane addresses where a tile has 16 filters (each wide load feeds one row of tiles) and at four fifths
// of the MFMA rate at 32.  Measured against the kernels that took these shapes before, us, float32 forward of one
// image: 64 -> 128 at 52 x 52 10.7 (14.0), 128 -> 256 at 26 x 26 9.2 (20.9), 256 -> 512 at 13 x 13 13.6 (32.8), 512 ->
// 1024 24.5 (59.4); of eight, 32 -> 64 at 52 x 52 16.0 (23.2); image gradient of two, 64 -> 128 at 26 x 26 8.0 (22.7).
// float64, 50 images: 32 -> 64 at 14 x 14 16.9 (28.5) and its image gradient 11.8 (72), 64 -> 128 at 7 x 7 15.3 (39.5)
// and 13.2 (81).
#include <algorithm>
#include <cstdlib>

#include "gh_conv_common.h"
#include "gh_internal.h"

namespace {

constexpr int kOutside = 0x7ffffff0;   // past every buffer: a load from there is zero

template <class T> struct Mac;
template <> struct Mac<float> {
  typedef float acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc run(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int q, int v) { return 4 * q + v; }   // result row of register v in lanes q
  static __device__ __forceinline__ float one(__amdgpu_buffer_rsrc_t r, int at, int s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, at, s, 0));
  }
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

template <class T, int WV, int TM, int V, int G, bool kSplit, bool kFlip, bool kPool>
__global__ __launch_bounds__(WV * 64) __attribute__((amdgpu_waves_per_eu(WV == 8 || TM * V * G * sizeof(T) <= 32 ? 2 : 1))) void k_conv3x3_lanes(const Lanes<T> g, const ConvTail tail) {
  typedef Mac<T> U;
  typedef typename U::acc Acc;
  constexpr int S = (int)sizeof(T), TN = V * G;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, q = lane >> 4;
  // Workgroup ids are dealt round-robin over eight XCDs with an L2 each: an XCD gets a contiguous run of tiles, along
  // whichever operand is the larger so that it is read by one XCD only.
  int ft, pt;
  {
    const int total = gridDim.x, id = blockIdx.x, xcd = id & 7, per = total >> 3, extra = total & 7;
    const int nid = xcd * per + min(xcd, extra) + (id >> 3);
    if (g.ft_major) { ft = nid / g.ptiles; pt = nid - ft * g.ptiles; }
    else { pt = nid / g.ftiles; ft = nid - pt * g.ftiles; }
  }
  const int f0 = ft * 16 * TM, g0 = (kSplit ? pt : pt * WV + wave) * 16 * G;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)g.x, 0, g.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)g.w, 0, g.w_bytes, 0x00020000);
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
  struct Frag { T a[TM][9]; T b[G][3][V + 2]; };
  auto load = [&](int quad, Frag& f) {
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
  const int quads = g.C >> 2;
  constexpr int step = kSplit ? WV : 1;
  const int first = kSplit ? wave : 0;
  if (first < quads) {
    Frag cur, ahead;
    load(first, cur);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // the loop is entered with nothing in flight, so its waits count its own loads only
    for (int c = first; c < quads; c += step) {
      load(c + step < quads ? c + step : c, ahead);   // (past the end the last quad again: no branch around the loads)
      multiply(cur);
      cur = ahead;
    }
  }

  __shared__ float tab[sizeof(T) == 4 ? 4 * 16 * TM : 1];
  if (fills) {
    const float a = 1.0f / sqrtf(bn_var + tail.eps);
    const int i = threadIdx.x;
    tab[i] = a;
    tab[16 * TM + i] = -bn_mean * a;
    tab[2 * 16 * TM + i] = bn_gamma;
    tab[3 * 16 * TM + i] = bn_beta;
  }
  __shared__ __attribute__((aligned(16))) T red[kSplit ? WV : 1][kSplit ? TN * 256 : 1];
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
    T sum = red[0][e];
#pragma unroll
    for (int v = 1; v < WV; v++) sum = sum + red[v][e];
    return sum;
  };
#pragma unroll
  for (int m = 0; m < TM; m++) {
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

template <class T, int WV, int TM, int V, int G, bool kSplit>
int launch(gh_ctx* ctx, Lanes<T> g, const ConvTail& tail, bool flip, bool pool) {
  constexpr int per = 16 * G * (kSplit ? 1 : WV);
  const int lines = g.groups;   // image rows (row pairs) in all, until here
  g.per_row = (g.cols + V - 1) / V;
  g.groups = lines * g.per_row * (pool ? 2 : 1);
  g.ftiles = (g.F + 16 * TM - 1) / (16 * TM);
  g.ptiles = (g.groups + per - 1) / per;
  g.ft_major = g.w_bytes > g.x_bytes;
  const dim3 grid((unsigned)(g.ftiles * g.ptiles));
  if constexpr (sizeof(T) == 4) {
    if (pool) {
      hipLaunchKernelGGL((k_conv3x3_lanes<T, WV, TM, V, G, kSplit, false, true>), grid, dim3(WV * 64), 0, ctx->stream, g, tail);
      return gh_check_hip(ctx, hipGetLastError(), "conv3x3 launch");
    }
  }
  if (flip) hipLaunchKernelGGL((k_conv3x3_lanes<T, WV, TM, V, G, kSplit, true, false>), grid, dim3(WV * 64), 0, ctx->stream, g, tail);
  else hipLaunchKernelGGL((k_conv3x3_lanes<T, WV, TM, V, G, kSplit, false, false>), grid, dim3(WV * 64), 0, ctx->stream, g, tail);
  return gh_check_hip(ctx, hipGetLastError(), "conv3x3 launch");
}

// The geometry of a forward command or (flip) of the convolution that an image-gradient command is; false where the
// kernel does not take it: 3x3, stride 1, whole quads of channels, byte offsets in 31 bits.
template <class T>
bool fill(const gh_cmd& c, bool flip, bool pool, Lanes<T>* g) {
  if (c.dim[5] != 3 || c.dim[6] != 3) return false;
  for (int i : {9, 10, 11, 12}) if (c.dim[i] != 1) return false;
  const int64_t B = c.dim[0], padH = c.dim[7], padW = c.dim[8];
  int64_t C = c.dim[1], H = c.dim[2], W = c.dim[3], F = c.dim[4];
  if (B <= 0 || C <= 0 || F <= 0 || H <= 0 || W <= 0 || padH < 0 || padW < 0 || padH > 2 || padW != 1 || W < 4) return false;
  if (H > (1 << 20) || W > (1 << 20) || C > (1 << 20) || F > (1 << 20) || B > (1 << 24)) return false;
  int64_t oh = H + 2 * padH - 2, ow = W + 2 * padW - 2;
  if (oh <= 0 || ow <= 0) return false;
  g->padH = (int)(flip ? 2 - padH : padH);
  if (flip) { std::swap(C, F); std::swap(H, oh); std::swap(W, ow); }
  const int64_t most = (0x7fff0000ll) / (int64_t)sizeof(T);   // below kOutside, the quad steps included
  if (C % 4 != 0 || B * C * H > most / W || B * F * oh > most / ow || C * F > most / 9) return false;
  g->x = (const T*)(uintptr_t)c.ptr[0]; g->w = (const T*)(uintptr_t)c.ptr[1]; g->y = (T*)(uintptr_t)c.ptr[2];
  g->C = (int)C; g->H = (int)H; g->W = (int)W; g->F = (int)F; g->oh = (int)oh; g->ow = (int)ow;
  g->rows = pool ? g->oh / 2 * 2 : g->oh;
  g->cols = pool ? g->ow / 2 * 2 : g->ow;
  g->groups = (int)B * (pool ? g->rows / 2 : g->rows);   // lines; the launch makes groups of them
  g->x_bytes = (int)(B * C * H * W * (int64_t)sizeof(T));
  g->w_bytes = (int)(C * F * 9 * (int64_t)sizeof(T));
  return g->groups > 0;
}

}  // namespace

// The forms: filter tiles x groups of V pixels of a workgroup's (or wavefront's) tile, its wavefronts, whether they
// split the channels, and what a round of such tiles over the compute units takes in us: per tile, and per quad of
// channels.  Fitted to 50 shapes of 1 to 256 images of 7 x 7 to 104 x 104, 16 to 512 channels, forward and gradient;
// the estimates are mostly within 15 % of the times.
struct Form { int tm, v, waves, groups; bool split; double per_tile, per_quad; };
static const Form kForms32[] = {{1, 4, 8, 1, true, 1.9, 0.160}, {2, 4, 8, 1, true, 3.2, 0.263}, {2, 4, 4, 1, true, 2.4, 0.24}, {2, 4, 4, 1, false, 2.6, 1.05}, {1, 4, 4, 1, false, 1.8, 0.52}};
// float64, where a forward pass's fragments of a quad come from rows C filters apart: its small forms take longer than a
// gradient's.  The last is one filter tile by two groups, between the first two in loads for a product, with their sums in
// their order: us, without it / with, 50 x 32 x 14 x 14 -> 64 16.4 / 14.3; 20 x 64 x 7 x 7 -> 128 10.8 / 9.0; 96 x 64 x 7 x 7 ->
// 128 29.5 / 22.2; 8 x 64 x 26 x 26 -> 128 29.1 / 22.0 (36 TFLOP/s); 64 x 32 x 14 x 14 -> 64, a little past
// three rounds of it, 16.6 in the second and 18.8 in it.  A gradient gains nothing from it.
static const Form kForward64[] = {{1, 2, 4, 1, true, 0.7, 0.20}, {2, 2, 4, 2, true, 3.4, 0.47}, {2, 2, 4, 2, false, 4.0, 2.2}, {1, 2, 4, 2, true, 1.15, 0.32}};
static const Form kGradient64[] = {{1, 2, 4, 1, true, 0.8, 0.17}, {2, 2, 4, 2, true, 3.4, 0.47}, {2, 2, 4, 2, false, 4.0, 2.2}};

// The quickest of the forms from..to - 1 and its time: a function of the plain command (a pooled one takes the same form
// and so sums in the same order).
static int quickest(const gh_cmd& c, bool flip, bool f64, int cus, int from, int to, double* us) {
  const int64_t B = c.dim[0], oh = c.dim[2] + 2 * c.dim[7] - 2, ow = c.dim[3];
  const int64_t K = flip ? c.dim[4] : c.dim[1], F = flip ? c.dim[1] : c.dim[4], lines = B * (flip ? c.dim[2] : oh);
  int best = -1;
  for (int i = from; i < to; i++) {
    const Form& f = (!f64 ? kForms32 : flip ? kGradient64 : kForward64)[i];
    // an image gradient gains nothing from the form that halves the wavefronts (8 x 32 x 52 x 52 <- 64: 14.5 us, 14.0 with
    // eight), and would add twice as many terms in a row
    if (!f64 && flip && f.split && f.waves == 4) continue;
    const int64_t per = 16 * f.groups * (f.split ? 1 : f.waves);
    const int64_t tiles = (F + 16 * f.tm - 1) / (16 * f.tm) * ((lines * ((ow + f.v - 1) / f.v) + per - 1) / per);
    // one tile of four wavefronts to a compute unit waits for its loads
    const bool lone = !f64 && f.waves == 4 && tiles <= cus;
    const double per_quad = !lone ? f.per_quad : f.split ? 0.33 : 1.27 * f.per_quad;
    const double est = 3.2 + (double)((tiles + cus - 1) / cus) * (f.per_tile + per_quad * (double)(K / 4));
    if (best < 0 || est < *us) { best = i; *us = est; }
  }
  return best;
}

// Which form takes a convolution (flip: an image gradient) that `other_us` is what the other kernels would take for, -1
// where they keep it; other_us 0: any shape that a form can take.  It has to be a sixth quicker by the estimates, which
// are that good.
//
// float32 where that is not so: a wavefront with a tile of its own and all channels, for few channels and many pixels, where
// the split forms have one or two quads to a wavefront and the wide-image kernel stages as much as it multiplies.  Only in place
// of a kernel whose sums run over all channels too (`whole`), since its own are longer than those of one that splits them: the
// gradient of 4 x 128 x 60 x 60 -> 64 would be off by 4.3e-7 of its norm instead of 1.6e-7, that of 13 x 96 x 45 x 45 -> 48, which
// runs as a split form over dy, by 2.9e-7 instead of 8.1e-8, that of 234 x 8 x 15 x 15 -> 32 by 2.5e-7, on the small-image
// kernel 2.0e-7.  us, before / now: 8 x 16 x 104 x 104 -> 32 22.9 / 15.9, pooled 17.9 / 13.6, its gradient 24.2 / 13.6; 8 x 16 x 104 x 104 -> 16
// 15.8 / 10.0 and its gradient 17.8 / 8.7; 8 x 32 x 104 x 104 -> 64 46.7 / 39.7 (80 TFLOP/s); 8 x 16 x 208 x 208 -> 32's
// gradient 45.8 / 36.1; 1 x 16 x 208 x 208 -> 32 pooled 11.0 / 8.7.
int gh_conv_lanes_form(const gh_cmd& c, bool flip, int cus, double other_us, bool whole) {
  if (getenv("GORGONIA_HIP_CONV_NO_LANES")) return -1;   // tuning switch: the other kernels only
  const bool f64 = gh_dtype_of(c.flags) == GH_F64;
  Lanes<double> g;   // (the narrower of the two in what its offsets reach)
  if (!fill(c, flip, false, &g) || g.F < 8 || g.C < 8 || g.oh < 2) return -1;
  double us;
  const int split = quickest(c, flip, f64, cus, 0, f64 && !flip ? 4 : 3, &us);
  if (other_us <= 0 || us < other_us / 1.17) return split;
  if (f64 || !whole) return -1;
  const int form = quickest(c, flip, false, cus, 3, 5, &us);
  return us < other_us / 1.1 ? form : -1;
}

int gh_launch_conv_lanes(gh_ctx* ctx, const gh_cmd& c, bool flip, int form) {
  const bool pool = !flip && (c.flags & GH_FLAG_CONV_POOL2);
  if (gh_dtype_of(c.flags) == GH_F64) {
    Lanes<double> g;
    if (!fill(c, flip, false, &g)) return gh_fail(ctx, GH_ESTATE, "conv3x3: not a shape of this kernel");
    const ConvTail t{};
    switch (form) {
      case 0: return launch<double, 4, 1, 2, 1, true>(ctx, g, t, flip, false);
      case 1: return launch<double, 4, 2, 2, 2, true>(ctx, g, t, flip, false);
      case 3: return launch<double, 4, 1, 2, 2, true>(ctx, g, t, flip, false);   // (forward)
      default: return launch<double, 4, 2, 2, 2, false>(ctx, g, t, flip, false);
    }
  }
  Lanes<float> g;
  if (!fill(c, flip, pool, &g)) return gh_fail(ctx, GH_ESTATE, "conv3x3: not a shape of this kernel");
  const ConvTail t = flip ? ConvTail{} : conv_tail(c);
  switch (form) {
    case 0: return launch<float, 8, 1, 4, 1, true>(ctx, g, t, flip, pool);
    case 1: return launch<float, 8, 2, 4, 1, true>(ctx, g, t, flip, pool);
    case 3: return launch<float, 4, 2, 4, 1, false>(ctx, g, t, flip, pool);
    case 4: return launch<float, 4, 1, 4, 1, false>(ctx, g, t, flip, pool);
    default: return launch<float, 4, 2, 4, 1, true>(ctx, g, t, flip, pool);
  }
}
