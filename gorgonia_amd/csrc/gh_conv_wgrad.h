// A workgroup of the 3x3 filter gradient with operands straight from memory (k_conv_wgrad.hip has the reasons and the
// figures; k_conv_gradients.hip runs it beside an image gradient).
#pragma once
#include <type_traits>

#include "gh_internal.h"

namespace conv_wgrad {

constexpr int kWaves = 4, kThreads = kWaves * 64;

template <class T> struct Mfma;
template <> struct Mfma<float> {
  typedef float acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc run(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int q, int v) { return 4 * q + v; }   // result row of register v in lanes q
};
template <> struct Mfma<double> {
  typedef double acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc run(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int q, int v) { return 4 * v + q; }
};

template <class T>
struct Wg {
  const T* x;
  const T* dy;
  T* out;                       // [slices][F][C * 9]
  int x_total, dy_total;        // elements
  int B, C, H, W, F, oh, ow, padH, padW;
  int nch;                      // chunks of a row
  int items, per;               // chunks in all, and per wavefront
};

// Waits for this wavefront's loads.  The compiler counts the loads in flight where paths meet by the worst of
// them, so a path that leaves some in flight makes the others wait for the next chunk's as well.
__device__ __forceinline__ void loads_done() { __builtin_amdgcn_s_waitcnt(0x0F70); }   // vmcnt(0), the other counters free

// N consecutive elements from p + off, moved into [0, total) where they stick out: branch-free, so that a chunk's
// loads stay in flight behind the chunk in front.  fix_n puts the elements right.
template <int N, class T>
__device__ __forceinline__ void load_n(const T* __restrict__ p, int off, int total, T* v) {
  typedef T V2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
  typedef T V4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  const unsigned at = (unsigned)min(max(off, 0), total - N);
  if constexpr (N >= 4 && sizeof(T) == 4) {
    const V4 a = *(const V4*)(p + at);
#pragma unroll
    for (int t = 0; t < 4; t++) v[t] = a[t];
    if constexpr (N == 6) {
      const V2 b = *(const V2*)(p + at + 4);
      v[4] = b[0]; v[5] = b[1];
    }
  } else {
#pragma unroll
    for (int t = 0; t < N; t += 2) {
      const V2 a = *(const V2*)(p + at + t);
      v[t] = a[0]; v[t + 1] = a[1];
    }
  }
}
// The elements of a load_n that was moved (the tensor's first and last few), one by one; those outside the tensor
// are whatever is inside (the caller drops them).
template <int N, class T>
__device__ __forceinline__ void fix_n(const T* __restrict__ p, int off, int total, T* v) {
  if (__any(off < 0 || off + N > total)) {
#pragma unroll
    for (int t = 0; t < N; t++) v[t] = p[(unsigned)min(max(off + t, 0), total - 1)];
    loads_done();   // here, not at the values' first use: that is where every chunk would wait
  }
}

// LDS of a workgroup: its wavefronts' sums of 16 filter rows
template <class T, int NT>
constexpr int lds_of() { return kWaves * 16 * 16 * NT * (int)sizeof(T); }

// Workgroup (bx, by, bz): slice, channel tile, filter tile; lds: lds_of bytes.
template <class T, int TM, int P, int NT, bool kPacked>
__device__ __forceinline__ void workgroup(const Wg<T>& g, int bx, int by, int bz, char* lds) {
  static_assert(kPacked || NT == 9, "a channel tile has nine taps");
  typedef typename Mfma<T>::acc Acc;
  constexpr int NB = kPacked ? NT * P : 3 * (P + 2);
  struct Frag { T a[TM][P]; T b[NB]; };
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, q = lane >> 4;
  const int f0 = bz * 16 * TM, c0 = kPacked ? 0 : by * 16;
  const int CKK = g.C * 9, last_image = g.B - 1;

  // element offsets: of a lane's dy rows and of its columns' channels inside an image, in 32 bits
  int f_at[TM];
#pragma unroll
  for (int m = 0; m < TM; m++) f_at[m] = min(f0 + 16 * m + i, g.F - 1) * g.oh * g.ow;
  const int f_image = g.F * g.oh * g.ow, c_image = g.C * g.H * g.W;
  constexpr int NC = kPacked ? NT : 1;
  int c_at[NC], ky[NC], kx[NC];
#pragma unroll
  for (int n = 0; n < NC; n++) {
    const int col = kPacked ? min(n * 16 + i, CKK - 1) : min(c0 + i, g.C - 1) * 9;
    const int c = col / 9, tap = col - c * 9;
    c_at[n] = c * g.H * g.W;
    ky[n] = tap / 3;
    kx[n] = tap - ky[n] * 3;
  }
  // where operand k of a chunk starts: k < TM is a dy row, then one per packed column or per filter row
  constexpr int NX = kPacked ? NT : 3, XN = kPacked ? P : P + 2;
  auto dy_off = [&](int m, int b, int oy, int ch) { return b * f_image + f_at[m] + oy * g.ow + (ch * 4 + q) * P; };
  auto x_off = [&](int n, int b, int oy, int ch) {
    const int iy = oy + (kPacked ? ky[kPacked ? n : 0] : n) - g.padH, ix = (ch * 4 + q) * P + (kPacked ? kx[kPacked ? n : 0] : 0) - g.padW;
    return b * c_image + c_at[kPacked ? n : 0] + min(max(iy, 0), g.H - 1) * g.W + ix;
  };
  // The values as they lie in memory: what is outside the row or the image is dropped in front of the MFMAs
  // (touching a value here would make the wavefront wait for it, and nothing would be in flight under the MFMAs).
  auto load = [&](int b, int oy, int ch, Frag& f) {
#pragma unroll
    for (int m = 0; m < TM; m++) load_n<P>(g.dy, dy_off(m, b, oy, ch), g.dy_total, f.a[m]);
#pragma unroll
    for (int n = 0; n < NX; n++) load_n<XN>(g.x, x_off(n, b, oy, ch), g.x_total, f.b + n * XN);
  };
  Acc acc[TM][NT];
#pragma unroll
  for (int m = 0; m < TM; m++)
#pragma unroll
    for (int n = 0; n < NT; n++) acc[m][n] = Acc{(T)0, (T)0, (T)0, (T)0};
  // A column past the row has to be zero on both sides: zero times an infinity or NaN of x is NaN.  A lane past the row
  // holds zeros, but where a lane's columns reach past the row, x values that taps 1 and 2 of the row's last columns read
  // meet the zero dy of the columns past it under another tap.  The walk notes whether there was one that was not finite
  // (`odd` is NaN then), and if so the wavefront walks its chunks again, choosing x for every step.  (The choice takes 8 to
  // 20 % of the kernel where every chunk makes it, 3 to 25 % where the rows' last ones do, the note 0 to 4 %: 128 -> 256
  // over 8 x 52 x 52 170 us without either, 206, 192 and 171; 308 -> 66 over 26 x 29 x 29 148, 180, 175 and 153.)
  T odd = (T)0;
  auto multiply = [&](auto exact, int b, int oy, int ch, Frag& f) {
    const int ox = (ch * 4 + q) * P;
    if (b == 0 || b == last_image) {   // the only images with loads that stick out of the tensors
#pragma unroll
      for (int m = 0; m < TM; m++) fix_n<P>(g.dy, dy_off(m, b, oy, ch), g.dy_total, f.a[m]);
#pragma unroll
      for (int n = 0; n < NX; n++) fix_n<XN>(g.x, x_off(n, b, oy, ch), g.x_total, f.b + n * XN);
    }
    // a chunk whose every value is inside its row and image has nothing to drop
    const int left = ch * 4 * P - g.padW, right = (ch + 1) * 4 * P + 2 - g.padW;
    if (left < 0 || right > g.W || (ch + 1) * 4 * P > g.ow || oy < g.padH || oy + 3 - g.padH > g.H) {
#pragma unroll
      for (int m = 0; m < TM; m++)
#pragma unroll
        for (int t = 0; t < P; t++) f.a[m][t] = ox + t < g.ow ? f.a[m][t] : (T)0;
      if constexpr (kPacked) {
#pragma unroll
        for (int n = 0; n < NT; n++) {
          const int iy = oy + ky[n] - g.padH, ix = ox + kx[n] - g.padW;
          const bool row = iy >= 0 && iy < g.H;
          const int end = row ? min(g.W - ix, g.ow - ox) : 0;   // the image's and the row's
#pragma unroll
          for (int t = 0; t < P; t++) f.b[n * P + t] = t >= -ix && t < end ? f.b[n * P + t] : (T)0;
        }
      } else {
        const int ix = ox - g.padW;
        const int end = ox < g.ow ? g.W - ix : 0;   // the image's; a lane that is past the row has none
#pragma unroll
        for (int r = 0; r < 3; r++) {
          const bool row = oy + r - g.padH >= 0 && oy + r - g.padH < g.H;
#pragma unroll
          for (int t = 0; t < P + 2; t++) f.b[r * (P + 2) + t] = row && t >= -ix && t < end ? f.b[r * (P + 2) + t] : (T)0;
        }
        if (!decltype(exact)::value && g.ow % P != 0 && (ch + 1) * 4 * P > g.ow) {
#pragma unroll
          for (int k = 0; k < NB; k++) odd = odd + f.b[k] * (T)0;
        }
      }
    }
#pragma unroll
    for (int t = 0; t < P; t++)
#pragma unroll
      for (int n = 0; n < NT; n++) {
        T bv = kPacked ? f.b[n * P + t] : f.b[(n / 3) * (P + 2) + t + n % 3];
        if constexpr (decltype(exact)::value) bv = ox + t < g.ow ? bv : (T)0;
#pragma unroll
        for (int m = 0; m < TM; m++) acc[m][n] = Mfma<T>::run(f.a[m][t], bv, acc[m][n]);
      }
  };

  const int first = (int)min((int64_t)(bx * kWaves + wave) * g.per, (int64_t)g.items);
  const int count = min(g.per, g.items - first);
  auto walk = [&](auto exact) {
    int ch = first % g.nch, row = first / g.nch;   // row of the batch
    int b = row / g.oh, oy = row - b * g.oh;
    auto next = [&]() {
      if (++ch == g.nch) {
        ch = 0;
        if (++oy == g.oh) { oy = 0; b++; }
      }
    };
    Frag cur, ahead;
    load(b, oy, ch, cur);
    loads_done();
    for (int k = 0; k < count; k++) {
      const int b0 = b, oy0 = oy, ch0 = ch;
      if (k + 1 < count) next();
      load(b, oy, ch, ahead);   // (past the end the last chunk again: no branch around a load)
      multiply(exact, b0, oy0, ch0, cur);
      cur = ahead;
    }
  };
  if (count > 0) {
    walk(std::false_type{});
    if (!kPacked && __any(odd != odd)) {
#pragma unroll
      for (int m = 0; m < TM; m++)
#pragma unroll
        for (int n = 0; n < NT; n++) acc[m][n] = Acc{(T)0, (T)0, (T)0, (T)0};
      walk(std::true_type{});
    }
  }

  // the wavefronts' sums, added in wavefront order and stored in the order of dW's rows
  constexpr int COLS = 16 * NT;
  T (* const red)[16 * COLS] = (T (*)[16 * COLS])lds;
  T* const slab = g.out + (int64_t)bx * g.F * CKK;
#pragma unroll
  for (int m = 0; m < TM; m++) {
    if (m) __syncthreads();
    // column of dW: packed tiles hold them in order, a channel tile's tap n of channel i is column 9 i + n
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
      for (int v = 0; v < 4; v++) red[wave][Mfma<T>::row(q, v) * COLS + (kPacked ? n * 16 + i : i * 9 + n)] = acc[m][n][v];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * COLS; e += kThreads) {
      const int f = f0 + 16 * m + e / COLS, col = c0 * 9 + e % COLS;
      if (f < g.F && col < CKK) slab[(int64_t)f * CKK + col] = ((red[0][e] + red[1][e]) + red[2][e]) + red[3][e];
    }
  }
}

}  // namespace conv_wgrad
