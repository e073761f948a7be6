// A workgroup of the 3x3 filter gradient over small images (k_conv_wgrad_small.hip has the reasons and the figures;
// k_conv_gradients.hip runs it beside an image gradient).
#pragma once
#include "gh_internal.h"

namespace conv_wgrad_small {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));   // a row of dy starts on any float

// n / d with magic = magic_of(d), exact while n * d < 2^32 (magic 0 stands for d = 1)
__device__ __forceinline__ int mdiv(int n, unsigned magic) {
  const unsigned q = __umulhi((unsigned)n, magic);
  return (int)(q | ((unsigned)n & (0u - (unsigned)(magic == 0))));
}

struct WgGeom {
  int B, C, H, W, F, pad, oh, ow;
  int npx;          // oh * ow
  int nb;           // images staged together
  int K;            // nb * npx
  int KW;           // K rounded up to a multiple of 4
  int DP;           // pitch of a dyL row, = 4 mod 64, >= KW
  int PW, PH;       // padded plane: (W + 2 pad) x (H + 2 pad)
  int XP;           // plane pitch in LDS (= 4 mod 32, >= PH rows)
  int HW;
  int CKK;          // C * 9
  int ngroups;      // ceil(B / nb)
  int gps;          // image groups per split
  unsigned mNPX, mOW, mHW, mW, mQIMG, mQX;
};

constexpr int kCT = 16;          // channels per workgroup
constexpr int kBM = 64;          // filters per workgroup
constexpr int kThreads = 512;
constexpr int kDy = 8, kX = 2;   // 128-bit loads a thread has in flight while staging: a group of up to 256 output pixels

// The row pitch of a staged plane: the widest padded image (16 + 2), or that of images of up to eight columns, whose planes
// take half the LDS.
constexpr int kWide = 18, kNarrow = 10;

// Workgroup (split, channel tile, filter tile); lds: the plan's bytes.
template <int kRowPitch>
__device__ __forceinline__ void workgroup(const float* __restrict__ x, const float* __restrict__ dy, float* __restrict__ out, const WgGeom& g, int64_t slab, int split,
                                          int ctile, int ftile, float* lds) {
  float* const dyL = lds;                                  // [64][DP]
  float* const xL = dyL + kBM * g.DP;                      // [nb][16][XP]
  int* const ptab = reinterpret_cast<int*>(xL + g.nb * kCT * g.XP);   // [KW]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mt = wave & 3, khalf = wave >> 2;   // tile row, half of the k steps
  const int li = lane & 15, lk = lane >> 4;
  const int c0 = ctile * kCT, f0 = ftile * kBM;

  // position of every k in the staged planes: image plane block + row + column
  for (int p = tid; p < g.KW; p += kThreads) {
    int pos = 0;
    if (p < g.K) {
      const int img = mdiv(p, g.mNPX), r = p - img * g.npx;
      const int row = mdiv(r, g.mOW), col = r - row * g.ow;
      pos = img * (kCT * g.XP) + row * kRowPitch + col;
    }
    ptab[p] = pos;
  }
  // B column of (tile t, lane li) is (tap t, channel li): the lane's plane, the tile's tap offset
  const int xlane = li * g.XP;
  f32x4 acc[9];
#pragma unroll
  for (int t = 0; t < 9; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // 128-bit pieces of a group's dy (64 npx an image) and x (16 H W), which are contiguous per image
  const int per_img = kBM * g.npx, q_img = per_img >> 2, nq = g.nb * q_img;
  const int nfv = min(kBM, g.F - f0) * g.npx;     // elements of an image's dy block that exist
  const int qx = kCT / 4 * g.HW, nx = g.nb * qx;
  f32x4 dv[kDy], xv[kX];
  // (Pieces' places are worked out where they are used: kept from one use to the next they would not fit the registers.)
  auto fetch = [&](int b0, int it) {
    int mine = tid;
    asm volatile("" : "+v"(mine));
#pragma unroll
    for (int u = 0; u < kDy; u++) {
      const int q = (it * kDy + u) * kThreads + mine;
      dv[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (q < nq) {
        const int img = mdiv(q, g.mQIMG), r = 4 * (q - img * q_img);
        if (b0 + img < g.B) {
          const float* const src = dy + ((int64_t)(b0 + img) * g.F + f0) * g.npx + r;
          if (r + 3 < nfv) dv[u] = *reinterpret_cast<const f32x4_a4*>(src);
          else
            for (int j = 0; j < 4; j++) if (r + j < nfv) dv[u][j] = src[j];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kX; u++) {
      const int q = (it * kX + u) * kThreads + mine;
      xv[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (q < nx) {
        const int img = mdiv(q, g.mQX), r = 4 * (q - img * qx);
        if (b0 + img < g.B) xv[u] = *reinterpret_cast<const f32x4_a4*>(x + ((int64_t)(b0 + img) * g.C + c0) * g.HW + r);
      }
    }
  };
  auto put = [&](int it) {
    int mine = tid;
    asm volatile("" : "+v"(mine));
#pragma unroll
    for (int u = 0; u < kDy; u++) {
      const int q = (it * kDy + u) * kThreads + mine;
      if (q >= nq) continue;
      const int img = mdiv(q, g.mQIMG), r = 4 * (q - img * q_img);
      const int f = mdiv(r, g.mNPX), pix = r - f * g.npx;
      const int dst = f * g.DP + img * g.npx + pix, left = g.npx - pix;
#pragma unroll
      for (int j = 0; j < 4; j++)   // past the row's last pixel: first pixel of the next row
        dyL[dst + j + (j >= left ? g.DP - g.npx : 0)] = dv[u][j];
    }
#pragma unroll
    for (int u = 0; u < kX; u++) {
      const int q = (it * kX + u) * kThreads + mine;
      if (q >= nx) continue;
      const int img = mdiv(q, g.mQX), r = 4 * (q - img * qx);
      const int c = mdiv(r, g.mHW), pix = r - c * g.HW;
      int row = mdiv(pix, g.mW), col = pix - row * g.W;
      int at = (img * kCT + c) * g.XP + (row + g.pad) * kRowPitch + col + g.pad;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        xL[at] = xv[u][j];
        at++;
        if (++col == g.W) {   // the next row, or the next channel's first
          col = 0;
          at += kRowPitch - g.W;
          if (++row == g.H) { row = 0; at += g.XP - g.H * kRowPitch; }
        }
      }
    }
  };

  const int gend = min(g.ngroups, (split + 1) * g.gps);
  for (int grp = split * g.gps; grp < gend; grp++) {
    const int b0 = grp * g.nb;
    // The loads of a group, dy's and x's, go out together before any value is stored: a memory latency to a group.
    fetch(b0, 0);
    if (grp == split * g.gps) {
      // what no value is ever stored to, once: the planes' halo, and the k that pad dy's last step
      for (int e = tid; e < g.nb * kCT * g.XP / 4; e += kThreads) reinterpret_cast<f32x4*>(xL)[e] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (g.KW > g.K)
        for (int e = tid; e < kBM * (g.KW - g.K); e += kThreads) {
          const int f = e / (g.KW - g.K);
          dyL[f * g.DP + g.K + (e - f * (g.KW - g.K))] = 0.f;
        }
      __syncthreads();
    }
    put(0);
    for (int it = 1; it * kDy * kThreads < nq || it * kX * kThreads < nx; it++) {
      fetch(b0, it);
      put(it);
    }
    __syncthreads();
    // ---- MFMA over the group's k: A = dy (filter x k), B = x (k x (channel, tap)).  The
    // operands of step s + 1 and the position of step s + 2 are fetched before the MFMAs of
    // step s: a position leads to nine B reads, two LDS latencies that would otherwise sit
    // between the steps of a wavefront that has its SIMD to itself.
    // this wavefront's half of the group's steps: [kb, ke)
    const int nsteps = g.KW >> 2, half = (nsteps + 1) >> 1;
    const int kb = 4 * (khalf ? half : 0), ke = 4 * (khalf ? nsteps : half);
    const float* const arow = dyL + (16 * mt + li) * g.DP + lk;
    const int* const prow = ptab + lk;
    // The k that pad the last step (K..KW) carry dy = 0 and table position 0, so their B operand is real x data; an Inf there
    // would put 0 * Inf = NaN into the sum where the reference has Inf or a number.  That step comes by itself, behind the
    // others, with those lanes' B registers cleared.
    const bool padded = g.KW > g.K && ke == g.KW && kb < ke;
    const int steps = (ke - kb) / 4 - padded;
    const float* const xb = xL + xlane;
    auto operands = [&](int k, int pos, float& a, float (&b)[9]) __attribute__((always_inline)) {
      a = arow[k];
#pragma unroll
      for (int t = 0; t < 9; t++) b[t] = xb[pos + (t / 3) * kRowPitch + t % 3];
    };
    auto multiply = [&](float a, const float (&b)[9]) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < 9; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[t], acc[t], 0, 0, 0);
    };
    if (steps > 0) {
      // two operand sets, used in turn: while one feeds the MFMAs the other is being read.  (The fences keep the reads of a
      // set in front of the MFMAs they are meant to run under.  One way out of the loop, and nothing in it that looks at a
      // value: with the clearing in every step and a way out between the two turns each step waited for its own reads.  us,
      // slab sum included, before / now: 128 x 32 x 14 x 14 -> 64 26.1 / 25.0, 128 x 64 x 7 x 7 -> 128 22.3 / 21.0, three times as many images 55.3 / 50.5
      // and 52.7 / 47.9; beside the image gradients 35.5 / 34.3 and 30.8 / 29.7.)
      const int klast = kb + 4 * (steps - 1);
      float a0, a1, b0v[9], b1v[9];
      operands(kb, prow[kb], a0, b0v);
      int k = kb, pn = prow[min(kb + 4, klast)];
      auto turn = [&](float a, const float (&b)[9], float& an, float (&bn)[9]) __attribute__((always_inline)) {
        operands(min(k + 4, klast), pn, an, bn);
        pn = prow[min(k + 8, klast)];
        __builtin_amdgcn_sched_barrier(0);
        multiply(a, b);
        __builtin_amdgcn_sched_barrier(0);
        k += 4;
      };
      for (int two = steps >> 1; two > 0; two--) {
        turn(a0, b0v, a1, b1v);
        turn(a1, b1v, a0, b0v);
      }
      if (steps & 1) multiply(a0, b0v);
    }
    if (padded) {
      float a, b[9];
      operands(ke - 4, prow[ke - 4], a, b);
      if (g.KW - 4 + lk >= g.K) {
#pragma unroll
        for (int t = 0; t < 9; t++) b[t] = 0.f;
      }
      multiply(a, b);
    }
    __syncthreads();   // every wavefront is done with the planes before the next group lands
  }

  // ---- the second half's partial tile onto the first's, through LDS (the last barrier of the
  // loop has every wavefront past its reads of dyL): [tile row][t][lane] as 128-bit values
  f32x4* const red = reinterpret_cast<f32x4*>(dyL) + (mt * 9) * 64 + lane;
  if (khalf) {
#pragma unroll
    for (int t = 0; t < 9; t++) red[t * 64] = acc[t];
  }
  __syncthreads();
  // ---- register v of acc[t] is filter f0 + 16 mt + 4 lk + v, channel c0 + li, tap t.  The sixteen rows of a tile row are as
  // many values as its partial tile: they take that one's place in the order of dW's rows, and all threads store them.
  float* const tile = dyL;
  constexpr int kCols = kCT * 9;
  if (!khalf) {
#pragma unroll
    for (int t = 0; t < 9; t++) acc[t] = acc[t] + red[t * 64];
    __builtin_amdgcn_wave_barrier();   // (a wavefront's accesses to LDS are in order: its reads are done)
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
      for (int t = 0; t < 9; t++) tile[(16 * mt + 4 * lk + v) * kCols + li * 9 + t] = acc[t][v];
  }
  __syncthreads();
  float* const o = out + (int64_t)split * slab + (int64_t)f0 * g.CKK + c0 * 9;
  for (int e = tid; e < kBM * kCols / 4; e += kThreads) {
    const int f = e / (kCols / 4), col = 4 * (e - f * (kCols / 4));
    if (f0 + f < g.F) *reinterpret_cast<f32x4_a4*>(o + (int64_t)f * g.CKK + col) = reinterpret_cast<const f32x4*>(tile)[e];
  }
}

}  // namespace conv_wgrad_small

struct gh_wgrad_small_args {
  const float* x;
  const float* dy;
  float* out;
  conv_wgrad_small::WgGeom g;
  int64_t slab;
};
