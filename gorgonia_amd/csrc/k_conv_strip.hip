// Conv2d 3x3 / stride 1 / padding 1 of three or four channels, float32: a network's first layer over large images.
//
// One quad of channels is all there is to multiply, so that what surrounds the MFMAs decides: the wide-image kernel stages
// a tile through LDS for 9 MFMAs a tile of results.  Here nothing is staged and a wavefront stays with its filters.  On the
// 16x16x4 MFMA, k is the channel (the fourth of three is zero): lane (i, q) holds channel q of filter i's nine taps for the
// whole run, and of four neighbouring columns and the one on each side the rows of channel q under them.  A wavefront has 64
// columns and walks down the image two rows at a time, so that a row of x is loaded once (one wide load and two single ones)
// and is the lower, middle and upper filter row in turn; the next two rows are on their way under the MFMAs.  A value outside
// the image has an offset that the buffer's range check turns into zero.  A result's sum takes the taps in order, as the
// wide-image kernel's does, to the same bits.  A lane ends with four columns of four filters in two rows: it normalises,
// rectifies and pools them in its registers.
//
// Bound: where there are many rows, the MFMAs (11 us of 8 x 3 x 416 x 416 -> 16) and the epilogue's vector instructions (8),
// which add up; else the first loads and the stores behind them, which all wavefronts come to together.  us, the wide-image
// kernel / here: 8 x 3 x 416 x 416 -> 16 with BatchNorm, LeakyRelu and pooling 37.9 / 30.1, plain 40.5 / 31.3; one image 11.2 /
// 8.4 and 11.8 / 8.0; 8 x 3 x 208 x 208 -> 16 plain 16.0 / 13.0; 4 x 3 x 320 x 320 21.0 / 13.5; 8 x 4 x 100 x 100 -> 20 13.8 / 8.3.
#include <algorithm>
#include <cstdlib>

#include "gh_conv_common.h"
#include "gh_internal.h"

namespace {

constexpr int kOutside = 0x7ffffff0;   // past every buffer: a load from there is zero
constexpr int kWaves = 4;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
typedef float f32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

struct Strip {
  const float* x; const float* w; float* y;
  int C, H, W, F;
  int x_bytes;
  int blocks, runs, rows, ftiles, total;   // column blocks of 64, runs of `rows` rows, filter tiles; strips in all
};

struct Row { float v[6]; };   // columns ox - 1 .. ox + 4 of the lane's channel

template <bool POOL>
__global__ __launch_bounds__(kWaves * 64) void k_conv3x3_strip(const Strip g, const ConvTail tail) {
  const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
  const int id = __builtin_amdgcn_readfirstlane(blockIdx.x * kWaves + (threadIdx.x >> 6));
  if (id >= g.total) return;
  // neighbours in a row first: they share the columns at their sides
  int r = id;
  const int cb = r % g.blocks; r /= g.blocks;
  const int run = r % g.runs; r /= g.runs;
  const int ft = r % g.ftiles, b = r / g.ftiles;
  const int f0 = ft * 16, y0 = run * g.rows, y1 = min(y0 + g.rows, g.H);
  const int ox = min(cb * 64 + 4 * i, g.W - 4);   // (past the row's end: its last four columns again, the same values)
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)g.x, 0, g.x_bytes, 0x00020000);
  const int base = q < g.C ? (((b * g.C + q) * g.H) * g.W + ox) * 4 : kOutside;
  const bool left = q < g.C && ox > 0, right = q < g.C && ox + 4 < g.W;
  auto load = [&](int iy, Row& row) __attribute__((always_inline)) {
    const bool in = (unsigned)iy < (unsigned)g.H;   // the same in all lanes
    const int s = in ? iy * g.W * 4 : 0;
    const f32x4 m = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, in ? base : kOutside, s, 0));
    row.v[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, in && left ? base - 4 : kOutside, s, 0));
    row.v[5] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, in && right ? base + 16 : kOutside, s, 0));
#pragma unroll
    for (int e = 0; e < 4; e++) row.v[1 + e] = m[e];
  };
  Row r0, r1, r2, r3;
  load(y0 - 1, r0);
  load(y0, r1);
  load(y0 + 1, r2);
  load(y0 + 2, r3);
  float w9[9];
#pragma unroll
  for (int t = 0; t < 9; t++) w9[t] = q < g.C ? g.w[(min(f0 + i, g.F - 1) * g.C + q) * 9 + t] : 0.0f;
  // the lane's filters f0 + 4 q .. + 3
  float ta[4], tb[4], tg[4], te[4];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int f = min(f0 + 4 * q + v, g.F - 1);
    ta[v] = tg[v] = 1.0f;
    tb[v] = te[v] = -0.0f;
    if (tail.mean) {   // (as conv_tail_table has them)
      const float a = 1.0f / sqrtf(tail.var[f] + tail.eps);
      ta[v] = a;
      tb[v] = -tail.mean[f] * a;
      if (tail.gamma) tg[v] = tail.gamma[f];
      if (tail.beta) te[v] = tail.beta[f];
    }
  }
  const bool mine = cb * 64 + 4 * i < g.W + 3;   // a lane past the row's last four has nothing to store
  auto step = [&](int y, Row& a, Row& b_, Row& c, Row& d, Row& e, Row& f) __attribute__((always_inline)) {
    // rows y - 1, y, y + 1, y + 2 are a .. d; y + 3 and y + 4 go to e and f
    const bool more = y + 2 < y1;
    load(more ? y + 3 : -1, e);
    load(more ? y + 4 : -1, f);
    f32x4 acc[2][4];
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int n = 0; n < 4; n++) acc[k][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
      for (int k = 0; k < 2; k++)
#pragma unroll
        for (int n = 0; n < 4; n++) {
          const Row& src = t / 3 + k == 0 ? a : t / 3 + k == 1 ? b_ : t / 3 + k == 2 ? c : d;
          acc[k][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(w9[t], src.v[n + t % 3], acc[k][n], 0, 0, 0);
        }
    conv_tail_dispatch(tail, [&](auto BN, auto ACT) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int fl = f0 + 4 * q + v;
        float z[2][4];
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
          for (int n = 0; n < 4; n++) {
            float u = acc[k][n][v];
            if constexpr (BN()) {
              u = u * ta[v];
              u = u + tb[v];
              u = tg[v] * u;
              u = u + te[v];
            }
            z[k][n] = act_apply(u, ACT(), tail.alpha);
          }
        if (fl >= g.F || !mine) continue;
        if constexpr (POOL) {
          if (y + 1 >= g.H) continue;
          float best[2];
#pragma unroll
          for (int k = 0; k < 2; k++) {
            best[k] = -3.402823466e+38f;   // scan order and strict > of the pooling kernel
            if (z[0][2 * k] > best[k]) best[k] = z[0][2 * k];
            if (z[0][2 * k + 1] > best[k]) best[k] = z[0][2 * k + 1];
            if (z[1][2 * k] > best[k]) best[k] = z[1][2 * k];
            if (z[1][2 * k + 1] > best[k]) best[k] = z[1][2 * k + 1];
          }
          *(f32x2_a4*)(g.y + (((int64_t)b * g.F + fl) * (g.H >> 1) + (y >> 1)) * (g.W >> 1) + (ox >> 1)) = f32x2_a4{best[0], best[1]};
        } else {
          float* const out = g.y + (((int64_t)b * g.F + fl) * g.H + y) * g.W + ox;
          *(f32x4_a4*)out = f32x4_a4{z[0][0], z[0][1], z[0][2], z[0][3]};
          if (y + 1 < g.H) *(f32x4_a4*)(out + g.W) = f32x4_a4{z[1][0], z[1][1], z[1][2], z[1][3]};
        }
      }
    });
  };
  Row r4, r5;
  for (int y = y0; y < y1; y += 6) {
    step(y, r0, r1, r2, r3, r4, r5);
    if (y + 2 >= y1) break;
    step(y + 2, r2, r3, r4, r5, r0, r1);
    if (y + 4 >= y1) break;
    step(y + 4, r4, r5, r0, r1, r2, r3);
  }
}

}  // namespace

// Three or four channels, an image whose rows hold a lane's four columns; of a pooled command even rows and columns.
bool gh_conv_strip_takes(const gh_cmd& c) {
  if (getenv("GORGONIA_HIP_CONV_NO_STRIP")) return false;   // tuning switch: the wide-image kernel
  if (c.flags & (GH_FLAG_CONV_PRE | GH_FLAG_CONV_KEEP)) return false;
  for (int k : {5, 6}) if (c.dim[k] != 3) return false;
  for (int k : {7, 8, 9, 10, 11, 12}) if (c.dim[k] != 1) return false;
  const int64_t B = c.dim[0], C = c.dim[1], H = c.dim[2], W = c.dim[3], F = c.dim[4];
  if (C < 3 || C > 4 || W < 4 || W % 2 || H % 2) return false;
  return B * C * H * W < (1 << 29) - 64 && B * F * H * W <= INT32_MAX && ((c.ptr[0] | c.ptr[1] | c.ptr[2]) & 3) == 0;
}

int gh_launch_conv_strip(gh_ctx* ctx, const gh_cmd& c) {
  Strip g;
  g.x = (const float*)(uintptr_t)c.ptr[0];
  g.w = (const float*)(uintptr_t)c.ptr[1];
  g.y = (float*)(uintptr_t)c.ptr[2];
  g.C = (int)c.dim[1];
  g.H = (int)c.dim[2];
  g.W = (int)c.dim[3];
  g.F = (int)c.dim[4];
  const int64_t B = c.dim[0];
  g.x_bytes = (int)(B * g.C * g.H * g.W * 4);
  g.blocks = (g.W + 63) / 64;
  g.ftiles = (g.F + 15) / 16;
  const int64_t columns = B * g.blocks * g.ftiles;
  // rows of a run: the more, the less is loaded twice, but sixteen wavefronts to a compute unit, of which twelve fit at once
  // (8 x 3 x 416 x 416 -> 16 with four rows 30.1 us, with 2, 6, 10 and 16 35.2, 34.1, 31.6 and 33.5)
  int rows = 16;
  while (rows > 2 && columns * ((g.H + rows - 1) / rows) < 16 * (int64_t)ctx->cu_count) rows -= 2;
  g.rows = rows;
  g.runs = (g.H + rows - 1) / rows;
  const int64_t total = columns * g.runs;
  if (total > INT32_MAX) return gh_fail(ctx, GH_EINVAL, "conv2d: tensor too large for 32-bit indexing");
  g.total = (int)total;
  const dim3 grid((unsigned)((total + kWaves - 1) / kWaves));
  const ConvTail tail = conv_tail(c);
  hipLaunchKernelGGL((c.flags & GH_FLAG_CONV_POOL2 ? k_conv3x3_strip<true> : k_conv3x3_strip<false>), grid, dim3(kWaves * 64), 0, ctx->stream, g, tail);
  return gh_check_hip(ctx, hipGetLastError(), "conv3x3 launch");
}
