// Filter gradient of Conv2d 3x3 / stride 1, float32 and float64, on the 16x16x4 MFMA with every operand
// taken from memory straight into the lane that feeds it.
//
// dW[f][c][ky][kx] is a sum over (image, output row, output column) of dy[f] * x[c] shifted by the tap: a small
// result summed over a long axis.  Tiled through LDS (64 x 64 results per workgroup, im2col gathers) a network's
// first layers leave most of a tile empty and their gathers, not the matrix cores, set the time.  Measured, slab sum
// included, against the kernels that took these shapes before: 3 -> 16 channels over 8 x 208 x 208 pixels 17.6 us
// (274), 16 -> 32 over 8 x 104 x 104 21.9 (75), 128 -> 256 over 8 x 52 x 52 170 (213: 75 against 60 TFLOP/s), float64
// 32 -> 64 over 50 x 14 x 14 19.8 (29.8).  Small ones are bound by what surrounds the MFMAs (first loads 1 us,
// meeting of the wavefronts 3, slab sum 5), large ones by address and edge arithmetic between them.  Here
//   * a wavefront owns 16 TM filters x 16 channels and all nine taps (TM * 9 accumulators) and walks chunks of
//     4 P consecutive output columns of one row.  Lane (i, q) of a chunk holds P consecutive columns: of dy row i
//     one P-wide load, of channel i the P + 2 values under each of the three filter rows.  MFMA step t of the
//     chunk takes element t of dy and element t + kx of x, so three loads feed nine taps and P steps, nothing
//     is staged, and no barrier stands in the loop; the loads of a chunk are issued before the MFMAs of the
//     chunk in front of it.
//   * with fewer than 16 channels the columns of a tile are (channel, tap) pairs instead, packed without gaps,
//     and each has its own P-wide load (kPacked).
//   * the long axis is cut among wavefronts and workgroups; the four wavefronts of a workgroup meet in LDS, the
//     workgroups' slabs in k_slab_sums, both in a fixed order.
// P is 4, or 2 where a row has at most eight columns.
#include <algorithm>

#include "gh_conv_wgrad.h"

namespace {

using namespace conv_wgrad;

template <class T, int TM, int P, int NT, bool kPacked>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void k_conv3x3_wgrad(const Wg<T> g) {
  __shared__ __attribute__((aligned(16))) char lds[lds_of<T, NT>()];
  workgroup<T, TM, P, NT, kPacked>(g, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, lds);
}

template <class T>
bool fill(const gh_cmd& c, Wg<T>* g) {
  for (int i : {5, 6}) if (c.dim[i] != 3) return false;
  for (int i : {9, 10, 11, 12}) if (c.dim[i] != 1) return false;
  const int64_t B = c.dim[0], C = c.dim[1], H = c.dim[2], W = c.dim[3], F = c.dim[4];
  const int64_t oh = gh_conv_out(H, 3, c.dim[7], 1, 1), ow = gh_conv_out(W, 3, c.dim[8], 1, 1);
  if (B <= 0 || C <= 0 || F <= 0 || oh <= 0 || ow <= 0 || c.dim[7] > 1024 || c.dim[8] > 1024) return false;
  if (H > (1 << 20) || W > (1 << 20) || C > (1 << 20) || F > 65535 * 16) return false;
  g->x = (const T*)(uintptr_t)c.ptr[0];
  g->dy = (const T*)(uintptr_t)c.ptr[1];
  // 32-bit byte offsets; an image holds a whole load, so that none but the first and last image's stick out of a tensor
  const int64_t most = ((int64_t)1 << 31) / (int64_t)sizeof(T) - 64;
  if (B * C * H > most / W || B * F * oh > most / ow || C * H * W < 6 || F * oh * ow < 4) return false;
  g->x_total = (int)(B * C * H * W);
  g->dy_total = (int)(B * F * oh * ow);
  g->B = (int)B; g->C = (int)C; g->H = (int)H; g->W = (int)W; g->F = (int)F; g->oh = (int)oh; g->ow = (int)ow;
  g->padH = (int)c.dim[7]; g->padW = (int)c.dim[8];
  const int px = ow <= 8 ? 8 : 16;
  g->nch = (int)((ow + px - 1) / px);
  const int64_t items = B * oh * g->nch;
  if (items > INT32_MAX / 2) return false;
  g->items = (int)items;
  return true;
}

// Workgroups along the long axis.  To a compute unit: what a wavefront does besides its MFMAs - the first loads, meeting the
// others, a slab to be summed - costs as much as some ten chunks of a channel tile, so one; packed tiles, three.
int64_t slices_of(int64_t tiles, int64_t items, int cus, bool packed) {
  const int64_t slices = std::max<int64_t>(1, (packed ? 3 : 1) * (int64_t)cus / tiles);
  return std::min<int64_t>(slices, std::max<int64_t>(1, items / (4 * kWaves)));
}

template <class T, int TM, int P, int NT, bool kPacked>
int launch(gh_ctx* ctx, Wg<T> g, T* dw) {
  const int64_t ft = (g.F + 16 * TM - 1) / (16 * TM), ct = kPacked ? 1 : (g.C + 15) / 16;
  const int64_t results = (int64_t)g.F * g.C * 9;
  int64_t slices = slices_of(ft * ct, g.items, ctx->cu_count, kPacked);
  if (slices > 1 && slices * results * (int64_t)sizeof(T) > ctx->workspace_bytes) {
    if (int rc = gh_ws_short(ctx, slices * results * (int64_t)sizeof(T))) return rc;
    slices = std::max<int64_t>(1, ctx->workspace_bytes / (results * (int64_t)sizeof(T)));
  }
  g.per = (int)((g.items + slices * kWaves - 1) / (slices * kWaves));
  slices = (g.items + (int64_t)g.per * kWaves - 1) / ((int64_t)g.per * kWaves);
  g.out = slices > 1 ? (T*)gh_slab_space(ctx, slices * results * (int64_t)sizeof(T)) : dw;
  const dim3 grid((unsigned)slices, (unsigned)ct, (unsigned)ft);
  constexpr int held = kPacked ? kHeldNone : sizeof(T) == 8 ? (P == 4 ? kHeldF64 : kHeldF64Narrow) : TM == 2 && P == 4 ? kHeldF32 : kHeldNone;
  int rc = GH_OK;
  if (held != kHeldNone && gh_may_hold(ctx, g.out)) {
    static_assert(sizeof(g) <= sizeof(ctx->held.args), "the argument fits");
    ctx->held.kind = held;
    ctx->held.grid = grid;
    memcpy(ctx->held.args, &g, sizeof(g));
  } else {
    hipLaunchKernelGGL((k_conv3x3_wgrad<T, TM, P, NT, kPacked>), grid, dim3(kThreads), 0, ctx->stream, g);
    rc = gh_check_hip(ctx, hipGetLastError(), "filter-gradient launch");
  }
  if (rc || slices == 1) return rc;
  // 64 results to a workgroup of the sum where that makes enough workgroups, else 16
  const bool many = results >= 64 * (int64_t)ctx->cu_count;
  return gh_sum_slabs(ctx, {g.out, dw, results, (int)slices, sizeof(T) == 8 ? (many ? kSumGroups64F64 : kSumGroups16F64) : many ? kSumGroups64 : kSumGroups16});
}

template <class T>
int pick(gh_ctx* ctx, const Wg<T>& g, T* dw) {
  // packed columns take fewer tiles than nine taps of a channel tile up to eight channels
  if (g.C == 1) return launch<T, 1, 4, 1, true>(ctx, g, dw);
  if (g.C <= 3) return launch<T, 1, 4, 2, true>(ctx, g, dw);
  if (g.C <= 5) return launch<T, 1, 4, 3, true>(ctx, g, dw);
  if (g.C <= 8) return launch<T, 1, 4, 5, true>(ctx, g, dw);
  // two filter tiles share the loads of x; of float64 one fills the registers
  if constexpr (sizeof(T) == 4) {
    if (g.F > 16) return g.ow <= 8 ? launch<T, 2, 2, 9, false>(ctx, g, dw) : launch<T, 2, 4, 9, false>(ctx, g, dw);
  }
  return g.ow <= 8 ? launch<T, 1, 2, 9, false>(ctx, g, dw) : launch<T, 1, 4, 9, false>(ctx, g, dw);
}

}  // namespace

int gh_launch_held_wgrad(gh_ctx* ctx) {
  if (ctx->held.kind == kHeldF32) {
    Wg<float> g;
    memcpy(&g, ctx->held.args, sizeof(g));
    hipLaunchKernelGGL((k_conv3x3_wgrad<float, 2, 4, 9, false>), ctx->held.grid, dim3(kThreads), 0, ctx->stream, g);
    return gh_check_hip(ctx, hipGetLastError(), "filter-gradient launch");
  }
  Wg<double> g;
  memcpy(&g, ctx->held.args, sizeof(g));
  hipLaunchKernelGGL((ctx->held.kind == kHeldF64 ? k_conv3x3_wgrad<double, 1, 4, 9, false> : k_conv3x3_wgrad<double, 1, 2, 9, false>), ctx->held.grid, dim3(kThreads), 0,
                     ctx->stream, g);
  return gh_check_hip(ctx, hipGetLastError(), "filter-gradient launch");
}

// Whether a channel tile's walk is the slower one.  Its tiles hold 16 channels, 16 or 32 filters and chunks of 16 (8)
// columns of a row, so few channels over a multiple of 16, or rows little longer than a chunk, leave much of it empty; the
// tiled kernel pads filters and (channel, tap) columns to 64 and no row.  Both are so many us per round of their tiles'
// chunks over the compute units, and per million slab values; fitted to 320 shapes in float32 and 277 in float64 of 1 to 64
// images of 3 x 3 to 208 x 208, 9 to 400 channels, 8 to 300 filters, within 10 % for most.  By it 55 x 21 x 90 x 3 -> 157 in
// float64 takes 54 us (120 here), 12 x 249 x 20 x 20 -> 376 119 (161), 11 x 198 x 21 x 21 -> 173 63 (77).
static bool tiled_is_quicker(const gh_cmd& c, const Wg<double>& g, int cus) {
  const bool f64 = gh_dtype_of(c.flags) == GH_F64;
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t results = (int64_t)g.F * g.C * 9, pixels = g.dy_total / g.F;
  const int64_t ft64 = cdiv(g.F, 64) * cdiv(g.C * 9, 64), nk = cdiv(pixels, f64 ? 16 : 32);
  int64_t slabs = std::min<int64_t>(std::min<int64_t>(cdiv(5 * (int64_t)cus / 2, ft64), nk / 4), f64 ? 512 : 64);
  slabs = std::max<int64_t>(1, std::min<int64_t>(slabs, GH_NOALLOC_SCRATCH_BYTES / (results * (f64 ? 8 : 4))));
  if (f64 && pixels * results < (int64_t)1 << 22) return false;   // the tiled kernel leaves these to one thread a result
  const int tm = !f64 && g.F > 16 ? 2 : 1;
  const int64_t tiles = cdiv(g.F, 16 * tm) * cdiv(g.C, 16), slices = slices_of(tiles, g.items, cus, false);
  const double chunks = (double)(cdiv(slices * tiles, cus) * cdiv(g.items, slices * kWaves)) * tm * (g.ow <= 8 ? 0.5 : 1.0);
  const double here = f64 ? 7.3 + 1.55 * chunks + 5.4e-6 * (double)(slices * results) : 6.6 + 0.80 * chunks + 4.5e-6 * (double)(slices * results);
  const double there = f64 ? 12.3 + 1.26 * (double)(ft64 * nk) / cus + 0.8e-6 * (double)(slabs * results)
                           : 11.0 + 1.06 * (double)(ft64 * nk) / cus + 1.0e-6 * (double)(slabs * results);
  return here > (f64 ? 1.06 : 1.0) * there;
}

// Whether k_conv3x3_wgrad takes a filter gradient: 3x3, stride 1.  Of float32, not the shapes the small-image and
// the single-channel kernel hold in LDS, and up to four channels only where there are enough pixels to cut up
// (below that the vector kernel's few workgroups do; of a single channel it wastes the least).
static bool can_take(const gh_cmd& c, Wg<double>* g) {   // (the narrower of the two in what its offsets reach)
  if (!fill(c, g) || g->F < 8) return false;
  const int64_t pixels = g->dy_total / g->F;
  if (g->C <= 8 && g->ow <= 8) return false;
  if (gh_dtype_of(c.flags) == GH_F64) return pixels >= 256;
  return pixels >= (g->C == 1 ? 65536 : g->C <= 4 ? 16384 : 256);
}
bool gh_conv_wgrad_takes(const gh_cmd& c, int cus) {
  Wg<double> g;
  return can_take(c, &g) && (g.C <= 8 || !tiled_is_quicker(c, g, cus));
}
// Slabs that the tiled kernels may use for a command: those of a shape that this one could take, and without scratch, fit
// any scratch, so that the choice refuses nothing.
int64_t gh_conv_wgrad_slab_limit(const gh_cmd& c, int64_t slab_bytes) {
  Wg<double> g;
  return can_take(c, &g) ? std::max<int64_t>(1, GH_NOALLOC_SCRATCH_BYTES / slab_bytes) : INT64_MAX;
}

int gh_launch_conv_wgrad(gh_ctx* ctx, const gh_cmd& c) {
  if (gh_dtype_of(c.flags) == GH_F64) {
    Wg<double> g;
    if (!fill(c, &g)) return gh_fail(ctx, GH_ESTATE, "filter gradient: not a shape of this kernel");
    return pick<double>(ctx, g, (double*)(uintptr_t)c.ptr[2]);
  }
  Wg<float> g;
  if (!fill(c, &g)) return gh_fail(ctx, GH_ESTATE, "filter gradient: not a shape of this kernel");
  return pick<float>(ctx, g, (float*)(uintptr_t)c.ptr[2]);
}
