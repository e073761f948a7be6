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
// wavefronts of a workgroup split the channels of one tile (kSplit), their sums meeting in LDS in wavefront order (of eight in
// float32 the upper four first each to the one four below), or
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

#include "gh_conv_lanes.h"

namespace {

using namespace conv_lanes;

// kRounds: a workgroup has every gridDim.x-th tile, of `tiles`.
template <class T, int WV, int TM, int V, int G, bool kSplit, bool kFlip, bool kPool, bool kRounds>
__global__ __launch_bounds__(WV * 64) __attribute__((amdgpu_waves_per_eu(WV == 8 || TM * V * G * sizeof(T) <= 32 ? 2 : 1))) void k_conv3x3_lanes(const Lanes<T> g, const ConvTail tail, int tiles) {
  constexpr int bytes = lds_of<T, WV, TM, V, G, kSplit>(kFlip);
  __shared__ __attribute__((aligned(16))) char lds[bytes ? bytes : 16];
  if constexpr (kRounds) {
    for (int tile = (int)blockIdx.x; tile < tiles; tile += (int)gridDim.x) {
      if (tile != (int)blockIdx.x) __syncthreads();   // before LDS is written again
      workgroup<T, WV, TM, V, G, kSplit, kFlip, kPool>(g, tail, tile, tiles, lds);
    }
  } else {
    workgroup<T, WV, TM, V, G, kSplit, kFlip, kPool>(g, tail, (int)blockIdx.x, (int)gridDim.x, lds);
  }
}

// How many workgroups of a kernel the device holds at once.
template <auto kKernel>
int64_t held_at_once(const gh_ctx* ctx, int threads) {
  static const int share = [&] {
    int n = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void*)kKernel, threads, 0) == hipSuccess && n > 0 ? n : 1 << 20;
  }();
  return (int64_t)share * ctx->cu_count;
}

// Where there are somewhat more tiles than workgroups that the device holds at once, a workgroup for each leaves the last ones to
// the places that fall free together, two on one compute unit and none on the next: 8 x 128 x 26 x 26 -> 256 pooled, 728 tiles
// for 512 places, 44.5 us, float64 8 x 32 x 104 x 104 -> 64, 676 for 512, 77.0.  With as many workgroups as places, each with
// every so many-th tile, the compute units have one more or none: 35.9 and 59.8.  From twice the places on the last round is
// the smaller part, and the kernel that walks takes some 0.2 us more.
template <class T, int WV, int TM, int V, int G, bool kSplit>
int launch(gh_ctx* ctx, Lanes<T> g, const ConvTail& tail, bool flip, bool pool) {
  constexpr int per = 16 * G * (kSplit ? 1 : WV);
  const int lines = g.groups;   // image rows (row pairs) in all, until here
  g.per_row = (g.cols + V - 1) / V;
  g.groups = lines * g.per_row * (pool ? 2 : 1);
  g.ftiles = (g.F + 16 * TM - 1) / (16 * TM);
  g.ptiles = (g.groups + per - 1) / per;
  g.ft_major = g.w_bytes > g.x_bytes;
  const int tiles = g.ftiles * g.ptiles;
  const auto go = [&](auto flips, auto pools) {
    constexpr bool F = decltype(flips)::value, P = decltype(pools)::value;
    constexpr auto one = k_conv3x3_lanes<T, WV, TM, V, G, kSplit, F, P, false>, rounds = k_conv3x3_lanes<T, WV, TM, V, G, kSplit, F, P, true>;
    const int64_t held = held_at_once<rounds>(ctx, WV * 64);
    const bool in_rounds = tiles > held && tiles < 2 * held;
    if (in_rounds) {
      ctx->joint[GH_JOINT_CONV_ROUNDS].launches++;
      ctx->joint[GH_JOINT_CONV_ROUNDS].form = 100 * WV + 10 * TM + kSplit;
    }
    hipLaunchKernelGGL((in_rounds ? rounds : one), dim3((unsigned)(in_rounds ? held : tiles)), dim3(WV * 64), 0, ctx->stream, g, tail, tiles);
    return gh_check_hip(ctx, hipGetLastError(), "conv3x3 launch");
  };
  using Yes = std::true_type;
  using No = std::false_type;
  if constexpr (sizeof(T) == 4) {
    if (pool) return go(No{}, Yes{});
  }
  if (G == 1 && flip && ctx->held.kind != kHeldNone)
    if (const int rc = gh_try_launch_gradients(ctx, g, WV, TM, kSplit, tiles); rc >= 0) return rc;
  return flip ? go(Yes{}, No{}) : go(No{}, No{});
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
// In place of the patch kernel (`patch`) a form of eight wavefronts, whose sums are as long as that kernel's, also where the estimates have it
// a sixth slower: both are high there, by more for these.  Of 520 drawn gradients and 200 forward passes the rule gives 58 and 20
// more to it, at 0.54 to 1.0 and 0.73 to 0.92 of the time.  us, before / now, with the launch that mirrors the filters: the gradient of
// 8 x 32 x 52 x 52 -> 64 16.6 / 13.6, with its filter gradient 39.3 / 31.7; 15 x 64 x 49 x 58 -> 128 77.5 / 64.0; forward 7 x 512 x 8 x 8 ->
// 1024 50.7 / 39.3, 5 x 256 x 9 x 9 -> 512 25.0 / 22.2.  The form of four wavefronts is quicker for some (6 x 512 x 10 x 10 ->
// 1024 81.2 / 72.2) and slower for others (8 x 512 x 13 x 13 -> 1024 116 / 145), and its sums are twice as long.
//
// float32 where that is not so: a wavefront with a tile of its own and all channels, for few channels and many pixels, where
// the split forms have one or two quads to a wavefront and the wide-image kernel stages as much as it multiplies.  Only in place
// of a kernel whose sums run over all channels too (`whole`), since its own are longer than those of one that splits them: the
// gradient of 4 x 128 x 60 x 60 -> 64 would be off by 4.3e-7 of its norm instead of 1.6e-7, that of 13 x 96 x 45 x 45 -> 48, which
// runs as a split form over dy, by 2.9e-7 instead of 8.1e-8, that of 234 x 8 x 15 x 15 -> 32 by 2.5e-7, on the small-image
// kernel 2.0e-7.  us, before / now: 8 x 16 x 104 x 104 -> 32 22.9 / 15.9, pooled 17.9 / 13.6, its gradient 24.2 / 13.6; 8 x 16 x 104 x 104 -> 16
// 15.8 / 10.0 and its gradient 17.8 / 8.7; 8 x 32 x 104 x 104 -> 64 46.7 / 39.7 (80 TFLOP/s); 8 x 16 x 208 x 208 -> 32's
// gradient 45.8 / 36.1; 1 x 16 x 208 x 208 -> 32 pooled 11.0 / 8.7.
int gh_conv_lanes_form(const gh_cmd& c, bool flip, int cus, double other_us, bool patch, bool whole) {
  if (getenv("GORGONIA_HIP_CONV_NO_LANES")) return -1;   // tuning switch: the other kernels only
  const bool f64 = gh_dtype_of(c.flags) == GH_F64;
  Lanes<double> g;   // (the narrower of the two in what its offsets reach)
  if (!fill(c, flip, false, &g) || g.F < 8 || g.C < 8 || g.oh < 2) return -1;
  double us;
  const int split = quickest(c, flip, f64, cus, 0, f64 && !flip ? 4 : 3, &us);
  if (other_us <= 0 || us < other_us / 1.17) return split;
  if (f64) return -1;
  if (patch) {
    const int eight = quickest(c, flip, false, cus, 0, 2, &us);
    return us < other_us / 0.85 ? eight : -1;
  }
  if (!whole) return -1;
  const int form = quickest(c, flip, false, cus, 3, 5, &us);
  return us < other_us / 1.1 ? form : -1;
}

// The quickest for a float32 forward command of the forms that add as `form` does: eight wavefronts' shares of the channels, four's, or
// all channels in one chain.
int gh_conv_lanes_form_like(const gh_cmd& c, int form, int cus) {
  double us;
  return form < 2 ? quickest(c, false, false, cus, 0, 2, &us) : form == 2 ? form : quickest(c, false, false, cus, 3, 5, &us);
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
