// A 3x3 convolution's filter gradient and its image gradient in one launch.
//
// The two read the same dy and neither reads what the other writes.  Each is some 12 to 20 us in a training step, of which its
// matrix instructions are a third: first loads, the wavefronts' meeting, a last round of few workgroups.  Here the filter
// gradient's workgroups, the longer ones, come first in the grid and the image gradient's behind them, so that one's waits run
// under the other's instructions.  Both are the workgroups of the kernels they have alone (gh_conv_wgrad.h,
// gh_conv_wgrad_small.h, gh_conv_lanes.h): the stored bits are theirs.
//
// Bound: the matrix instructions of both and, of small ones, the launch; where both kernels fill the device by themselves one
// launch takes what two do.  us, slab sum included, apart / together: float32 128 x 32 x 14 x 14 -> 64 38.7 / 36.5, 128 x 64 x 7 x 7
// -> 128 34.9 / 31.3, three times as many images 90.6 / 80.2 and 82.8 / 72.6, 8 x 64 x 26 x 26 -> 128 34.9 / 32.9, 8 x 16 x 52 x 52 -> 32
// 23.4 / 19.3, 8 x 16 x 104 x 104 -> 32 34.5 / 33.8; float64 50 x 64 x 7 x 7 -> 128 31.0 / 28.1, 96 x 32 x 14 x 14 -> 64 47.1 / 40.3,
// 8 x 32 x 26 x 26 -> 64 23.9 / 20.0.  Of 350 drawn shapes of 1 to 360 images of 4 x 4 to 110 x 110 (float64 to 32 x 32) none was
// slower by more than 2.4 % and the 249 that a kernel here has both of took 0.85 of their time, so there is no rule but that.  (Registers
// for a third workgroup to a compute unit, float64's by two meetings of half the LDS, spill and lose what they gain: 96 x 32 x 14 x 14
// 48.7.  The float32 form that had two filter-gradient workgroups side by side in eight wavefronts spilled, 57 for 35.)
//
// Where the convolution's input was pooled (2x2 / 2, even extents), the pooling's gradient and its Rectify's, which take the image
// gradient value by value, are in the launch as well (gh_unpool_follows): the windows are loaded under the meeting of the wavefronts
// that share a tile's channels, and the pass over memory runs under the other workgroups' matrix instructions.  Only behind the
// kernels whose wavefronts share the channels; the others store whole rows from registers.  Bound: the matrix instructions, and the
// stores of those workgroups that end last.  Beside a small-image filter gradient the image gradient's therefore stand in front where
// there are more of both than begin at once (two to a compute unit): 128 x 32 x 14 x 14 -> 64 in two launches 25.4 + 7.2 us, in one
// behind the filter gradient 33.3, in front 31.4; of 128 x 64 x 7 x 7 -> 128, 480 workgroups, 24.4 + 5.3, 25.8, 26.7; float64's are slower in
// front (50 x 32 x 14 x 14 -> 64 27.8 / 34.1).  (The windows loaded in front of the channels: 35.8, with spilled registers.)
// A training step of the example's network, two such layers: 128 images 181.0 / 176.2, 50 in float64 181.1 / 175.4, 13 images 132.9 / 128.0.
//
// gh_submit holds a filter gradient back (gh_held_filter) where an image gradient that has nothing to do with its result
// stands beside it; the image gradient's launch takes it along, or it is launched by itself behind that.
#include <algorithm>
#include <cstdlib>
#include <mutex>

#include "gh_conv_lanes.h"
#include "gh_conv_wgrad.h"
#include "gh_conv_wgrad_small.h"

namespace {

using conv_lanes::Lanes;
using conv_lanes::Unpool;
using conv_wgrad::Wg;

// The filter gradient's grid: x, y and all workgroups.
struct Grid {
  int x, y, all;
  __device__ __forceinline__ void at(int b, int* bx, int* by, int* bz) const {
    const int r = b / x;
    *bx = b - r * x;
    *bz = r / y;
    *by = r - *bz * y;
  }
};

template <int kRowPitch, int TM, bool kUnpool>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void k_conv3x3_gradients_small(const gh_wgrad_small_args w, const Grid grid, const Lanes<float> g,
                                                                                                          const Unpool<float> u, const int front) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  int b = (int)blockIdx.x;
  if (kUnpool && front) b = b < front ? b + grid.all : b - front;   // the image gradient's workgroups stand in front
  if (b < grid.all) {
    int bx, by, bz;
    grid.at(b, &bx, &by, &bz);
    conv_wgrad_small::workgroup<kRowPitch>(w.x, w.dy, w.out, w.g, w.slab, bx, by, bz, (float*)lds);
  } else {
    conv_lanes::workgroup<float, 8, TM, 4, 1, true, true, false, kUnpool>(g, ConvTail{}, b - grid.all, (int)gridDim.x - grid.all, lds, u);
  }
}

// (Where the image gradient's workgroups have eight wavefronts, the filter gradient's use the first four of theirs.)
template <class T, int TMW, int P, int WV, int TM, int V, bool kSplit, bool kUnpool>
__global__ __launch_bounds__(WV * 64) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : 3))) void k_conv3x3_gradients(const Wg<T> w, const Grid grid, const Lanes<T> g,
                                                                                                                          const Unpool<T> u) {
  constexpr int wl = conv_wgrad::lds_of<T, 9>(), ll = conv_lanes::lds_of<T, WV, TM, V, 1, kSplit>(true);
  __shared__ __attribute__((aligned(16))) char lds[wl > ll ? wl : ll];
  const int b = (int)blockIdx.x;
  if (b < grid.all) {
    if (WV > conv_wgrad::kWaves && (int)threadIdx.x >= conv_wgrad::kThreads) return;
    int bx, by, bz;
    grid.at(b, &bx, &by, &bz);
    conv_wgrad::workgroup<T, TMW, P, 9, false>(w, bx, by, bz, lds);
  } else {
    conv_lanes::workgroup<T, WV, TM, V, 1, kSplit, true, false, kUnpool>(g, ConvTail{}, b - grid.all, (int)gridDim.x - grid.all, lds, u);
  }
}

Grid grid_of(const gh_held_filter& h) { return {(int)h.grid.x, (int)h.grid.y, (int)(h.grid.x * h.grid.y * h.grid.z)}; }

template <class T> Unpool<T> unpool_of(const gh_ctx* ctx) {
  const gh_unpool& u = ctx->unpool;
  return {(const T*)(uintptr_t)u.a, (const T*)(uintptr_t)u.z, (T*)(uintptr_t)u.da, (T*)(uintptr_t)u.dz};
}

template <int kRowPitch, int TM, bool kUnpool>
int go_small_as(gh_ctx* ctx, const Lanes<float>& g, int blocks) {
  static std::once_flag once;
  static hipError_t attr_rc = hipSuccess;
  std::call_once(once, [] { attr_rc = hipFuncSetAttribute((const void*)k_conv3x3_gradients_small<kRowPitch, TM, kUnpool>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); });
  if (attr_rc != hipSuccess) return gh_check_hip(ctx, attr_rc, "hipFuncSetAttribute(conv3x3 gradients)");
  const Grid grid = grid_of(ctx->held);
  gh_wgrad_small_args w;
  memcpy(&w, ctx->held.args, sizeof w);
  const size_t lds = std::max<size_t>(ctx->held.lds, conv_lanes::lds_of<float, 8, TM, 4, 1, true>(true));
  hipLaunchKernelGGL((k_conv3x3_gradients_small<kRowPitch, TM, kUnpool>), dim3((unsigned)(grid.all + blocks)), dim3(512), lds, ctx->stream, w, grid, g, unpool_of<float>(ctx),
                     grid.all + blocks > 2 * ctx->cu_count ? blocks : 0);
  ctx->unpool.done = kUnpool;
  return GH_OK;
}
template <int kRowPitch, int TM>
int go_small(gh_ctx* ctx, const Lanes<float>& g, int blocks) {
  return ctx->unpool.dz ? go_small_as<kRowPitch, TM, true>(ctx, g, blocks) : go_small_as<kRowPitch, TM, false>(ctx, g, blocks);
}

template <class T, int TMW, int P, int WV, int TM, int V, bool kSplit, bool kUnpool = false>
int go(gh_ctx* ctx, const Lanes<T>& g, int blocks) {
  const Grid grid = grid_of(ctx->held);
  Wg<T> w;
  memcpy(&w, ctx->held.args, sizeof w);
  hipLaunchKernelGGL((k_conv3x3_gradients<T, TMW, P, WV, TM, V, kSplit, kUnpool>), dim3((unsigned)(grid.all + blocks)), dim3(WV * 64), 0, ctx->stream, w, grid, g, unpool_of<T>(ctx));
  ctx->unpool.done = kUnpool;
  return GH_OK;
}

int done(gh_ctx* ctx, int rc, int tm, bool split) {
  auto& j = ctx->joint[GH_JOINT_CONV_GRADIENTS];
  j.launches += rc == GH_OK;
  j.form = 100 * ctx->held.kind + 10 * tm + split;
  if (ctx->unpool.done) {
    ctx->joint[GH_JOINT_UNPOOLED].launches += rc == GH_OK;
    ctx->joint[GH_JOINT_UNPOOLED].form = j.form;
  }
  ctx->held.kind = kHeldNone;
  return rc ? rc : gh_check_hip(ctx, hipGetLastError(), "convolution gradients launch");
}

bool apart(uint64_t a, int64_t na, uint64_t b, int64_t nb) { return a + (uint64_t)na <= b || b + (uint64_t)nb <= a; }

}  // namespace

int gh_try_launch_gradients(gh_ctx* ctx, const conv_lanes::Lanes<float>& g, int waves, int tm, bool split, int blocks) {
  using namespace conv_wgrad_small;
  if ((waves == 8) != split || getenv("GORGONIA_HIP_CONV_APART")) return -1;   // tuning switch: a launch each
  switch (ctx->held.kind) {
    case kHeldSmall: return !split ? -1 : done(ctx, tm == 1 ? go_small<kWide, 1>(ctx, g, blocks) : go_small<kWide, 2>(ctx, g, blocks), tm, split);
    case kHeldSmallNarrow: return !split ? -1 : done(ctx, tm == 1 ? go_small<kNarrow, 1>(ctx, g, blocks) : go_small<kNarrow, 2>(ctx, g, blocks), tm, split);
    case kHeldF32:
      if (split) return done(ctx, tm == 1 ? go<float, 2, 4, 8, 1, 4, true>(ctx, g, blocks) : go<float, 2, 4, 8, 2, 4, true>(ctx, g, blocks), tm, split);
      return done(ctx, tm == 1 ? go<float, 2, 4, 4, 1, 4, false>(ctx, g, blocks) : go<float, 2, 4, 4, 2, 4, false>(ctx, g, blocks), tm, split);
  }
  return -1;
}

int gh_try_launch_gradients(gh_ctx* ctx, const conv_lanes::Lanes<double>& g, int waves, int tm, bool split, int blocks) {
  if (waves != 4 || tm != 1 || !split || getenv("GORGONIA_HIP_CONV_APART")) return -1;
  switch (ctx->held.kind) {
    case kHeldF64: return done(ctx, ctx->unpool.dz ? go<double, 1, 4, 4, 1, 2, true, true>(ctx, g, blocks) : go<double, 1, 4, 4, 1, 2, true>(ctx, g, blocks), tm, split);
    case kHeldF64Narrow: return done(ctx, ctx->unpool.dz ? go<double, 1, 2, 4, 1, 2, true, true>(ctx, g, blocks) : go<double, 1, 2, 4, 1, 2, true>(ctx, g, blocks), tm, split);
  }
  return -1;
}

// The filter gradient that no image gradient took along.
int gh_launch_held(gh_ctx* ctx) {
  if (ctx->held.kind == kHeldNone) return GH_OK;
  const int rc = ctx->held.kind == kHeldSmall || ctx->held.kind == kHeldSmallNarrow ? gh_launch_held_wgrad_small(ctx) : gh_launch_held_wgrad(ctx);
  ctx->held.kind = kHeldNone;
  return rc;
}

// Whether cmds[0] and cmds[1] are the two gradients of 3x3 convolutions, in either order, and neither meets the other's result.
// (The first command is a valid one.)
bool gh_gradient_pair(const gh_cmd* cmds, int n) {
  if (n < 2) return false;
  const uint32_t a = cmds[0].opcode, b = cmds[1].opcode;
  if (!(a == GH_OP_CONV2D_BWD_FILTER && b == GH_OP_CONV2D_BWD_DATA) && !(a == GH_OP_CONV2D_BWD_DATA && b == GH_OP_CONV2D_BWD_FILTER)) return false;
  std::string m;
  if (gh_validate_cmd(cmds[1], m) != GH_OK) return false;
  const gh_cmd &f = a == GH_OP_CONV2D_BWD_FILTER ? cmds[0] : cmds[1], &d = a == GH_OP_CONV2D_BWD_FILTER ? cmds[1] : cmds[0];
  if (f.dim[5] != 3 || f.dim[6] != 3 || d.dim[5] != 3 || d.dim[6] != 3 || gh_dtype_of(f.flags) != gh_dtype_of(d.flags)) return false;
  const int64_t item = gh_dtype_of(f.flags) == GH_F64 ? 8 : 4;
  auto x_of = [&](const gh_cmd& c) { return c.dim[0] * c.dim[1] * c.dim[2] * c.dim[3] * item; };
  auto w_of = [&](const gh_cmd& c) { return c.dim[4] * c.dim[1] * 9 * item; };
  auto y_of = [&](const gh_cmd& c) {
    return c.dim[0] * c.dim[4] * gh_conv_out(c.dim[2], 3, c.dim[7], c.dim[9], c.dim[11]) * gh_conv_out(c.dim[3], 3, c.dim[8], c.dim[10], c.dim[12]) * item;
  };
  const uint64_t dw = f.ptr[2], dx = d.ptr[2];
  return apart(dx, x_of(d), f.ptr[0], x_of(f)) && apart(dx, x_of(d), f.ptr[1], y_of(f)) && apart(dx, x_of(d), dw, w_of(f)) && apart(dw, w_of(f), d.ptr[0], y_of(d)) &&
         apart(dw, w_of(f), d.ptr[1], w_of(d));
}

// Whether the gradient of a 2x2 / 2 pooling, with its Rectify's, stands behind the two commands of gh_gradient_pair, takes the
// image gradient's result and lies apart from what the two touch: how many commands it is (float32 1: one command does both; float64
// 2), or 0.
int gh_unpool_follows(const gh_cmd* c, int n, gh_unpool* out) {
  if (n < 3 || c[2].opcode != GH_OP_MAXPOOL2D_BWD) return 0;
  const gh_cmd &f = c[0].opcode == GH_OP_CONV2D_BWD_FILTER ? c[0] : c[1], &d = c[0].opcode == GH_OP_CONV2D_BWD_FILTER ? c[1] : c[0], &p = c[2];
  const bool wide = gh_dtype_of(d.flags) == GH_F64;
  std::string m;
  if (gh_dtype_of(p.flags) != gh_dtype_of(d.flags) || p.ptr[1] != d.ptr[2] || gh_validate_cmd(p, m)) return 0;
  if ((p.flags & GH_FLAG_BN_REMADE) || !(p.flags & GH_FLAG_ACT_RELU) != wide) return 0;
  if (p.dim[0] != d.dim[0] || p.dim[1] != d.dim[1] || p.dim[2] != 2 * d.dim[2] || p.dim[3] != 2 * d.dim[3]) return 0;
  for (int i : {4, 5, 10, 11}) if (p.dim[i] != 2) return 0;
  for (int i : {6, 7, 8, 9}) if (p.dim[i] != 0) return 0;
  const int64_t item = wide ? 8 : 4, whole = p.dim[0] * p.dim[1] * p.dim[2] * p.dim[3] * item;
  *out = {p.ptr[0], p.ptr[0], p.ptr[2], p.ptr[2], false};
  if (wide) {
    if (n < 4 || c[3].opcode != GH_OP_RELU_BWD || gh_dtype_of(c[3].flags) != GH_F64 || c[3].ptr[1] != p.ptr[2] || c[3].dim[0] * item != whole || gh_validate_cmd(c[3], m)) return 0;
    out->z = c[3].ptr[0];
    out->dz = c[3].ptr[2];
    if (out->da != out->dz && !apart(out->da, whole, out->dz, whole)) return 0;
  }
  auto x_of = [&](const gh_cmd& k) { return k.dim[0] * k.dim[1] * k.dim[2] * k.dim[3] * item; };
  auto w_of = [&](const gh_cmd& k) { return k.dim[4] * k.dim[1] * 9 * item; };
  auto y_of = [&](const gh_cmd& k) {
    return k.dim[0] * k.dim[4] * gh_conv_out(k.dim[2], 3, k.dim[7], k.dim[9], k.dim[11]) * gh_conv_out(k.dim[3], 3, k.dim[8], k.dim[10], k.dim[12]) * item;
  };
  for (uint64_t to : {out->da, out->dz}) {
    if ((to & (uint64_t)(item - 1)) || !apart(to, whole, d.ptr[0], y_of(d)) || !apart(to, whole, d.ptr[1], w_of(d)) || !apart(to, whole, d.ptr[2], x_of(d)) ||
        !apart(to, whole, f.ptr[0], x_of(f)) || !apart(to, whole, f.ptr[1], y_of(f)) || !apart(to, whole, f.ptr[2], w_of(f)))
      return 0;
    for (uint64_t from : {out->a, out->z})
      if (!apart(to, whole, from, whole)) return 0;
  }
  for (uint64_t from : {out->a, out->z})
    if ((from & (uint64_t)(item - 1)) || !apart(from, whole, d.ptr[2], x_of(d)) || !apart(from, whole, f.ptr[2], w_of(f))) return 0;
  return wide ? 2 : 1;
}
