// Filter gradient of Conv2d 3x3 / stride 1 over small images (up to 16 x 16), float32, on the
// 16x16x4 MFMA.
//
// Replaces cuDNN ConvolutionBackwardFilter (ops/nn/convolution_cuda.go:182-189) for the layers
// whose images are small and many: dW[f][c][kr][kc] = sum over (image, output pixel) of
// dy[image][f][pixel] * x[image][c][pixel + tap].  As a GEMM that is M = filters,
// N = C * 9 in the reference's (c, kr, kc) order, K = B * oh * ow: a small result summed over
// a long K, so K is what gets divided among workgroups.
//
//   * One workgroup of eight wavefronts owns 64 filters x 16 channels (a 64 x 144 tile of dW:
//     wavefront w has filter rows 16 (w & 3) .. + 15, all nine 16-column tiles and one half
//     of every group's k steps; the two halves meet through LDS at the end, second onto
//     first, a fixed order) and a run of images.  Two wavefronts per SIMD: one's LDS and
//     issue latencies run under the other's MFMAs.  It takes the images a few at a time (as many as give about 200 output pixels):
//     their dy rows go to LDS as dyL[filter][k] with k = (image, pixel) and a pitch of 4 mod
//     64, so the 64 lanes of an A fetch hit 64 banks; their x planes go to LDS with a zero
//     halo, rows at a fixed pitch (18, or 10 for up to eight columns) and planes at a pitch of 4 mod 32.  The tile's 144
//     columns are taken tap-major: MFMA tile t is tap t and lane column c is channel c, so a
//     step's nine B fetches are one address - channel plane + the pixel position a table
//     gives for every k - plus nine compile-time offsets (tap row * pitch + tap column), and
//     the 64 lanes of each land in 64 banks.  Per step of four k: one A read, one table read,
//     one address add and nine B reads feed nine MFMAs.
//     Loads are 128 bits of what is contiguous, dy's 64 rows and x's 16 channels of an image, all of a group's in flight
//     before the first is stored: one memory latency to a group.
//   * The tile is accumulated in registers over all of the workgroup's images and stored
//     once, as slab `split` of the workspace; slabs are summed in slab order by the
//     reduction kernel the other filter-gradient kernels use, so results repeat bit for bit.
//     It is stored from LDS in the order of dW's rows, 128 bits a lane: straight from the registers, 36 bytes apart, every
//     store touched twenty lines.  us with the slab sum, with loads one value wide in four batches and those stores / now:
//     128 x 32 x 14 x 14 -> 64 28.4 / 26.0, 128 x 64 x 7 x 7 -> 128 24.7 / 22.2, 384 x 64 x 7 x 7 -> 128 64.9 / 52.6.
//     With enough (filter, channel) tiles to fill the device there is one slab and the tile
//     is stored straight into dW.
#include <algorithm>
#include <cstdlib>
#include <mutex>

#include "gh_conv_wgrad_small.h"

namespace {

using namespace conv_wgrad_small;

inline unsigned magic_of(unsigned d) { return d <= 1 ? 0u : (unsigned)((0x100000000ull + d - 1) / d); }

// Held to 128 registers: two workgroups then share a compute unit where their LDS allows (long K, few images).
template <int kRowPitch>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_conv3x3_wgrad_small(const gh_wgrad_small_args a) {
  extern __shared__ float lds[];
  workgroup<kRowPitch>(a.x, a.dy, a.out, a.g, a.slab, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, lds);
}

struct WgPlan {
  WgGeom g;
  int splits;
  size_t lds;
};

bool wgrad_small_plan(const gh_ctx* ctx, const gh_cmd& c, WgPlan* out) {
  if (gh_dtype_of(c.flags) != GH_F32) return false;
  const int64_t B = c.dim[0], C = c.dim[1], H = c.dim[2], W = c.dim[3], F = c.dim[4];
  const int64_t pad = c.dim[7];
  if (c.dim[5] != 3 || c.dim[6] != 3 || c.dim[9] != 1 || c.dim[10] != 1 || c.dim[11] != 1 || c.dim[12] != 1 ||
      c.dim[8] != pad || pad < 0 || pad > 1)
    return false;
  if (B < 1 || B > (1 << 20) || F < 16 || F > (1 << 16) || C < 16 || C % 16 != 0 || C > 4096 || H < 3 || W < 3 ||
      H > 16 || W > 16)
    return false;
  if (getenv("GORGONIA_HIP_WGRAD_NO_SMALL")) return false;   // tuning switch: the general kernel only
  WgGeom g{};
  g.B = (int)B; g.C = (int)C; g.H = (int)H; g.W = (int)W; g.F = (int)F; g.pad = (int)pad;
  g.oh = g.H + 2 * g.pad - 2; g.ow = g.W + 2 * g.pad - 2;
  if (g.oh <= 0 || g.ow <= 0 || g.oh * g.ow < 4) return false;   // a 128-bit piece of dy spans at most two rows
  g.npx = g.oh * g.ow;
  g.PW = g.W + 2 * g.pad; g.PH = g.H + 2 * g.pad;
  g.XP = g.PH * (g.PW <= kNarrow ? kNarrow : kWide);
  while (g.XP % 32 != 4) g.XP++;
  // images staged at a time: about 208 output pixels, fewer where their padded planes (tiny images
  // have more halo than pixels) would not fit LDS beside the dy rows
  constexpr size_t kLdsLimit = 150 * 1024;
  g.nb = g.npx >= 208 ? 1 : 208 / g.npx;
  if (g.nb > g.B) g.nb = g.B;
  for (;; g.nb--) {
    g.K = g.nb * g.npx; g.KW = (g.K + 3) & ~3;
    g.DP = g.KW + ((4 - g.KW % 64) + 64) % 64;
    if (g.nb == 1 || ((size_t)kBM * g.DP + (size_t)g.nb * kCT * g.XP + g.KW) * 4 <= kLdsLimit) break;
  }
  g.HW = g.H * g.W; g.CKK = g.C * 9;
  g.ngroups = (g.B + g.nb - 1) / g.nb;
  const int64_t tiles = (C / kCT) * ((F + kBM - 1) / kBM);
  // slabs: enough workgroups for two per compute unit, each with at least one image group
  int64_t splits = (2 * (int64_t)ctx->cu_count + tiles - 1) / tiles;
  if (splits > g.ngroups) splits = g.ngroups;
  if (splits < 1) splits = 1;
  g.gps = (int)((g.ngroups + splits - 1) / splits);
  splits = (g.ngroups + g.gps - 1) / g.gps;
  g.mNPX = magic_of(g.npx); g.mOW = magic_of(g.ow); g.mHW = magic_of(g.HW); g.mW = magic_of(g.W);
  g.mQIMG = magic_of(kBM * g.npx / 4); g.mQX = magic_of(kCT * g.HW / 4);
  out->g = g;
  out->splits = (int)splits;
  out->lds = ((size_t)kBM * g.DP + (size_t)g.nb * kCT * g.XP + g.KW) * 4;
  out->lds = std::max<size_t>(out->lds, (size_t)4 * 9 * 64 * 16);   // the two halves' partial tiles meet in it
  return out->lds <= kLdsLimit;
}

}  // namespace

// Whether the kernel takes the command: a function of its shape alone.
bool gh_conv_wgrad_small_takes(const gh_cmd& c) {
  gh_ctx probe;   // only its compute-unit count is read, for the slab count
  WgPlan p;
  return wgrad_small_plan(&probe, c, &p);
}

// Returns -1 when the shape is not one this kernel takes (or its slabs do not fit the
// workspace); otherwise the partial sums are at *slabs, *splits slabs of F x C*9
// (or, with *splits == 1, dW is complete).
int gh_try_launch_conv_wgrad_small(gh_ctx* ctx, const gh_cmd& c, int* splits, float** slabs) {
  WgPlan p;
  if (!wgrad_small_plan(ctx, c, &p)) return -1;
  const int64_t slab = (int64_t)p.g.F * p.g.CKK;
  if (p.splits > 1 && slab * 4 * p.splits > ctx->workspace_bytes) {
    // fewer, longer runs of images: as many slabs as the workspace holds
    if (int rc = gh_ws_short(ctx, slab * 4 * p.splits)) return rc;
    const int64_t fit = std::max<int64_t>(1, ctx->workspace_bytes / (slab * 4));
    p.g.gps = (int)((p.g.ngroups + fit - 1) / fit);
    p.splits = (p.g.ngroups + p.g.gps - 1) / p.g.gps;
  }
  static std::once_flag once;
  static hipError_t attr_rc = hipSuccess;
  std::call_once(once, [] {
    for (const void* k : {(const void*)k_conv3x3_wgrad_small<kWide>, (const void*)k_conv3x3_wgrad_small<kNarrow>})
      if (attr_rc == hipSuccess) attr_rc = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  });
  if (attr_rc != hipSuccess) return gh_check_hip(ctx, attr_rc, "hipFuncSetAttribute(conv3x3 wgrad small)");
  float* const dst = p.splits > 1 ? (float*)gh_slab_space(ctx, slab * 4 * p.splits) : (float*)(uintptr_t)c.ptr[2];
  *slabs = dst;
  const dim3 grid((unsigned)p.splits, (unsigned)(p.g.C / kCT), (unsigned)((p.g.F + kBM - 1) / kBM));
  const gh_wgrad_small_args a{(const float*)(uintptr_t)c.ptr[0], (const float*)(uintptr_t)c.ptr[1], dst, p.g, slab};
  *splits = p.splits;
  if (gh_may_hold(ctx, dst)) {
    static_assert(sizeof(a) <= sizeof(ctx->held.args), "the argument fits");
    ctx->held.kind = p.g.PW <= kNarrow ? kHeldSmallNarrow : kHeldSmall;
    ctx->held.grid = grid;
    ctx->held.lds = p.lds;
    memcpy(ctx->held.args, &a, sizeof(a));
    return GH_OK;
  }
  hipLaunchKernelGGL((p.g.PW <= kNarrow ? k_conv3x3_wgrad_small<kNarrow> : k_conv3x3_wgrad_small<kWide>), grid, dim3(kThreads), p.lds, ctx->stream, a);
  return gh_check_hip(ctx, hipGetLastError(), "conv3x3 wgrad small launch");
}

int gh_launch_held_wgrad_small(gh_ctx* ctx) {
  gh_wgrad_small_args a;
  memcpy(&a, ctx->held.args, sizeof(a));
  hipLaunchKernelGGL((a.g.PW <= kNarrow ? k_conv3x3_wgrad_small<kNarrow> : k_conv3x3_wgrad_small<kWide>), ctx->held.grid, dim3(kThreads), ctx->held.lds, ctx->stream, a);
  return gh_check_hip(ctx, hipGetLastError(), "conv3x3 wgrad small launch");
}
