// A dense layer's weight gradient and its input gradient in one launch.
//
// x transposed times dy and dy times w transposed read the same dy and neither reads what the other writes.  In a training step
// both are small: a launch each is 4 to 10 us, most of it the way from the first load to the last store.  Here the workgroups
// of the one stand in the grid behind those of the other, and run while those wait.  They are the workgroups of the kernels the
// two products have alone (gh_gemm_direct.h, gh_gemm_skinny.h), chosen by gh_choose_gemm as gh_launch_gemm chooses: the
// stored bits are theirs.
//
// Bound: the latency of the longer product, and its matrix instructions where it fills the device.  us apart / together (batch x
// inputs -> outputs): float32 128 x 1152 -> 625 16.0 / 11.6, 128 x 625 -> 10 6.8 / 4.6, 64 x 300 -> 100 6.0 / 2.9; float64 50 x 1152 -> 625
// 14.2 / 11.0, 50 x 625 -> 10 6.3 / 3.6.  Of 207 drawn pairs of 2 to 512 rows and 4 to 4096 inputs and outputs the 150 that have a kernel
// here took 0.65 of their time, none more than before.  The input gradient stands first, whose contraction is the longer one
// (float32 257 x 54 -> 1536 8.5 us, behind the weight gradient 10.3; float64 51 x 778 -> 2019 19.5 and 29.3), but where float64's weight
// gradient has a compute unit for each of its workgroups: all begin at once, and its larger tiles take longer (50 x 1152 -> 625 12.1 us
// behind the input gradient, 96 x 1152 -> 625 15.0 and 13.3 in front of it).  A float64 weight gradient in eight slices (640 rows and
// more) has its four-wavefront input gradient beside it in workgroups of eight: 1448 x 96 -> 1582 38.6 with four / 37.3, 2035 x 129 ->
// 1529 76.1 / 70.8, but 930 x 142 -> 1859 41.3 / 44.1 and 1610 x 120 -> 1605 35.9 / 37.3; the bits are those of the product alone.
//
// The gradient of the Rectify in front of the layer, which takes the input gradient value by value, is done where that is stored: a
// training step of the example's network 178.5 / 176.2 us at 128 images, 405.9 / 403.5 at 384, float64 at fifty 177.3 / 175.4.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "gh_gemm_direct.h"
#include "gh_gemm_skinny.h"

namespace {

template <class T, int TM, int TN, bool kSplitK, bool kTA, int WV = 4>
struct Direct {
  static constexpr bool kDirect = true;
  static constexpr int kWaves = WV, kLds = gemm_direct::lds_of<T, kWaves, TN, kSplitK>();
  gemm_direct::Gemm<T> g;
  gh_rectify_behind<T> behind;
  int gx, gy;
  explicit Direct(const gh_cmd& c) {
    constexpr int rows = 16 * TM * (kSplitK ? 1 : kWaves);
    int batch;
    g = gemm_direct::gemm_of<T>(c, &batch);
    gx = (g.N + 16 * TN - 1) / (16 * TN);
    gy = (g.M + rows - 1) / rows;
  }
  int all() const { return gx * gy; }
  __device__ __forceinline__ void run(int id, char* lds) const { gemm_direct::workgroup<T, kWaves, TM, TN, kSplitK, kTA, !kTA, !kTA>(g, id, gx, gy, 0, lds, behind); }
};

template <int WV, int NT, bool kTA>
struct Skinny32 {
  static constexpr bool kDirect = false;
  static constexpr int kWaves = WV, kLds = gemm_skinny::lds16<WV, NT>();
  gemm_skinny::Args32 g;
  gh_rectify_behind<float> behind;
  int gx, gy;
  explicit Skinny32(const gh_cmd& c) : g(gemm_skinny::args32_of(c)), gx((g.N + 16 * NT - 1) / (16 * NT)), gy((g.M + 15) / 16) {}
  int all() const { return gx * gy; }
  __device__ __forceinline__ void run(int id, char* lds) const { gemm_skinny::workgroup16<WV, NT, kTA, !kTA, true, false, !kTA>(g, id, gx, gy, 0, 1, lds, {}, behind); }
};

template <int WV, bool kTA>
struct Skinny64 {
  static constexpr int kWaves = WV, kLds = gemm_skinny::lds64<WV>();
  gemm_skinny::Args64 g;
  gh_rectify_behind<double> behind;
  int gx, gy;
  explicit Skinny64(const gh_cmd& c) : g(gemm_skinny::args64_of(c)), gx((g.N + 15) / 16), gy((g.M + 15) / 16) {}
  int all() const { return gx * gy; }
  __device__ __forceinline__ void run(int id, char* lds) const {
    const int by = id / gx;
    gemm_skinny::workgroup64<WV, !kTA, !kTA, !kTA>(g, id - by * gx, by, 0, lds, behind);
  }
};

// (A workgroup of which the product has fewer wavefronts than the launch uses the first of them.)
template <class P, class Q>
constexpr int waves_of() { return P::kWaves > Q::kWaves ? P::kWaves : Q::kWaves; }

template <class P, class Q>
__global__ __launch_bounds__((waves_of<P, Q>() * 64)) __attribute__((amdgpu_waves_per_eu((waves_of<P, Q>() == 16 ? 4 : 2)))) void k_gemm_gradients(const P p, const Q q, const int first) {
  __shared__ __attribute__((aligned(16))) char lds[P::kLds > Q::kLds ? P::kLds : Q::kLds];
  const int b = (int)blockIdx.x;
  if (b < first) {
    if (P::kWaves < waves_of<P, Q>() && (int)threadIdx.x >= P::kWaves * 64) return;
    p.run(b, lds);
  } else {
    if (Q::kWaves < waves_of<P, Q>() && (int)threadIdx.x >= Q::kWaves * 64) return;
    q.run(b - first, lds);
  }
}

template <class P, class Q>
int go(gh_ctx* ctx, const P& p, const Q& q) {
  if ((int64_t)p.all() + q.all() > (1 << 20)) return -1;
  hipLaunchKernelGGL((k_gemm_gradients<P, Q>), dim3((unsigned)(p.all() + q.all())), dim3(waves_of<P, Q>() * 64), 0, ctx->stream, p, q, p.all());
  return gh_check_hip(ctx, hipGetLastError(), "dense gradients launch");
}

// Calls body(product) with the workgroups of a choice, or returns -1.  (kSplit: fewer rows than the small-output kernel takes, so
// that the weight gradient, whose contraction they are, is one of the first two.)
template <bool kTA, bool kSplit, class Body>
int with32(const gh_gemm_choice& k, const gh_cmd& c, Body&& body) {
  if (k.kind == kGemmDirect) {
    if (k.form == 4) return body(Direct<float, 1, 4, false, kTA>(c));
    if (k.form == 5) return body(Direct<float, 2, 4, false, kTA>(c));
    if constexpr (!kTA && kSplit)
      if (k.form == 0 && k.waves == 8) return body(Direct<float, 2, 4, true, kTA, 8>(c));
  } else if (k.kind == kGemmSkinny) {
    if (k.waves == 8) return k.columns == 1 ? body(Skinny32<8, 1, kTA>(c)) : body(Skinny32<8, 2, kTA>(c));
    if constexpr (!kTA) return k.columns == 1 ? body(Skinny32<16, 1, kTA>(c)) : body(Skinny32<16, 2, kTA>(c));
  }
  return -1;
}

template <int WV, bool kTA, class Body>
int direct64(int form, const gh_cmd& c, Body&& body) {
  if (form == 0) return body(Direct<double, 2, 2, true, kTA, WV>(c));
  if constexpr (kTA) {
    switch (form) {
      case 1: return body(Direct<double, 2, 4, true, kTA, WV>(c));
      case 2: return body(Direct<double, 3, 4, true, kTA, WV>(c));
      case 3: return body(Direct<double, 4, 4, true, kTA, WV>(c));
      case 4: return body(Direct<double, 5, 4, true, kTA, WV>(c));
    }
  }
  return -1;
}

template <bool kTA, class Body>
int with64(const gh_gemm_choice& k, const gh_cmd& c, Body&& body) {
  if (k.kind == kGemmDirect) {
    if (k.waves != 8) return direct64<4, kTA>(k.form, c, body);
    if constexpr (kTA) return direct64<8, kTA>(k.form, c, body);
  }
  if (k.kind == kGemmSkinny) {
    if (k.waves == 4) return body(Skinny64<4, kTA>(c));
    if constexpr (!kTA) return body(Skinny64<8, kTA>(c));
  }
  return -1;
}

struct Span { uint64_t at; int64_t bytes; };
bool apart(const Span& a, const Span& b) { return a.at + (uint64_t)a.bytes <= b.at || b.at + (uint64_t)b.bytes <= a.at; }

}  // namespace

int gh_try_launch_gemm_gradients(gh_ctx* ctx, const gh_cmd* cmds, bool rectified) {
  if (getenv("GORGONIA_HIP_GEMM_APART")) return -1;   // tuning switch: a launch each
  const int w = (cmds[0].flags & GH_FLAG_TRANS_A) ? 0 : 1;
  const gh_cmd &dw = cmds[w], &dx = cmds[1 - w];
  const gh_gemm_choice kw = gh_choose_gemm(ctx, dw);
  if (kw.kind == kGemmOther) return -1;
  const gh_gemm_choice kx = gh_choose_gemm(ctx, dx);
  if (kx.kind == kGemmOther) return -1;
  int rc;
  // the input gradient's, with the Rectify's gradient where that rides along
  auto behind = [&](auto q) {
    if (rectified) q.behind = {(decltype(q.behind.z))(uintptr_t)cmds[2].ptr[0], (decltype(q.behind.out))(uintptr_t)cmds[2].ptr[2]};
    return q;
  };
  if (gh_dtype_of(dw.flags) == GH_F64)
    rc = with64<true>(kw, dw, [&](const auto& p) {
      return with64<false>(kx, dx, [&](const auto& plain) { const auto q = behind(plain); return p.all() <= ctx->cu_count ? go(ctx, p, q) : go(ctx, q, p); });
    });
  else
    rc = with32<true, false>(kw, dw, [&](const auto& p) {
      constexpr bool kDirect = std::decay_t<decltype(p)>::kDirect;
      return with32<false, kDirect>(kx, dx, [&](const auto& q) { return go(ctx, behind(q), p); });
    });
  if (rc != GH_OK) return rc;
  for (int k = 0; k < 2 + rectified; k++)
    for (uint64_t p : cmds[k].ptr) ctx->llc.touch(p, 0, false);
  if (rectified) {
    ctx->joint[GH_JOINT_RECTIFIED].launches++;
    ctx->joint[GH_JOINT_RECTIFIED].form = 0;
  }
  auto& j = ctx->joint[GH_JOINT_DENSE_GRADIENTS];
  j.launches++;
  auto digits = [](const gh_gemm_choice& k) { return 10000 * k.kind + 1000 * k.form + 10 * k.waves + k.columns; };
  j.form = (int64_t)100000 * digits(kw) + digits(kx);
  return GH_OK;
}

// Whether cmds[0] and cmds[1] are products of one size of float with the left operand of the one and the right operand of
// the other a transposed view, nothing behind them, and neither's result in what the other reads or writes.  (The first
// command is a valid one.)
bool gh_gemm_gradient_pair(const gh_cmd* cmds, int n) {
  if (n < 2 || cmds[0].opcode != GH_OP_GEMM || cmds[1].opcode != GH_OP_GEMM) return false;
  const uint32_t both = GH_FLAG_TRANS_A | GH_FLAG_TRANS_B, plain = both | GH_FLAG_DTYPE(0xf), a = cmds[0].flags & both, b = cmds[1].flags & both;
  if ((a ^ b) != both || a == both || b == both || ((cmds[0].flags | cmds[1].flags) & ~plain) || gh_dtype_of(cmds[0].flags) != gh_dtype_of(cmds[1].flags)) return false;
  std::string m;
  if (gh_validate_cmd(cmds[1], m) != GH_OK) return false;
  const int64_t item = gh_dtype_of(cmds[0].flags) == GH_F64 ? 8 : 4;
  Span at[2][3];
  for (int i = 0; i < 2; i++) {
    const gh_cmd& c = cmds[i];
    if (c.dim[6] > 1 || std::max({c.dim[0], c.dim[1], c.dim[2], c.dim[3], c.dim[4], c.dim[5]}) >= (int64_t)1 << 24) return false;   // (spans in 64 bits)
    auto span = [&](int p, int64_t rows, int64_t cols, int64_t ld) { at[i][p] = {c.ptr[p], ((rows - 1) * ld + cols) * item}; };
    const bool ta = c.flags & GH_FLAG_TRANS_A;
    span(0, ta ? c.dim[2] : c.dim[0], ta ? c.dim[0] : c.dim[2], c.dim[3]);
    span(1, ta ? c.dim[2] : c.dim[1], ta ? c.dim[1] : c.dim[2], c.dim[4]);
    span(2, c.dim[0], c.dim[1], c.dim[5]);
  }
  return apart(at[0][2], at[1][0]) && apart(at[0][2], at[1][1]) && apart(at[0][2], at[1][2]) && apart(at[1][2], at[0][0]) && apart(at[1][2], at[0][1]);
}

// Whether behind the two commands of gh_gemm_gradient_pair stands the gradient of a Rectify, of what the input gradient writes, into
// the same memory or into memory that lies apart from all that the two touch.
bool gh_rectify_gradient_follows(const gh_cmd* c, int n) {
  if (n < 3 || c[2].opcode != GH_OP_RELU_BWD) return false;
  const gh_cmd &dx = (c[0].flags & GH_FLAG_TRANS_A) ? c[1] : c[0], &r = c[2];
  std::string m;
  if (gh_dtype_of(r.flags) != gh_dtype_of(dx.flags) || r.ptr[1] != dx.ptr[2] || dx.dim[5] != dx.dim[1] || r.dim[0] != dx.dim[0] * dx.dim[1] || gh_validate_cmd(r, m)) return false;
  const int64_t item = gh_dtype_of(dx.flags) == GH_F64 ? 8 : 4;
  if ((r.ptr[0] | r.ptr[2]) & (uint64_t)(item - 1)) return false;
  const Span z = {r.ptr[0], r.dim[0] * item}, out = {r.ptr[2], r.dim[0] * item};
  if (!apart(z, out)) return false;
  for (int i = 0; i < 2; i++) {
    const gh_cmd& p = c[i];
    const bool ta = p.flags & GH_FLAG_TRANS_A;
    auto span = [&](int k, int64_t rows, int64_t cols, int64_t ld) { return Span{p.ptr[k], ((rows - 1) * ld + cols) * item}; };
    const Span a = span(0, ta ? p.dim[2] : p.dim[0], ta ? p.dim[0] : p.dim[2], p.dim[3]), b = span(1, ta ? p.dim[2] : p.dim[1], ta ? p.dim[1] : p.dim[2], p.dim[4]),
               y = span(2, p.dim[0], p.dim[1], p.dim[5]);
    if (!apart(z, y) || !apart(out, a) || !apart(out, b) || (!(&p == &dx && out.at == y.at) && !apart(out, y))) return false;
  }
  return true;
}
