// Two commands in one launch.
//
// Where a command reads what the one in front of it wrote, value by value, the second costs a launch (about 2.5 us) and a
// pass over memory to read the value again.  gh_submit gives such a pair to a kernel of this file: the tensors both
// commands write are written, with the arithmetic of their own kernels, so the stored bits are theirs.
//
//   * float64 Rectify and the 2x2 pooling behind it (training keeps the rectified tensor): a thread per window.
//   * float64 gradient of that pooling and the Rectify gradient behind it, in place or not.
//   * a tensor times a scalar and the SoftMax gradient that takes it as dy: a wavefront per row.
//
//   * a SoftMax in front of these two, of up to 64 columns: the row's values stay in the wavefront's registers.  (A product
//     with its SoftMax in front of them: k_gemm.hip.)
//
// Bound: HBM for large tensors, the launch for small ones.  us, apart / as a pair: Rectify and pooling of 50 x 32 x 28 x 28
// 10.5 / 4.2 (3.7 TB/s from the caches), of 128 images 18.3 / 9.8 (5.9 TB/s); the gradients 14.5 / 4.6 and 22.6 / 13.1; a
// float64 training step of the example's network at batch 50 253 / 225.  50 x 10, scaled and SoftMax gradient 5.3 / 3.1,
// float32 128 x 10 6.0 / 3.2.
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "gh_internal.h"

namespace {

constexpr int kBlock = 256;

template <class T>
__device__ __forceinline__ T relu_of(T x) { return x * (x >= (T)0 ? (T)1 : (T)0); }

// A window's four values and, of the last column's and row's windows, what an odd extent leaves outside every window.
template <bool VEC>
struct Windows {
  typedef double V2 __attribute__((ext_vector_type(2)));
  int H, W;
  int64_t at;
  bool right, below;
  __device__ __forceinline__ Windows(int H_, int W_, int64_t idx) : H(H_), W(W_) {
    const int oh = H / 2, ow = W / 2;
    const int64_t row = idx / ow;
    const int pw = (int)(idx - row * ow);
    const int64_t bc = row / oh;
    const int ph = (int)(row - bc * oh);
    at = (bc * H + 2 * ph) * (int64_t)W + 2 * pw;
    right = (W & 1) && pw == ow - 1;
    below = (H & 1) && ph == oh - 1;
  }
  __device__ __forceinline__ void load(const double* x, V2& r0, V2& r1) const {
    if constexpr (VEC) {
      r0 = *(const V2*)(x + at);
      r1 = *(const V2*)(x + at + W);
    } else {
      r0 = V2{x[at], x[at + 1]};
      r1 = V2{x[at + W], x[at + W + 1]};
    }
  }
  __device__ __forceinline__ void store(double* y, V2 r0, V2 r1) const {
    if constexpr (VEC) {
      *(V2*)(y + at) = r0;
      *(V2*)(y + at + W) = r1;
    } else {
      y[at] = r0[0]; y[at + 1] = r0[1];
      y[at + W] = r1[0]; y[at + W + 1] = r1[1];
    }
  }
  template <class F>
  __device__ __forceinline__ void outside(F&& f) const {   // the elements past the last windows
    if (right) { f(at + 2); f(at + W + 2); }
    if (below) {
      f(at + 2 * (int64_t)W);
      f(at + 2 * (int64_t)W + 1);
      if (right) f(at + 2 * (int64_t)W + 2);
    }
  }
};

// scan order and strict > of the pooling kernels: the window's maximum and its place, -1 where nothing is above -DBL_MAX
template <class V2>
__device__ __forceinline__ int scan(V2 r0, V2 r1, double* best) {
  int arg = -1;
  *best = -DBL_MAX;
  if (r0[0] > *best) { *best = r0[0]; arg = 0; }
  if (r0[1] > *best) { *best = r0[1]; arg = 1; }
  if (r1[0] > *best) { *best = r1[0]; arg = 2; }
  if (r1[1] > *best) { *best = r1[1]; arg = 3; }
  return arg;
}

// (x and a may be one tensor: every element is read and written by one thread)
template <bool VEC>
__global__ __launch_bounds__(kBlock) void k_relu_pool_f64(const double* x, double* a, double* __restrict__ p, int H, int W, int64_t windows) {
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < windows; i += stride) {
    const Windows<VEC> w(H, W, i);
    typename Windows<VEC>::V2 r0, r1;
    w.load(x, r0, r1);
#pragma unroll
    for (int e = 0; e < 2; e++) { r0[e] = relu_of(r0[e]); r1[e] = relu_of(r1[e]); }
    w.store(a, r0, r1);
    w.outside([&](int64_t o) { a[o] = relu_of(x[o]); });
    double best;
    scan(r0, r1, &best);
    p[i] = best;
  }
}

// da, the pooling's gradient, is stored where it is not the tensor that the Rectify gradient overwrites
template <bool VEC>
__global__ __launch_bounds__(kBlock) void k_pool_relu_bwd_f64(const double* __restrict__ a, const double* __restrict__ dy, const double* __restrict__ z,
                                                              double* da, double* dz, int H, int W, int64_t windows) {
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  const bool both = da != dz;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < windows; i += stride) {
    const Windows<VEC> w(H, W, i);
    typename Windows<VEC>::V2 r0, r1, z0, z1;
    w.load(a, r0, r1);
    w.load(z, z0, z1);
    double best;
    const int arg = scan(r0, r1, &best);
    const double v = 0.0 + dy[i];
    r0[0] = arg == 0 ? v : 0.0; r0[1] = arg == 1 ? v : 0.0;
    r1[0] = arg == 2 ? v : 0.0; r1[1] = arg == 3 ? v : 0.0;
    if (both) w.store(da, r0, r1);
#pragma unroll
    for (int e = 0; e < 2; e++) { r0[e] = r0[e] * (z0[e] >= 0.0 ? 1.0 : 0.0); r1[e] = r1[e] * (z1[e] >= 0.0 ? 1.0 : 0.0); }
    w.store(dz, r0, r1);
    w.outside([&](int64_t o) {
      if (both) da[o] = 0.0;
      dz[o] = 0.0 * (z[o] >= 0.0 ? 1.0 : 0.0);
    });
  }
}

// g = x s; dx = y (g - sum of g y), the sum in column order.  (x and g may be one tensor.)
template <class T>
__global__ __launch_bounds__(kBlock) void k_scale_softmax_bwd(const T* x, const T* __restrict__ s, T* g, const T* __restrict__ y, T* __restrict__ dx,
                                                              int64_t rows, int cols) {
  const int lane = (int)threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T scale = *s;
  const int64_t at = row * cols;
  T dot = (T)0;
  for (int j0 = 0; j0 < cols; j0 += 64) {
    const int j = j0 + lane;
    T p = (T)0;
    if (j < cols) {
      const T v = x[at + j] * scale;
      g[at + j] = v;
      p = v * y[at + j];
    }
    const int lim = min(64, cols - j0);
    for (int l = 0; l < lim; l++) dot = dot + __shfl(p, l, 64);
  }
  for (int j = lane; j < cols; j += 64) {   // (read back by the lane that wrote it)
    const T t = g[at + j] - dot;
    dx[at + j] = y[at + j] * t;
  }
}

// y = SoftMax(z), g = x s and dx of y and g, with the arithmetic of k_softmax, k_softmax_f64 and the kernel above.  (x and g
// may be one tensor, and z any of those written: a wavefront reads a row before it writes it.)
template <class T>
__global__ __launch_bounds__(kBlock) void k_softmax_gradient(const T* z, T* y, const gh_softmax_gradient<T> t, int64_t rows, int cols) {
  const int lane = (int)threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int64_t at = row * cols + lane;
  const bool there = lane < cols;
  const T v = there ? z[at] : (T)-INFINITY, scaled = there ? t.x[at] * *t.s : (T)0;
  T mx = there ? fmax((T)-INFINITY, v) : (T)-INFINITY;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
  const T e = there ? (T)exp((double)(v - mx)) : (T)0;
  T sum = (T)0;
  for (int l = 0; l < cols; l++) sum = sum + __shfl(e, l, 64);
  T mine;
  if constexpr (sizeof(T) == 8) {
    mine = e / sum;
  } else {
    const T inv = 1.0f / sum;
    mine = e * inv;
  }
  const T p = scaled * mine;
  T dot = (T)0;
  for (int l = 0; l < cols; l++) dot = dot + __shfl(p, l, 64);
  if (!there) return;
  y[at] = mine;
  t.g[at] = scaled;
  const T d = scaled - dot;
  t.dx[at] = mine * d;
}

// ---- which commands ---------------------------------------------------------------------

enum { kNone, kReluPool, kPoolReluBwd, kScaleSoftmaxBwd };

bool apart(uint64_t p, int64_t bytes, uint64_t q, int64_t other) { return p + (uint64_t)bytes <= q || q + (uint64_t)other <= p; }

// a float64 2x2 / stride-2 pooling (or its gradient) without padding that reads its input as it is
bool pools(const gh_cmd& c) {
  if (gh_dtype_of(c.flags) != GH_F64 || (c.flags & GH_FLAG_ACT_RELU)) return false;
  for (int i : {4, 5, 10, 11}) if (c.dim[i] != 2) return false;
  for (int i : {6, 7, 8, 9}) if (c.dim[i] != 0) return false;
  return c.dim[0] > 0 && c.dim[1] > 0 && c.dim[2] >= 2 && c.dim[3] >= 2;
}

// Every tensor that the pair writes has to lie apart from all others it touches (or be exactly the one it may overwrite): a
// thread reads its elements when other threads have written theirs.
int kind_of(const gh_cmd* c) {
  const gh_cmd &f = c[0], &s = c[1];
  if (gh_dtype_of(f.flags) != gh_dtype_of(s.flags)) return kNone;
  if (f.opcode == GH_OP_RELU && s.opcode == GH_OP_MAXPOOL2D) {
    if (!pools(s) || s.ptr[0] != f.ptr[1] || ((f.ptr[0] | f.ptr[1] | s.ptr[1]) & 7)) return kNone;
    const int64_t whole = s.dim[0] * s.dim[1] * s.dim[2] * s.dim[3] * 8, pooled = s.dim[0] * s.dim[1] * (s.dim[2] / 2) * (s.dim[3] / 2) * 8;
    if (f.dim[0] * 8 != whole) return kNone;
    const bool ok = (f.ptr[0] == f.ptr[1] || apart(f.ptr[0], whole, f.ptr[1], whole)) && apart(s.ptr[1], pooled, f.ptr[0], whole) && apart(s.ptr[1], pooled, f.ptr[1], whole);
    return ok ? kReluPool : kNone;
  }
  if (f.opcode == GH_OP_MAXPOOL2D_BWD && s.opcode == GH_OP_RELU_BWD) {
    if (!pools(f) || s.ptr[1] != f.ptr[2] || ((f.ptr[0] | f.ptr[1] | f.ptr[2] | s.ptr[0] | s.ptr[2]) & 7)) return kNone;
    const int64_t whole = f.dim[0] * f.dim[1] * f.dim[2] * f.dim[3] * 8, pooled = f.dim[0] * f.dim[1] * (f.dim[2] / 2) * (f.dim[3] / 2) * 8;
    if (s.dim[0] * 8 != whole) return kNone;
    for (uint64_t out : {f.ptr[2], s.ptr[2]})
      if (!apart(out, whole, f.ptr[0], whole) || !apart(out, whole, f.ptr[1], pooled) || !apart(out, whole, s.ptr[0], whole)) return kNone;
    return s.ptr[2] == f.ptr[2] || apart(s.ptr[2], whole, f.ptr[2], whole) ? kPoolReluBwd : kNone;
  }
  if (f.opcode == GH_OP_ELEM_BIN && s.opcode == GH_OP_SOFTMAX_BWD) {
    const int64_t item = gh_dtype_of(f.flags) == GH_F64 ? 8 : 4;
    if (gh_dtype_of(f.flags) > GH_F64 || gh_fn(f.flags) != GH_MUL || gh_mode(f.flags) != GH_VS || s.dim[0] <= 0 || s.dim[1] <= 0) return kNone;
    const uint64_t g = f.ptr[2] ? f.ptr[2] : f.ptr[0];
    const int64_t bytes = s.dim[0] * s.dim[1] * item;
    if (s.ptr[1] != g || f.dim[0] * item != bytes || s.dim[0] > INT32_MAX || ((f.ptr[0] | f.ptr[1] | g | s.ptr[0] | s.ptr[2]) & (uint64_t)(item - 1))) return kNone;
    const bool ok = (g == f.ptr[0] || apart(g, bytes, f.ptr[0], bytes)) && apart(g, bytes, f.ptr[1], item) && apart(g, bytes, s.ptr[0], bytes) &&
                    apart(s.ptr[2], bytes, g, bytes) && apart(s.ptr[2], bytes, f.ptr[0], bytes) && apart(s.ptr[2], bytes, f.ptr[1], item) && apart(s.ptr[2], bytes, s.ptr[0], bytes);
    return ok ? kScaleSoftmaxBwd : kNone;
  }
  return kNone;
}

template <class T> T* at(uint64_t p) { return (T*)(uintptr_t)p; }

}  // namespace

// (the first command is a valid one; the second is looked at only where its opcode makes it a candidate)
bool gh_is_pair(const gh_cmd* cmds, int n) {
  if (n < 2) return false;
  const uint32_t a = cmds[0].opcode, b = cmds[1].opcode;
  if (!(a == GH_OP_RELU && b == GH_OP_MAXPOOL2D) && !(a == GH_OP_MAXPOOL2D_BWD && b == GH_OP_RELU_BWD) && !(a == GH_OP_ELEM_BIN && b == GH_OP_SOFTMAX_BWD)) return false;
  std::string m;
  return gh_validate_cmd(cmds[1], m) == GH_OK && kind_of(cmds) != kNone;
}

// A SOFTMAX, or a GEMM with one: the two commands behind it take its result, and write nothing that it or another row's
// workgroup reads.
bool gh_softmax_gradient_follows(const gh_cmd* c, int n) {
  if (n < 3 || c[1].opcode != GH_OP_ELEM_BIN || c[2].opcode != GH_OP_SOFTMAX_BWD) return false;
  const bool product = c[0].opcode == GH_OP_GEMM;
  if (product ? !(c[0].flags & GH_FLAG_GEMM_SOFTMAX) || c[0].dim[6] > 1 || c[0].dim[5] != c[0].dim[1] : c[0].opcode != GH_OP_SOFTMAX) return false;
  std::string m;
  if (gh_dtype_of(c[0].flags) != gh_dtype_of(c[1].flags) || gh_validate_cmd(c[1], m) || gh_validate_cmd(c[2], m) || kind_of(c + 1) != kScaleSoftmaxBwd) return false;
  const gh_cmd &f = c[1], &s = c[2];
  const int64_t item = gh_dtype_of(f.flags) == GH_F64 ? 8 : 4, bytes = s.dim[0] * s.dim[1] * item;
  const uint64_t y = c[0].ptr[product ? 2 : 1], g = f.ptr[2] ? f.ptr[2] : f.ptr[0], dx = s.ptr[2];
  if (s.ptr[0] != y || s.dim[0] != c[0].dim[0] || s.dim[1] != c[0].dim[1]) return false;
  if (!apart(y, bytes, f.ptr[0], bytes) || !apart(y, bytes, f.ptr[1], item)) return false;
  if (!product) {
    const uint64_t z = c[0].ptr[0];
    for (uint64_t out : {y, g, dx})
      if (out != z && !apart(out, bytes, z, bytes)) return false;
    return (z & (uint64_t)(item - 1)) == 0;
  }
  const int64_t rows = c[0].dim[0], cols = c[0].dim[1], depth = c[0].dim[2];
  for (uint64_t out : {g, dx})
    if (!apart(out, bytes, c[0].ptr[0], ((rows - 1) * c[0].dim[3] + depth) * item) || !apart(out, bytes, c[0].ptr[1], ((depth - 1) * c[0].dim[4] + cols) * item) ||
        ((c[0].flags & GH_FLAG_GEMM_BIAS) && !apart(out, bytes, c[0].ptr[3], cols * item)))
      return false;
  return true;
}

int gh_try_launch_softmax_gradient(gh_ctx* ctx, const gh_cmd* c) {
  const int64_t rows = c[0].dim[0];
  const int cols = (int)c[0].dim[1];
  if (c[0].dim[1] > 64) return -1;
  for (int k = 0; k < 3; k++)
    for (uint64_t p : c[k].ptr) ctx->llc.touch(p, 0, false);
  auto go = [&](auto* zero) {
    typedef std::remove_pointer_t<decltype(zero)> T;
    const gh_softmax_gradient<T> t = {at<const T>(c[1].ptr[0]), at<const T>(c[1].ptr[1]), at<T>(c[1].ptr[2] ? c[1].ptr[2] : c[1].ptr[0]), at<T>(c[2].ptr[2])};
    hipLaunchKernelGGL(k_softmax_gradient<T>, dim3((unsigned)((rows + kBlock / 64 - 1) / (kBlock / 64))), dim3(kBlock), 0, ctx->stream, at<const T>(c[0].ptr[0]),
                       at<T>(c[0].ptr[1]), t, rows, cols);
  };
  if (gh_dtype_of(c[0].flags) == GH_F64) go((double*)nullptr);
  else go((float*)nullptr);
  ctx->joint[GH_JOINT_SOFTMAX_GRADIENT].launches++;
  ctx->joint[GH_JOINT_SOFTMAX_GRADIENT].form = 1;
  return gh_check_hip(ctx, hipGetLastError(), "softmax and its gradient launch");
}

int gh_launch_pair(gh_ctx* ctx, const gh_cmd* c) {
  const gh_cmd &f = c[0], &s = c[1];
  for (int k = 0; k < 2; k++)
    for (uint64_t p : c[k].ptr) ctx->llc.touch(p, 0, false);
  const int kind = kind_of(c);
  if (kind == kScaleSoftmaxBwd) {
    const dim3 grid((unsigned)((s.dim[0] + kBlock / 64 - 1) / (kBlock / 64)));
    auto go = [&](auto* zero) {
      typedef std::remove_pointer_t<decltype(zero)> T;
      hipLaunchKernelGGL(k_scale_softmax_bwd<T>, grid, dim3(kBlock), 0, ctx->stream, at<const T>(f.ptr[0]), at<const T>(f.ptr[1]), at<T>(f.ptr[2] ? f.ptr[2] : f.ptr[0]),
                         at<const T>(s.ptr[0]), at<T>(s.ptr[2]), s.dim[0], (int)s.dim[1]);
    };
    if (gh_dtype_of(f.flags) == GH_F64) go((double*)nullptr);
    else go((float*)nullptr);
    return gh_check_hip(ctx, hipGetLastError(), "softmax backward launch");
  }
  const gh_cmd& pool = kind == kReluPool ? s : f;
  const int H = (int)pool.dim[2], W = (int)pool.dim[3];
  const int64_t windows = pool.dim[0] * pool.dim[1] * (H / 2) * (W / 2);
  const int64_t blocks = std::min<int64_t>((windows + kBlock - 1) / kBlock, (int64_t)ctx->cu_count * 16);
  // rows of 16-byte pairs
  if (kind == kReluPool) {
    const bool vec = W % 2 == 0 && ((f.ptr[0] | f.ptr[1]) & 15) == 0;
    hipLaunchKernelGGL((vec ? k_relu_pool_f64<true> : k_relu_pool_f64<false>), dim3((unsigned)blocks), dim3(kBlock), 0, ctx->stream, at<const double>(f.ptr[0]),
                       at<double>(f.ptr[1]), at<double>(s.ptr[1]), H, W, windows);
    return gh_check_hip(ctx, hipGetLastError(), "maxpool2d launch");
  }
  if (kind == kPoolReluBwd) {
    const bool vec = W % 2 == 0 && ((f.ptr[0] | f.ptr[2] | s.ptr[0] | s.ptr[2]) & 15) == 0;
    hipLaunchKernelGGL((vec ? k_pool_relu_bwd_f64<true> : k_pool_relu_bwd_f64<false>), dim3((unsigned)blocks), dim3(kBlock), 0, ctx->stream, at<const double>(f.ptr[0]),
                       at<const double>(f.ptr[1]), at<const double>(s.ptr[0]), at<double>(f.ptr[2]), at<double>(s.ptr[2]), H, W, windows);
    return gh_check_hip(ctx, hipGetLastError(), "maxpool backward launch");
  }
  return gh_fail(ctx, GH_EINVAL, "not a pair of commands that one launch takes");
}
