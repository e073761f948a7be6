// Solver steps: one fused pass for the tensors of a model, float32 and float64, and the sums of filter-gradient slabs that the
// steps read.
//
// One pass per tensor instead of the reference's 6-15 tensor ops (solvers.go:273-372, 461-640, 780-870); every intermediate is
// rounded where a tensor op of the reference would round it, so the weights and caches get the reference's bits.
//
// A model's solver steps are many small tensors, and one launch per tensor costs more than the arithmetic (five tensors of the
// example's convnet in float64: 25.3 us as five launches, 7.3 as one).  Where the sums of its filter gradients wait
// (k_slab_sums.hip) they are added in the same launch, each result stepped by the thread that has it: a launch less, and the
// gradient is not read again.  us of a training step, the sums in a launch of their own / in this one: the convnet at batch 128 in
// float32 200.7 / 196.4, in float64 at 50 197.1 / 193.4.  Bound: the slabs' way from the caches (14 MB for the former) and the launch.
#include <algorithm>
#include <cstring>

#include "gh_slab_sums.h"

namespace {

constexpr int kBlock = 256;

template <class T>
struct Par { T eta, eps, l1reg, l2reg, clip, one_per_batch, a, b, corr1, corr2; };

template <class T>
__device__ __forceinline__ T clamped(T v, T lo, T hi) { return v < lo ? lo : (v > hi ? hi : v); }
__device__ __forceinline__ float root(float v) { return sqrtf(v); }
__device__ __forceinline__ double root(double v) { return sqrt(v); }

template <class T>
__device__ __forceinline__ T prep_grad(T g, T w, int use, const Par<T>& p) {
  if (use & 1) { const T t = p.l1reg * (T)((w > (T)0) - (w < (T)0)); g = g + t; }
  if (use & 2) { const T t = w * p.l2reg; g = g + t; }
  if (use & 8) g = g * p.one_per_batch;
  if ((use & 4) && p.clip > (T)0) g = clamped(g, -p.clip, p.clip);
  return g;
}

// Element i of a tensor, whose gradient is gi.
template <class T, int KIND>
__device__ __forceinline__ void step(T* __restrict__ w, T* __restrict__ c1, T* __restrict__ c2, int64_t i, T gi, int use, const Par<T>& p) {
  const T neg_eta = -p.eta;
  if (KIND == GH_SOLVER_VANILLA) {
    gi = prep_grad(gi, w[i], use, p);
    gi = gi * neg_eta;
    w[i] = w[i] + gi;
  } else if (KIND == GH_SOLVER_RMSPROP) {
    T gt2 = gi * gi;
    T cw = c1[i] * p.a;
    gt2 = gt2 * p.b;
    cw = cw + gt2;
    c1[i] = cw;
    if (use & 4) gi = clamped(gi, -p.clip, p.clip);
    T upd = cw + p.eps;
    upd = (T)1 / root(upd);
    gi = gi * neg_eta;
    upd = upd * gi;
    if (use & 2) { const T reg = w[i] * p.l2reg; upd = upd - reg; }
    w[i] = w[i] + upd;
  } else {
    gi = prep_grad(gi, w[i], use, p);
    const T omb1 = (T)1 - p.a, omb2 = (T)1 - p.b;
    T t1 = gi * omb1;
    T g2 = gi * gi;
    g2 = g2 * omb2;
    const T mb = c1[i] * p.a;
    t1 = t1 + mb;
    const T vb = c2[i] * p.b;
    g2 = g2 + vb;
    c1[i] = t1;
    c2[i] = g2;
    T mh = t1 * p.corr1;
    T vh = g2 * p.corr2;
    vh = root(vh);
    vh = vh + p.eps;
    mh = mh * neg_eta;
    mh = mh / vh;
    w[i] = w[i] + mh;
  }
}

// Up to kTensors weight tensors per launch.  Tensor t owns workgroups [first[t], first[t + 1]).
constexpr int kTensors = 8;
template <class T>
struct Tensors {
  T* w[kTensors]; const T* g[kTensors]; T* c1[kTensors]; T* c2[kTensors];
  int64_t n[kTensors];
  int first[kTensors + 1];
  int count;
};
// Sums and the tensors whose gradients they are; w null: a sum that no tensor of the run has to do with.
template <class T>
struct Sums {
  slab_sums::Batch batch;
  T* w[kSlabSums]; T* c1[kSlabSums]; T* c2[kSlabSums];
};

template <class T, int KIND>
__device__ __forceinline__ void workgroup(const Tensors<T>& sb, int block, int use, Par<T> p, const T* __restrict__ corr, const gh_small_copy& copy) {
  if (block >= sb.first[kTensors]) {
    const int i = (block - sb.first[kTensors]) * kBlock + (int)threadIdx.x;
    if (i < copy.words) copy.dst[i] = copy.src[i];
    return;
  }
  // Adam's two bias corrections from device memory when the command names it: they change
  // every step, and as command constants they would make every step a new command
  if (KIND == GH_SOLVER_ADAM && corr) { p.corr1 = corr[0]; p.corr2 = corr[1]; }
  int t = 0;
#pragma unroll
  for (int q = 1; q < kTensors; q++)
    if (q < sb.count && block >= sb.first[q]) t = q;
  const T* __restrict__ g = sb.g[t];
  const int64_t n = sb.n[t], nblk = sb.first[t + 1] - sb.first[t];
  for (int64_t i = (int64_t)(block - sb.first[t]) * kBlock + threadIdx.x; i < n; i += nblk * kBlock)
    step<T, KIND>(sb.w[t], sb.c1[t], sb.c2[t], i, g[i], use, p);
}

template <class T, int KIND>
__global__ __launch_bounds__(kBlock) void k_solver_step(const Tensors<T> sb, int use, Par<T> p, const T* __restrict__ corr, gh_small_copy copy) {
  workgroup<T, KIND>(sb, (int)blockIdx.x, use, p, corr, copy);
}

template <class T, int KIND>
__global__ __launch_bounds__(kBlock) void k_solver_step_sums(const Sums<T> sums, const Tensors<T> sb, int use, Par<T> p, const T* __restrict__ corr, gh_small_copy copy) {
  __shared__ double sh[256];
  const slab_sums::Batch& b = sums.batch;
  const int block = (int)blockIdx.x;
  if (block >= b.first[kSlabSums]) {
    workgroup<T, KIND>(sb, block - b.first[kSlabSums], use, p, corr, copy);
    return;
  }
  if (KIND == GH_SOLVER_ADAM && corr) { p.corr1 = corr[0]; p.corr2 = corr[1]; }
  int t = 0;
#pragma unroll
  for (int q = 1; q < kSlabSums; q++)
    if (block >= b.first[q]) t = q;
  T* const out = (T*)b.out[t];
  T* const w = sums.w[t];
  T *const c1 = sums.c1[t], *const c2 = sums.c2[t];
  slab_sums::workgroup<T>(b, t, block - b.first[t], sh, [&](int64_t e, T sum) {
    out[e] = sum;
    if (w) step<T, KIND>(w, c1, c2, e, sum, use, p);
  });
}

template <class T, int KIND>
void go(gh_ctx* ctx, const Sums<T>* sums, const Tensors<T>& sb, int blocks, int use, const Par<T>& p, const T* corr, const gh_small_copy& tail) {
  if (sums)
    hipLaunchKernelGGL((k_solver_step_sums<T, KIND>), dim3((unsigned)(sums->batch.first[kSlabSums] + blocks)), dim3(kBlock), 0, ctx->stream, *sums, sb, use, p, corr, tail);
  else
    hipLaunchKernelGGL((k_solver_step<T, KIND>), dim3((unsigned)blocks), dim3(kBlock), 0, ctx->stream, sb, use, p, corr, tail);
}

template <class T>
Par<T> par_of(const gh_cmd& c) {
  if constexpr (sizeof(T) == 8) {   // float64 settings are bit patterns in dim[1..10]
    double v[10];
    static_assert(sizeof(v) == 10 * sizeof(c.dim[0]), "a setting to a dimension");
    memcpy(v, c.dim + 1, sizeof v);
    return {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9]};
  } else {
    return {c.f[0], c.f[1], c.f[2], c.f[3], c.f[4], c.f[5], c.f[6], c.f[7], c.f[8], c.f[9]};
  }
}

// One launch for cmds[0..count), for the copy behind them and for the sums; of_sum: the tensor's sum, or -1.
template <class T>
int launch(gh_ctx* ctx, const gh_cmd* cmds, int count, bool copy, const gh_slab_sum* waiting, int waits, const int* of_sum) {
  const gh_cmd& c = cmds[0];
  const int kind = (int)gh_fn(c.flags), use = (int)gh_mode(c.flags);
  Tensors<T> sb{};
  Sums<T> sums{};
  if (waits) slab_sums::batch_of(waiting, waits, &sums.batch);
  int nt = 0, blocks = 0;
  for (int i = 0; i < count; i++) {
    const int64_t n = cmds[i].dim[0];
    if (n == 0) continue;
    T *const w = (T*)(uintptr_t)cmds[i].ptr[0], *const c1 = (T*)(uintptr_t)cmds[i].ptr[2], *const c2 = (T*)(uintptr_t)cmds[i].ptr[3];
    if (waits && of_sum[i] >= 0) {
      sums.w[of_sum[i]] = w;
      sums.c1[of_sum[i]] = c1;
      sums.c2[of_sum[i]] = c2;
      continue;
    }
    sb.w[nt] = w;
    sb.g[nt] = (const T*)(uintptr_t)cmds[i].ptr[1];
    sb.c1[nt] = c1;
    sb.c2[nt] = c2;
    sb.n[nt] = n;
    sb.first[nt] = blocks;
    blocks += (int)std::min<int64_t>((n + kBlock - 1) / kBlock, (int64_t)ctx->cu_count * 32);
    nt++;
  }
  if (nt == 0 && !copy && !waits) return GH_OK;
  for (int i = nt; i <= kTensors; i++) sb.first[i] = blocks;
  sb.count = nt;
  gh_small_copy tail{};
  if (copy) tail = {(const uint32_t*)(uintptr_t)cmds[count].ptr[1], (uint32_t*)(uintptr_t)cmds[count].ptr[0], (int)(cmds[count].dim[0] / 4)};
  blocks += (tail.words + kBlock - 1) / kBlock;
  const Par<T> p = par_of<T>(c);
  const T* const corr = (const T*)(uintptr_t)c.ptr[4];
  const Sums<T>* const with = waits ? &sums : nullptr;
  if (kind == GH_SOLVER_VANILLA) go<T, GH_SOLVER_VANILLA>(ctx, with, sb, blocks, use, p, corr, tail);
  else if (kind == GH_SOLVER_RMSPROP) go<T, GH_SOLVER_RMSPROP>(ctx, with, sb, blocks, use, p, corr, tail);
  else go<T, GH_SOLVER_ADAM>(ctx, with, sb, blocks, use, p, corr, tail);
  return gh_check_hip(ctx, hipGetLastError(), "solver step launch");
}

// Whether step b, of a's solver and type, has to come after step a: one of them writes what the other reads or writes.
bool follows(const gh_cmd& a, const gh_cmd& b) {
  const int kind = (int)gh_fn(a.flags), caches = kind == GH_SOLVER_VANILLA ? 0 : kind == GH_SOLVER_RMSPROP ? 1 : 2;
  const int64_t size = gh_dtype_of(a.flags) == GH_F64 ? 8 : 4;
  auto meet = [](uint64_t p, int64_t np, uint64_t q, int64_t nq) { return p && q && p < q + (uint64_t)nq && q < p + (uint64_t)np; };
  auto written = [&](const gh_cmd& x, const gh_cmd& y) {   // by x, and of y's
    for (int i = 0; i < 2 + caches; i++) {
      if (i == 1) continue;   // the gradient
      for (int k = 0; k < 2 + caches; k++)
        if (meet(x.ptr[i], x.dim[0] * size, y.ptr[k], y.dim[0] * size)) return true;
      if (kind == GH_SOLVER_ADAM && meet(x.ptr[i], x.dim[0] * size, y.ptr[4], 2 * size)) return true;   // the corrections
    }
    return false;
  };
  return written(a, b) || written(b, a);
}

}  // namespace

// How many of the commands cmds[0..n) form one solver launch: consecutive
// SOLVER_STEP commands with the same solver, options and hyper-parameters.
int gh_solver_run_length(const gh_cmd* cmds, int n) {
  if (n <= 0 || cmds[0].opcode != GH_OP_SOLVER_STEP) return 0;
  // (float64 settings are bit patterns in dim[1..10], float32 ones are in f)
  int len = 1;
  while (len < n && len < kTensors && cmds[len].opcode == GH_OP_SOLVER_STEP && cmds[len].flags == cmds[0].flags &&
         cmds[len].ptr[4] == cmds[0].ptr[4] && memcmp(cmds[len].f, cmds[0].f, sizeof(cmds[0].f)) == 0 &&
         memcmp(cmds[len].dim + 1, cmds[0].dim + 1, sizeof(cmds[0].dim) - sizeof(cmds[0].dim[0])) == 0) {
    // steps that have to do with each other keep their order: the run ends before the later one
    bool later = false;
    for (int j = 0; j < len; j++) later = later || follows(cmds[j], cmds[len]);
    if (later) break;
    len++;
  }
  return len;
}

// The network's result leaves the device behind the solver's steps: of up to 64 KB, by more workgroups of their launch (a
// launch of its own some 3 us).
bool gh_solver_copy_rides(const gh_cmd* cmds, int count, int n) {
  if (count >= n || cmds[count].opcode != GH_OP_MEMCPY_D2D) return false;
  const gh_cmd& c = cmds[count];
  const int64_t bytes = c.dim[0];
  if (bytes <= 0 || bytes > 65536 || ((c.ptr[0] | c.ptr[1] | (uint64_t)bytes) & 3) || !c.ptr[0] || !c.ptr[1]) return false;
  auto meets = [&](uint64_t p, int64_t size, uint64_t q) { return q && q < p + (uint64_t)bytes && p < q + (uint64_t)size; };
  if (meets(c.ptr[0], bytes, c.ptr[1])) return false;
  for (int i = 0; i < count; i++) {
    const int64_t size = cmds[i].dim[0] * (gh_dtype_of(cmds[i].flags) == GH_F64 ? 8 : 4);
    for (int k = 0; k < 4; k++)
      if (meets(c.ptr[0], size, cmds[i].ptr[k]) || (k != 1 && meets(c.ptr[1], size, cmds[i].ptr[k]))) return false;
    if (meets(c.ptr[0], 16, cmds[i].ptr[4])) return false;   // the corrections
  }
  return true;
}

// One launch for cmds[0..count) (count from gh_solver_run_length), and for the copy behind them.
int gh_launch_solver_steps(gh_ctx* ctx, const gh_cmd* cmds, int count, bool copy) {
  return gh_dtype_of(cmds[0].flags) == GH_F64 ? launch<double>(ctx, cmds, count, copy, nullptr, 0, nullptr) : launch<float>(ctx, cmds, count, copy, nullptr, 0, nullptr);
}

int gh_launch_solver_step(gh_ctx* ctx, const gh_cmd& c) { return gh_launch_solver_steps(ctx, &c, 1, false); }

// The same with the sums that wait, where each of them is of the steps' type and is either one step's whole gradient and meets
// nothing else of what the steps and the copy read or write, or meets none of it: -1 where that is not so, or none is a step's gradient.
// (The commands are valid ones.)
int gh_try_launch_solver_sums(gh_ctx* ctx, const gh_cmd* cmds, int count, bool copy) {
  const int64_t size = gh_dtype_of(cmds[0].flags) == GH_F64 ? 8 : 4;
  int of_sum[kTensors];
  std::fill(of_sum, of_sum + kTensors, -1);
  bool any = false;
  for (int s = 0; s < ctx->pending; s++) {
    const gh_slab_sum& sum = ctx->sums[s];
    if (slab_sums::item(sum.how) != size) return -1;
    const uint64_t from = (uint64_t)(uintptr_t)sum.out, to = from + (uint64_t)(sum.total * size);
    auto meets = [&](uint64_t p, int64_t bytes) { return p && p < to && from < p + (uint64_t)bytes; };
    int taken = -1;
    for (int i = 0; i < count; i++) {
      const int64_t bytes = cmds[i].dim[0] * size;
      const bool own = cmds[i].ptr[1] == from && cmds[i].dim[0] == sum.total && taken < 0;
      if (own) taken = i;
      for (int k = 0; k < 4; k++)
        if (!(k == 1 && own) && meets(cmds[i].ptr[k], bytes)) return -1;
      if (meets(cmds[i].ptr[4], 2 * size)) return -1;   // the corrections
    }
    if (copy && (meets(cmds[count].ptr[0], cmds[count].dim[0]) || meets(cmds[count].ptr[1], cmds[count].dim[0]))) return -1;
    if (taken >= 0) {
      of_sum[taken] = s;
      any = true;
    }
  }
  if (!any) return -1;
  // (as a step by itself is in the account; longer runs never were)
  if (count + copy == 1)
    for (uint64_t p : cmds[0].ptr) ctx->llc.touch(p, 0, false);
  const int waits = ctx->pending;
  ctx->pending = 0;
  ctx->slabs_used = 0;
  ctx->joint[GH_JOINT_SOLVER_SUMS].launches++;
  ctx->joint[GH_JOINT_SOLVER_SUMS].form = std::count_if(of_sum, of_sum + kTensors, [](int s) { return s >= 0; });
  return size == 8 ? launch<double>(ctx, cmds, count, copy, ctx->sums, waits, of_sum) : launch<float>(ctx, cmds, count, copy, ctx->sums, waits, of_sum);
}
