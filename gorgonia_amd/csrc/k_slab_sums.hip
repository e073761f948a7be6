// Sums of filter-gradient slabs, several gradients in one launch.
//
// A filter gradient's long axis is cut among workgroups, whose slabs of partial results a second launch adds up: some 5 us
// each, of which the additions take one or two.  A training step has one for each layer, and nobody reads a gradient before
// the solver.  So the sums are put off while the commands behind the gradient, of the kinds that stand between the layers of
// a backward pass, neither read nor write its result: the slabs lie in 24 MB of the context's that nothing else uses (made for
// its first submission of several commands with a filter gradient, given back with the context), and the next command of another kind, one that touches a result, or the end of the submission has them added in one launch
// (the solver's steps in theirs, k_solver.hip).
// us of a training step, a launch for each sum / one: the convnet at batch 128 in float32 229 / 222, the four-block network at
// batch 8 431 / 424.
#include <algorithm>

#include "gh_slab_sums.h"

namespace {

using namespace slab_sums;

__global__ __launch_bounds__(256) void k_slab_sums(const Batch b) {
  __shared__ double sh[256];
  int t = 0;
#pragma unroll
  for (int q = 1; q < kSlabSums; q++)
    if ((int)blockIdx.x >= b.first[q]) t = q;
  const int block = blockIdx.x - b.first[t];
  if (b.how[t] == kSumGroups64F64 || b.how[t] == kSumGroups16F64) {
    double* const out = (double*)b.out[t];
    workgroup<double>(b, t, block, sh, [&](int64_t e, double sum) { out[e] = sum; });
  } else {
    float* const out = (float*)b.out[t];
    workgroup<float>(b, t, block, sh, [&](int64_t e, float sum) { out[e] = sum; });
  }
}

int launch(gh_ctx* ctx, const gh_slab_sum* sums, int n) {
  Batch b;
  const int blocks = batch_of(sums, n, &b);
  hipLaunchKernelGGL(k_slab_sums, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, b);
  return gh_check_hip(ctx, hipGetLastError(), "slab sum launch");
}

struct Range {
  uint64_t from, to;
};

// What a command of a backward pass reads and writes; 0 for other commands.
int ranges_of(const gh_cmd& c, Range (&r)[8]) {
  const int64_t size = gh_dtype_of(c.flags) == GH_F64 ? 8 : 4;
  int n = 0;
  auto add = [&](int slot, int64_t values) { r[n++] = {c.ptr[slot], c.ptr[slot] + (uint64_t)(values * size)}; };
  const int64_t B = c.dim[0], C = c.dim[1];
  switch (c.opcode) {
    case GH_OP_CONV2D_BWD_DATA: case GH_OP_CONV2D_BWD_FILTER: {
      const int64_t x = B * C * c.dim[2] * c.dim[3], w = c.dim[4] * C * c.dim[5] * c.dim[6];
      const int64_t dy = B * c.dim[4] * gh_conv_out(c.dim[2], c.dim[5], c.dim[7], c.dim[9], c.dim[11]) * gh_conv_out(c.dim[3], c.dim[6], c.dim[8], c.dim[10], c.dim[12]);
      const bool data = c.opcode == GH_OP_CONV2D_BWD_DATA;   // dy, w, dx; else x, dy, dw
      add(0, data ? dy : x);
      add(1, data ? w : dy);
      add(2, data ? x : w);
      return n;
    }
    case GH_OP_MAXPOOL2D_BWD: {
      const int64_t x = B * C * c.dim[2] * c.dim[3];
      add(0, x);
      add(1, B * C * gh_pool_out(c.dim[2], c.dim[4], c.dim[6], c.dim[7], c.dim[10]) * gh_pool_out(c.dim[3], c.dim[5], c.dim[8], c.dim[9], c.dim[11]));
      add(2, x);
      return n;
    }
    case GH_OP_BN_BWD:
      for (int k = 0; k < 3; k++) add(k, B * C * c.dim[2]);
      add(3, C);
      add(4, C);
      return n;
    case GH_OP_RELU_BWD:
      for (int k = 0; k < 3; k++) add(k, c.dim[0]);
      return n;
  }
  return 0;
}

}  // namespace

// Where a filter gradient puts its slabs: in memory of its own if its sum may be put off, else in the workspace.
void* gh_slab_space(gh_ctx* ctx, int64_t bytes) {
  if (!ctx->defer_sums || ctx->pending == kSlabSums || ctx->slabs_used + bytes > kSlabSpace) return ctx->workspace;
  void* const p = (char*)ctx->slab_space + ctx->slabs_used;
  ctx->slabs_used += (bytes + 255) / 256 * 256;
  return p;
}

int gh_sum_slabs(gh_ctx* ctx, const gh_slab_sum& s) {
  const char *p = (const char*)s.ws, *base = (const char*)ctx->slab_space;
  if (!base || p < base || p >= base + kSlabSpace) return launch(ctx, &s, 1);
  ctx->sums[ctx->pending++] = s;
  return GH_OK;
}

int gh_flush_sums(gh_ctx* ctx) {
  const int n = ctx->pending;
  ctx->pending = 0;
  ctx->slabs_used = 0;
  return n ? launch(ctx, ctx->sums, n) : GH_OK;
}

// The sums that were put off, in front of a command that may have to do with their results.  (c is a valid command.)
int gh_flush_sums_before(gh_ctx* ctx, const gh_cmd& c) {
  if (!ctx->pending) return GH_OK;
  Range r[8];
  const int n = ranges_of(c, r);
  bool meets = n == 0;
  for (int i = 0; i < ctx->pending; i++) {
    const gh_slab_sum& s = ctx->sums[i];
    const uint64_t from = (uint64_t)(uintptr_t)s.out, to = from + (uint64_t)(s.total * item(s.how));
    for (int k = 0; k < n; k++) meets = meets || (r[k].from < to && from < r[k].to);
  }
  return meets ? gh_flush_sums(ctx) : GH_OK;
}
