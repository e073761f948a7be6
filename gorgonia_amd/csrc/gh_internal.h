// Internal declarations shared by the translation units of libgorgonia_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "gorgonia_hip.h"

struct gh_graph_slot {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  bool used = false;
};

// A model of what the 256 MB last-level cache still holds, for the streaming kernels'
// choice between plain and non-temporal accesses: the buffers commands touched lately and
// how many bytes of streaming traffic have gone by since.  Operands the cache still holds are
// quicker through plain accesses (non-temporal ones lose 5-10 % there), operands it has lost
// are quicker streamed (6-13 % on a binary kernel).  The model only steers that choice; both
// forms store the same bits.
struct gh_llc_model {
  struct Entry { uint64_t lo, hi, stamp; };
  static constexpr int kEntries = 48;
  Entry e[kEntries] = {};
  int next = 0;
  uint64_t clock = 0;   // bytes the streaming kernels have moved so far
  // a buffer starting at p was touched within the last `window` bytes of traffic
  bool warm(uint64_t p, uint64_t window) const {
    for (const Entry& x : e)
      if (x.hi > x.lo && p >= x.lo && p < x.hi && clock - x.stamp <= window) return true;
    return false;
  }
  void touch(uint64_t p, uint64_t bytes, bool counts) {
    if (!p) return;
    if (counts) clock += bytes;
    const uint64_t hi = p + (bytes ? bytes : 1);   // size unknown: the start address alone
    for (Entry& x : e)
      if (x.hi > x.lo && p < x.hi && x.lo < hi) { x = Entry{p, hi, clock}; return; }
    e[next] = Entry{p, hi, clock};
    next = (next + 1) % kEntries;
  }
};

constexpr int kBnHeldSlots = 2048;
constexpr int64_t kBnHeldPage = kBnHeldSlots * (8 + 8 + 4 + 4);

// One sum of slabs (k_slab_sums.hip): out[e] = the sum over the slabs of ws[s][e], in one of these orders.
enum { kSumGroups64, kSumGroups16, kSumGroups64F64, kSumGroups16F64, kSumLanes16, kSumLanes4, kSumPlain };
struct gh_slab_sum {
  const void* ws;
  void* out;
  int64_t total;
  int slabs, how;
};
// A filter gradient whose launch waits for the image gradient beside it (k_conv_gradients.hip): which kernel, its grid, its
// dynamic LDS and its argument.
enum { kHeldNone, kHeldSmall, kHeldSmallNarrow, kHeldF32, kHeldF64, kHeldF64Narrow };
struct gh_held_filter {
  int kind = kHeldNone;
  dim3 grid;
  size_t lds = 0;
  alignas(16) unsigned char args[192];
};
// a pooling's gradient that an image gradient's launch takes along (k_conv_gradients.hip); dz 0: none
struct gh_unpool { uint64_t a = 0, z = 0, da = 0, dz = 0; bool done = false; };

constexpr int kUnits = 256;   // the MI355X's compute units
constexpr int kSlabSums = 8;
constexpr int64_t kSlabSpace = 24ll << 20;
constexpr int kPieces = 8;

struct gh_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  void* arena = nullptr;
  int64_t arena_bytes = 0;
  int err = GH_OK;          // sticky status
  std::string errmsg;
  bool capturing = false;
  std::vector<gh_graph_slot> graphs;
  hipEvent_t events[64] = {};
  int cu_count = kUnits;
  // scratch owned by the context (split-K partials, reduction flags)
  void* workspace = nullptr;
  int64_t workspace_bytes = 0;
  // what the workgroups of k_bn_held.hip pass to each other: two slots of 8 bytes, a claim and a count of 4 for each of
  // kBnHeldSlots, zero whenever no kernel runs; null where the device's pages were all taken
  void* bn_page = nullptr;
  // slabs whose sums gh_submit has put off, in memory of their own (kSlabSpace, or null so far), and those sums
  void* slab_space = nullptr;
  bool no_slab_space = false;   // there was none to be had
  int64_t slabs_used = 0;
  gh_slab_sum sums[kSlabSums];
  int pending = 0;
  bool defer_sums = false;
  bool hold_filter = false;   // the next filter gradient may be held
  gh_held_filter held;
  gh_unpool unpool;
  struct { int64_t launches = 0, form = 0; } joint[GH_JOINT__COUNT];   // gh_joint_launches
  // set while gh_submit_noalloc runs: the scratch is the library's fixed array and a
  // plan may not shrink to fit it (results must not depend on the scratch size)
  bool ws_strict = false;
  // gh_sync's completion word: pinned host memory the stream writes `done_seq` to (gh_api.hip)
  uint32_t* done_word = nullptr;
  uint32_t done_seq = 0;
  bool idle = true;         // nothing has been put on the stream since the last completed gh_sync
  bool runtime_wait = false;  // a copy to or from pageable memory is under way: the runtime has its own part in finishing it
  bool sync_block = false;  // gh_sync waits in the runtime only
  bool sync_spin = false;   // gh_sync never gives up its core: where it would leave the wait to the runtime it asks the stream again and again
  gh_llc_model llc;
  // uploads in pieces (gh_pieces.hip): the stream that copies them, an event for the work in front, the words they are passed
  // on by, and how many there have been
  hipStream_t pieces = nullptr;
  hipEvent_t pieces_after = nullptr;
  void* piece_words = nullptr;
  uint64_t piece_seq = 0;
  bool no_pieces = false;   // they were not to be had, or are given up too often
  // while a piece's layers are submitted: the images of the whole batch and the compute units that it would be planned for
  int64_t whole_images = 0;
  int whole_units = 0;
  // pinned host buffers handed out by gh_host_alloc: [start, end)
  std::vector<std::pair<uint64_t, uint64_t>> host_ranges;
};

// A launcher calls this where `need` bytes of scratch do not fit the workspace,
// before it shrinks its plan (fewer split-K slices, a kernel without scratch).
// Returns GH_OK to go on shrinking; under gh_submit_noalloc it records the
// sticky error instead and returns its code, which the launcher passes on.
int gh_ws_short(gh_ctx* ctx, int64_t need);

// Record a sticky error on the context and return its code.
int gh_fail(gh_ctx* ctx, int code, const std::string& msg);
int gh_check_hip(gh_ctx* ctx, hipError_t e, const char* what);

// Per-family validators (host only) and launchers.  Launchers assume a
// validated command.  Each returns GH_OK or a code with `msg` filled in.
int gh_validate_cmd(const gh_cmd& c, std::string& msg);

// whether the last-level cache has lost the buffer at p; whether a streaming kernel that moves `bytes`, all its
// inputs lost (`cold`) or not, goes past the cache (k_elem.hip)
bool gh_llc_cold(const gh_ctx* ctx, uint64_t p);
bool gh_llc_stream(int64_t bytes, bool cold);
// a copy out of pinned host memory and the commands behind it in pieces of the batch (gh_pieces.hip): how many commands it
// has submitted (0: none), *rc what came of them
int gh_submit_pieces(gh_ctx* ctx, const gh_cmd* cmds, int n, int* rc);
extern "C" int gh_submit_each(gh_ctx* ctx, const gh_cmd* cmds, int n, int before);   // before: commands of the caller's in front of these, for messages
bool gh_in_pinned_host(const gh_ctx* ctx, uint64_t p);
void gh_drop_pieces(gh_ctx* ctx);
// sums of filter-gradient slabs, put off where gh_submit allows it (k_slab_sums.hip)
void* gh_slab_space(gh_ctx* ctx, int64_t bytes);
int gh_sum_slabs(gh_ctx* ctx, const gh_slab_sum& s);
int gh_flush_sums(gh_ctx* ctx);
int gh_flush_sums_before(gh_ctx* ctx, const gh_cmd& c);
int gh_bn_groups(int64_t n, int64_t S);   // the groups of 256 threads that k_bn_reduce cuts a channel of n values in planes of S into (k_bwd.hip)
// {BN_TRAIN, MAXPOOL2D} and {MAXPOOL2D_BWD, BN_BWD} in one launch (k_bn_held.hip)
bool gh_bn_held_pair(const gh_ctx* ctx, const gh_cmd* cmds, int n);
bool gh_bn_remade_follows(const gh_cmd* c, int n);
int gh_launch_bn_remake(gh_ctx* ctx, const gh_cmd* c);
int gh_launch_bn_held_pair(gh_ctx* ctx, const gh_cmd* cmds);
// a run of elementwise commands in one pass (k_chain.hip): how many commands at the front of cmds one pass can take and is
// quicker for (0 or >= 2; gh_elementwise_run asks the same), and the launch
int gh_chain_length(const gh_cmd* cmds, int n);
int gh_launch_chain(gh_ctx* ctx, const gh_cmd* cmds, int count);
// two commands in one launch (k_pairs.hip)
bool gh_is_pair(const gh_cmd* cmds, int n);
int gh_launch_pair(gh_ctx* ctx, const gh_cmd* cmds);
// a product and the Rectify behind it (k_gemm.hip)
bool gh_rectify_follows(const gh_cmd* cmds, int n);
int gh_try_launch_gemm_rectify(gh_ctx* ctx, const gh_cmd* cmds);   // -1: no kernel has both
// a SoftMax, the tensor times a scalar behind it and the SoftMax gradient that takes both (k_pairs.hip, k_gemm.hip): what is
// behind the SoftMax's own values, row by row
template <class T> struct gh_softmax_gradient { const T* x; const T* s; T* g; T* dx; };
bool gh_softmax_gradient_follows(const gh_cmd* cmds, int n);
int gh_try_launch_softmax_gradient(gh_ctx* ctx, const gh_cmd* cmds);        // of a SOFTMAX; -1: no kernel has the three
int gh_try_launch_gemm_softmax_gradient(gh_ctx* ctx, const gh_cmd* cmds);   // of a GEMM with its SoftMax
int gh_launch_elem_bin(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_elem_unary(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_bcast_bin(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_relu(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_relu_bwd(gh_ctx* ctx, const gh_cmd& c);
// float64 twins of the backward operators (k_bwd64.hip)
int gh_launch_relu_bwd_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_dropout_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_dropout_bwd_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_softmax_bwd_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_maxpool2d_bwd_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_bn_train_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_bn_bwd_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_conv2d_bwd_data_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_conv2d_bwd_filter_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_leaky_relu(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_fill(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_has_nan_inf(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_gemm(gh_ctx* ctx, const gh_cmd& c);
// products with operands straight from memory (k_gemm_direct.hip)
int gh_gemm_direct_form(const gh_cmd& c, int cus, double* us, int* rounds);   // -1: not taken
int gh_gemm_direct_slices(const gh_cmd& c, int form, int cus);
int gh_launch_gemm_direct(gh_ctx* ctx, const gh_cmd& c, int form);
// a dense layer's two gradients in one launch (k_gemm_gradients.hip)
enum { kGemmOther, kGemmDirect, kGemmSkinny };
struct gh_gemm_choice { int kind = kGemmOther, form = 0, waves = 0, columns = 0; };   // form: k_gemm_direct's; waves, columns: the small-output kernels'; waves: k_gemm_direct's that share K, of float64 0 for four
gh_gemm_choice gh_choose_gemm(const gh_ctx* ctx, const gh_cmd& c);
bool gh_gemm_gradient_pair(const gh_cmd* cmds, int n);
// (`rectified`: cmds[2] is a Rectify's gradient and rides along)
bool gh_rectify_gradient_follows(const gh_cmd* cmds, int n);
int gh_try_launch_gemm_gradients(gh_ctx* ctx, const gh_cmd* cmds, bool rectified);   // -1: no kernel has both
// float32 products on the bf16 matrix instructions (k_gemm_split.hip)
int gh_gemm_split_form(const gh_cmd& c, int cus, double other_us, int other_slices);   // -1: not taken; the other kernel's time and its slices of K
int gh_launch_gemm_split(gh_ctx* ctx, const gh_cmd& c, int form);
// products of one to four rows (k_gemm_thin.hip)
bool gh_gemm_thin_takes(const gh_cmd& c);
int gh_launch_gemm_thin(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_gemv(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_outer(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_conv2d(gh_ctx* ctx, const gh_cmd& c);
bool gh_conv2d_in_pieces(const gh_cmd& c, int64_t images, int units, int part_units);
// small-image 3x3 convolution (k_conv_small.hip): -1 when the shape is not one it takes
int gh_try_launch_conv_small(gh_ctx* ctx, const gh_cmd& c);
int gh_try_launch_conv_wgrad_small(gh_ctx* ctx, const gh_cmd& c, int* splits, float** slabs);
bool gh_conv_wgrad_small_takes(const gh_cmd& c);
// 3x3 stride-1 filter gradient with operands straight from memory, both float types (k_conv_wgrad.hip)
bool gh_conv_wgrad_takes(const gh_cmd& c, int cus);
int64_t gh_conv_wgrad_slab_limit(const gh_cmd& c, int64_t slab_bytes);
int gh_launch_conv_wgrad(gh_ctx* ctx, const gh_cmd& c);
// both gradients of a 3x3 convolution in one launch (k_conv_gradients.hip)
bool gh_gradient_pair(const gh_cmd* cmds, int n);
int gh_launch_held(gh_ctx* ctx);
int gh_unpool_follows(const gh_cmd* cmds, int n, gh_unpool* out);
int gh_launch_held_wgrad(gh_ctx* ctx);         // k_conv_wgrad.hip
int gh_launch_held_wgrad_small(gh_ctx* ctx);   // k_conv_wgrad_small.hip
// whether a filter gradient that writes `out` (slabs, or the result itself) may be held: not where it uses the workspace
static inline bool gh_may_hold(const gh_ctx* ctx, const void* out) { return ctx->hold_filter && out != ctx->workspace; }
bool gh_conv_small_takes(const gh_cmd& c);
bool gh_conv_small_can_pool(const gh_cmd& c);
// its 32- and 64-channel kernel (k_conv_rows.hip), same conventions
int gh_try_launch_conv_rows(gh_ctx* ctx, const gh_cmd& c);
bool gh_conv_rows_takes(const gh_cmd& c);
bool gh_conv_rows_can_pool(const gh_cmd& c);
bool gh_conv_rows_can_pre(const gh_cmd& c);
// single-channel 3x3 convolution on the matrix cores (k_conv_rows1.hip), same conventions
int gh_try_launch_conv_rows1(gh_ctx* ctx, const gh_cmd& c);
bool gh_conv_rows1_takes(const gh_cmd& c);
// 3x3 convolution over patches with K split across wavefronts (k_conv_patch.hip), same conventions
int gh_try_launch_conv_patch(gh_ctx* ctx, const gh_cmd& c);
bool gh_conv_patch_takes(const gh_cmd& c);
bool gh_conv_patch_can_pool(const gh_cmd& c);
double gh_conv_patch_us(const gh_cmd& c, int cus);   // an estimate of its time
// k_conv_wide.hip: 3x3 stride-1 convolution over large images with up to 64 channels
int gh_try_launch_conv_wide(gh_ctx* ctx, const gh_cmd& c);
bool gh_conv_wide_takes(const gh_cmd& c);
bool gh_conv_wide_can_pool(const gh_cmd& c);
// k_conv_pointwise.hip: 1x1 stride-1 convolution whose result is too small for K-wide 64x64 tiles to fill the device
int gh_try_launch_conv_pointwise(gh_ctx* ctx, const gh_cmd& c);
bool gh_conv_pointwise_takes(const gh_cmd& c, int cus);
// 3x3 / padding 1 over three or four channels, in place of the wide-image kernel (k_conv_strip.hip)
bool gh_conv_strip_takes(const gh_cmd& c);
int gh_launch_conv_strip(gh_ctx* ctx, const gh_cmd& c);
// 3x3 stride-1 convolution with operands straight from memory, both float types; flip: of an image-gradient command (k_conv_lanes.hip)
int gh_conv_lanes_form(const gh_cmd& c, bool flip, int cus, double other_us, bool patch = false, bool whole = false);   // -1: not taken; the other: k_conv3x3_patch, one whose sums run over all channels
int gh_conv_lanes_form_like(const gh_cmd& c, int form, int cus);
int gh_launch_conv_lanes(gh_ctx* ctx, const gh_cmd& c, bool flip, int form);
int gh_launch_maxpool2d(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_bn_infer(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_softmax(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_maxpool2d_bwd(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_conv2d_bwd_data(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_conv2d_bwd_filter(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_bn_train(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_bn_bwd(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_softmax_bwd(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_solver_step(gh_ctx* ctx, const gh_cmd& c);
int gh_solver_run_length(const gh_cmd* cmds, int n);
int gh_launch_solver_steps(gh_ctx* ctx, const gh_cmd* cmds, int count, bool copy);   // copy: cmds[count] rides along
int gh_try_launch_solver_sums(gh_ctx* ctx, const gh_cmd* cmds, int count, bool copy);   // with the sums that wait; -1: not together
// whether the command behind a run of `count` solver steps is a small copy that has nothing to do with their tensors
bool gh_solver_copy_rides(const gh_cmd* cmds, int count, int n);
// a copy of words by the workgroups behind a launch's own
struct gh_small_copy {
  const uint32_t* src;
  uint32_t* dst;
  int words;
};
int gh_launch_rand_uniform(gh_ctx* ctx, const gh_cmd& c);
// float64 twins of the forward neural-network operators (k_nn64.hip)
int gh_launch_relu_f64(gh_ctx* ctx, const gh_cmd& c, bool leaky);
int gh_launch_maxpool2d_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_bn_infer_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_softmax_f64(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_conv2d_f64(gh_ctx* ctx, const gh_cmd& c);
bool gh_try_launch_conv2d_f64_mfma(gh_ctx* ctx, const gh_cmd& c);
bool gh_try_launch_conv2d_bwd_data_f64_mfma(gh_ctx* ctx, const gh_cmd& c);
bool gh_try_launch_conv2d_bwd_filter_f64_mfma(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_dropout(gh_ctx* ctx, const gh_cmd& c);
int gh_launch_dropout_bwd(gh_ctx* ctx, const gh_cmd& c);

// A convolution kernel's plan (geometry and workgroup shape) is a function of the command's shape,
// its dtype and of whether a pooling rides in the epilogue - and of tuning switches in the environment,
// which are read when a shape is first seen.  Finding one costs tens of microseconds on the host and a
// command asks several times (validation, the pooling query, the launcher), which an eager submit
// cannot hide behind kernels of a few microseconds: gh_plan_memo keeps the answers.  One table per call
// site (the lambda's type makes the instantiation unique); bounded, cleared when full.
template <class Plan, class Fn>
bool gh_plan_memo(const gh_cmd& c, bool pool, Plan* out, Fn&& compute) {
  struct Entry { int64_t dim[13]; uint32_t dtype; bool pool, ok; Plan plan; };
  static std::mutex mu;
  static std::vector<Entry> table;
  const uint32_t dtype = (c.flags >> 12) & 0xfu;
  {
    std::lock_guard<std::mutex> lock(mu);
    for (const Entry& e : table)
      if (e.pool == pool && e.dtype == dtype && memcmp(e.dim, c.dim, sizeof(e.dim)) == 0) {
        if (e.ok) *out = e.plan;
        return e.ok;
      }
  }
  Entry e;
  memcpy(e.dim, c.dim, sizeof(e.dim));
  e.dtype = dtype; e.pool = pool;
  e.ok = compute(&e.plan);
  std::lock_guard<std::mutex> lock(mu);
  if (table.size() >= 256) table.clear();
  table.push_back(e);
  if (e.ok) *out = e.plan;
  return e.ok;
}

static inline uint32_t gh_fn(uint32_t flags) { return flags & 0xffu; }
static inline uint32_t gh_mode(uint32_t flags) { return (flags >> 8) & 0xfu; }
static inline uint32_t gh_dtype_of(uint32_t flags) { return (flags >> 12) & 0xfu; }

// Output sizes shared by validators, launchers and the host mirror.
static inline int64_t gh_conv_out(int64_t in, int64_t k, int64_t pad, int64_t stride, int64_t dil) {
  return (in + 2 * pad - (dil * (k - 1) + 1)) / stride + 1;  // op_nn.go:311-315
}
static inline int64_t gh_pool_out(int64_t in, int64_t k, int64_t padA, int64_t padB, int64_t stride) {
  return (in + padA + padB - (k - 1) - 1) / stride + 1;      // op_nn.go:810-816
}
