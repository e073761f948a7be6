// A batch out of pinned host memory and the layers behind it, in pieces of some images: while the bus brings one piece, the
// convolutions and poolings at the front of the network work on the one before.
//
// The copy is one kernel on a stream of its own, with one workgroup for each XCD; in front of a piece's layers, on the
// context's stream, stands a kernel that waits until the copy's workgroups have all said that the piece is there.  (Events
// between the streams cost 10 us a piece, and the copy engine pauses as long between two copies.)
//
// Bound: the bus, then the layers of the last piece and what follows them.  Where both run, they are in each other's way at
// two places, which decide the copy's form:
//   * A compute unit returns loads in order, so that a convolution's wait behind the host's where both are on one: the copy's
//     workgroups take all registers of eight compute units.
//   * A kernel begins and ends with its caches in order, and that waits for what is under way to and from memory: with 16
//     workgroups of 1024 threads and 8 loads each, 2 MB under way, a pooling of 4 us took 29.  One load each (128 KB) is as
//     quick for the bus, and stores that go through to memory leave nothing to be written back.
// us, whole / in pieces: a detector of eight convolutions, 8 x 3 x 416 x 416 695 / 619, five images 510 / 474, two 233 / 225,
// 8 x 3 x 320 x 320 450 / 410, five of them 311 / 299, 8 x 3 x 224 x 224 251 / 240.
//
// Nothing waits for a workgroup that has not begun: a part of a piece is copied by whoever claims it first, the copy's
// workgroup or, after some time of the device's clock, the kernel that waits for it (where something runs the streams one after
// the other, the copy behind: a process has four hardware queues, and the copies of two contexts may each stand behind the other's
// layers).  That is about three times what the bus takes, and once in an upload: the pieces behind are copied without a wait for
// who has not begun by then.  A part that is claimed is being copied, and waited for without a limit.  After kMisses such uploads
// close to each other the context's batches go whole.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "gh_internal.h"

namespace {

constexpr int kThreads = 1024, kCopiers = 8;
constexpr int kThrough = 1 | 16;                      // a store's sc0 and sc1 bits: to memory, past the caches
constexpr int64_t kBegin = 20000;                     // ticks of 10 ns for a workgroup to begin, and one more for 200 bytes
constexpr int64_t kGiveUp = 400000;                   // and to claim a part, and one more for 100 bytes (GORGONIA_HIP_PIECES_TICKS: fewer of both)
constexpr int kMisses = 3, kWithin = 64;              // uploads that were given up, and how many may lie between two of them
constexpr int64_t kLeast = GH_PIECES_FROM, kMost = 1 << 30;  // bytes of an upload (the least: two images of 3 x 416 x 416 gain 3 %)
constexpr int64_t kPieceBytes = 4 << 20;              // (8 x 3 x 416 x 416 in two, three, four and eight: 637, 635, 618 and 700 us)
constexpr int kHead = 12;
constexpr int kTries = 6;
constexpr int64_t kTryFor = 30000;                    // ticks of 10 ns
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Who copies part b of piece p (2 s: the copy's workgroup, 2 s + 1: the kernel that waits), and that it is there (s), for the
// context's s-th upload.  late: the last upload of which a kernel that waits has given something up; missed, misses: the last one
// that counts, and how many there have been in a row.
struct Words { unsigned long long claim[kPieces][kCopiers], there[kPieces][kCopiers], late, missed, misses; };
struct Ends { int n16[kPieces]; };

__device__ __forceinline__ bool claims(unsigned long long* word, unsigned long long seq, int who) {
  return __hip_atomic_fetch_max(word, 2 * seq + who, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < 2 * seq;
}

// Part `part` of the 16-byte words from .. to, and of the last piece the 4-byte words behind them.
__device__ __forceinline__ void copy_part(const __amdgpu_buffer_rsrc_t& out, const u32x4* src, int from, int to, int tail_words, int part) {
  for (int i = from + part * kThreads + (int)threadIdx.x; i < to; i += kCopiers * kThreads) __builtin_amdgcn_raw_buffer_store_b128(src[i], out, i * 16, 0, kThrough);
  if (part == 0 && (int)threadIdx.x < tail_words)
    __builtin_amdgcn_raw_buffer_store_b32(((const unsigned*)(src + to))[threadIdx.x], out, to * 16 + (int)threadIdx.x * 4, 0, kThrough);
}

__global__ __launch_bounds__(kThreads) void k_copy_pieces(void* dst, const u32x4* __restrict__ src, const Ends ends, int pieces, int tail_words, Words* words,
                                                          unsigned long long seq) {
  asm volatile("" ::: "v127");   // 16 wavefronts of 128 registers: all of a compute unit's
  __shared__ bool mine;
  const int part = blockIdx.x;
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(dst, 0, ends.n16[pieces - 1] * 16 + tail_words * 4, 0x00020000);
  for (int p = 0; p < pieces; p++) {
    if (threadIdx.x == 0) mine = claims(&words->claim[p][part], seq, 0);
    __syncthreads();
    const bool go = mine;   // the same in all threads
    if (go) copy_part(out, src, p ? ends.n16[p - 1] : 0, ends.n16[p], p == pieces - 1 ? tail_words : 0, part);
    __builtin_amdgcn_s_waitcnt(0);   // the wavefront's stores have reached memory
    __syncthreads();
    if (go && threadIdx.x == 0) __hip_atomic_store(&words->there[p][part], seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

__global__ __launch_bounds__(kThreads) void k_await_piece(void* dst, const u32x4* __restrict__ src, int bytes, int from, int to, int tail_words, Words* words,
                                                          int p, unsigned long long seq, int64_t begin, int64_t give_up, unsigned* misses) {
  __shared__ unsigned long long left;   // the parts that are copied here
  if (threadIdx.x < 64) {
    const int part = threadIdx.x;
    const int64_t t0 = wall_clock64();
    const bool late = words->late == seq;
    bool waits = part < kCopiers, mine = false, tried = false;
    for (;;) {
      if (waits) waits = __hip_atomic_load(&words->there[p][part], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) < seq;
      if (__ballot(waits) == 0) break;
      const int64_t t = (int64_t)wall_clock64() - t0;
      if (waits && !tried && (late || t >= begin)) {
        // (a workgroup that has had its part of the first piece comes to this one)
        const bool begun = __hip_atomic_load(&words->claim[0][part], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 2 * seq;
        if (!begun || t >= give_up) {
          tried = true;
          mine = claims(&words->claim[p][part], seq, 1);
          waits = !mine;
        }
      }
      __builtin_amdgcn_s_sleep(2);
    }
    const unsigned long long all = __ballot(mine);
    if (part == 0) {
      left = all;
      if (all && !late) {
        words->late = seq;
        if (misses) {
          words->misses = words->missed && seq - words->missed <= kWithin ? words->misses + 1 : 1;
          words->missed = seq;
          __hip_atomic_store(misses, (unsigned)words->misses, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
      }
    }
  }
  __syncthreads();
  if (left == 0) return;
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(dst, 0, bytes, 0x00020000);
  for (int part = 0; part < kCopiers; part++)
    if (left >> part & 1) copy_part(out, src, from, to, tail_words, part);
}

__global__ void k_clear_words(Words* words) { ((unsigned long long*)words)[threadIdx.x] = 0; }
constexpr int kWordCount = sizeof(Words) / 8;

// the compute units that layers beside the copy are planned for
int units_beside(int units) { return std::max(1, units - kCopiers); }

struct Span { uint64_t lo, hi; };
bool meet(const Span& a, const Span& b) { return a.lo < b.hi && b.lo < a.hi; }

// A command that makes each image's result from that image alone: the pointer it writes through, the bytes of one image that
// it reads and writes, and about what it takes.
struct Layer { int out; int64_t in_bytes, out_bytes; double us; };

bool by_image(const gh_cmd& c, Layer* l) {
  if (gh_dtype_of(c.flags) != 0) return false;
  const int64_t B = c.dim[0], C = c.dim[1], H = c.dim[2], W = c.dim[3];
  l->in_bytes = C * H * W * 4;
  if (c.opcode == GH_OP_CONV2D) {
    if (c.flags & (GH_FLAG_CONV_PRE | GH_FLAG_CONV_KEEP)) return false;
    const int64_t F = c.dim[4];
    int64_t oh = gh_conv_out(H, c.dim[5], c.dim[7], c.dim[9], c.dim[11]), ow = gh_conv_out(W, c.dim[6], c.dim[8], c.dim[10], c.dim[12]);
    l->us = 7 + 2.0 * (double)(B * C * F) * (double)(c.dim[5] * c.dim[6]) * (double)(oh * ow) / 100e6;
    if (c.flags & GH_FLAG_CONV_POOL2) oh /= 2, ow /= 2;
    l->out = 2;
    l->out_bytes = F * oh * ow * 4;
    return true;
  }
  if (c.opcode == GH_OP_MAXPOOL2D) {
    l->us = 5;
    l->out = 1;
    l->out_bytes = C * gh_pool_out(H, c.dim[4], c.dim[6], c.dim[7], c.dim[10]) * gh_pool_out(W, c.dim[5], c.dim[8], c.dim[9], c.dim[11]) * 4;
    return true;
  }
  return false;
}

// Whether the kernels take a valid command's shape with `fewest` and with `most` of its images, too, and add there as they do for
// the whole batch.  Asking them all takes 5 to 10 us of host time a layer, in front of a copy of 70 and more; the answers are a
// function of the shape, of the alignment that kernels ask for (k_conv1x1: whole lines of filters) and of the switches that take
// kernels out, and are kept, one for each of kKept places.  (Other tuning switches are read when a shape is first seen, as for plans.)
// us of host time for a detector's front, asked / kept: 8 x 3 x 416 x 416 21 / 3, 8 x 3 x 320 x 320 40 / 3.
constexpr int kKept = 64;
int64_t switches() {
  int64_t set = 0;
  for (const char* name : {"GORGONIA_HIP_CONV_NO_LANES", "GORGONIA_HIP_CONV_NO_STRIP", "GORGONIA_HIP_CONV_NO_DIRECT", "GORGONIA_HIP_CONV_NO_ROWS1", "GORGONIA_HIP_CONV_NO_POINTWISE"})
    set = set << 1 | (getenv(name) != nullptr);
  return set;
}
bool runs_in_pieces(const gh_cmd& c, int64_t fewest, int64_t most, int units, int64_t set) {
  struct Shape { int64_t dim[16]; int64_t fewest, most, code, units, aligned; };
  struct Place { Shape shape; bool known, fits; };
  static std::mutex mu;
  static Place places[kKept] = {};
  Shape s;
  memcpy(s.dim, c.dim, sizeof s.dim);
  s.fewest = fewest;
  s.most = most;
  s.code = (int64_t)c.opcode << 32 | c.flags;
  s.units = (int64_t)units << 8 | set;
  s.aligned = (int64_t)(c.ptr[1] & 15) << 2 | (int64_t)((c.ptr[0] | c.ptr[1] | c.ptr[2]) & 3);
  uint64_t h = 0;
  for (size_t i = 0; i < sizeof s / 8; i++) h = (h ^ (uint64_t)((const int64_t*)&s)[i]) * 0x9E3779B97F4A7C15ull;
  Place& p = places[h >> 32 & (kKept - 1)];
  {
    std::lock_guard<std::mutex> lock(mu);
    if (p.known && memcmp(&p.shape, &s, sizeof s) == 0) return p.fits;
  }
  std::string m;
  bool fits = true;
  for (int64_t images : {fewest, most}) {
    gh_cmd part = c;
    part.dim[0] = images;
    fits = fits && gh_validate_cmd(part, m) == GH_OK;
    if (c.opcode == GH_OP_CONV2D)
      for (int u : {units, units_beside(units)}) fits = fits && gh_conv2d_in_pieces(c, images, units, u);
  }
  std::lock_guard<std::mutex> lock(mu);
  p = Place{s, true, fits};
  return fits;
}

// The layers behind the upload that run in pieces: as many as take, whole, about half of the upload's time (8 x 3 x 416 x 416:
// three layers 628 us, with the fourth and its pooling 619), each reads what the one in front wrote, image by image, and the kernels take their shapes
// with a piece's images, too, and add there as they do for the whole batch: whether a batch goes in pieces (eagerly) or whole (under
// capture) changes no bits.  A layer's work on the first piece comes before the work of those in front of it on the last: what it
// writes lies apart from all that they read and write, their filters and constants among it.
template <class InHost>
int head_of(const gh_cmd* cmds, int n, int64_t fewest, int64_t most, Layer* layers, int units, InHost&& in_host) {
  const gh_cmd& up = cmds[0];
  const int64_t B = cmds[1].dim[0];
  std::string m;
  Span values[kHead + 1], constants[5 * kHead];
  uint64_t from = up.ptr[0];
  values[0] = Span{from, from + (uint64_t)up.dim[0]};
  double us = 0;
  const int64_t set = switches();
  int head = 0, held = 0;
  for (; head < kHead && head + 1 < n; head++) {
    const gh_cmd& c = cmds[head + 1];
    Layer& l = layers[head];
    if (c.dim[0] != B || gh_validate_cmd(c, m) || !by_image(c, &l) || c.ptr[0] != from) break;
    if (head == 0 ? B * l.in_bytes != up.dim[0] : l.in_bytes != layers[head - 1].out_bytes) break;
    if ((us += l.us) > 0.55 * (double)up.dim[0] / 56e3) break;
    from = c.ptr[l.out];
    values[head + 1] = Span{from, from + (uint64_t)(B * l.out_bytes)};
    if (c.opcode == GH_OP_CONV2D)
      for (int k : {1, 3, 4, 5, 6}) {
        const int64_t bytes = (k == 1 ? c.dim[1] * c.dim[4] * c.dim[5] * c.dim[6] : c.dim[4]) * 4;
        if (c.ptr[k]) constants[held++] = Span{c.ptr[k], c.ptr[k] + (uint64_t)bytes};
      }
    bool fits = !in_host(from);
    for (int k = 0; k <= head; k++) fits = fits && !meet(values[k], values[head + 1]);
    for (int k = 0; k < held; k++)
      for (int s = 0; s <= head + 1; s++) fits = fits && !meet(values[s], constants[k]);
    if (!fits || !runs_in_pieces(c, fewest, most, units, set)) break;
  }
  return head;
}

// How many pieces the commands' batch would be in, 0 where it goes whole.
int pieces_of(const gh_cmd* cmds, int n) {
  if (n < 2) return 0;
  const gh_cmd& up = cmds[0];
  const int64_t bytes = up.dim[0], B = cmds[1].dim[0];
  if (up.opcode != GH_OP_MEMCPY_D2D || bytes < kLeast || bytes > kMost || bytes % 4 || B < 2 || ((up.ptr[0] | up.ptr[1]) & 15)) return 0;
  std::string m;
  if (gh_validate_cmd(up, m)) return 0;
  return (int)std::min({B, (int64_t)kPieces, std::max<int64_t>(2, (bytes + kPieceBytes - 1) / kPieceBytes)});
}

template <class InHost>
int layers_of(const gh_cmd* cmds, int n, int pieces, Layer* layers, int units, InHost&& in_host) {
  const int64_t B = cmds[1].dim[0];
  return head_of(cmds, n, B / pieces, (B + pieces - 1) / pieces, layers, units, in_host);
}

// Streams share a few hardware queues, and two of one queue run one behind the other (a batch of 8 then takes 740 us).  Which
// have one is not told, so a stream is tried: a kernel on the context's stream waits, for a limited time, for what a kernel
// on the other writes.
__global__ void k_try_wait(unsigned* word) {
  const int64_t t0 = wall_clock64();
  while (!__hip_atomic_load(word, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) && (int64_t)wall_clock64() - t0 < kTryFor) __builtin_amdgcn_s_sleep(2);
  word[1] = __hip_atomic_load(word, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
}
__global__ void k_try_say(unsigned* word) { __hip_atomic_store(word, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT); }

bool side_by_side(gh_ctx* ctx, hipStream_t s) {
  unsigned* const word = (unsigned*)ctx->piece_words;
  unsigned seen = 0;
  hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(kWordCount), 0, s, (Words*)ctx->piece_words);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) return false;
  hipLaunchKernelGGL(k_try_wait, dim3(1), dim3(1), 0, ctx->stream, word);
  hipLaunchKernelGGL(k_try_say, dim3(1), dim3(1), 0, s, word);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(ctx->stream) != hipSuccess || hipStreamSynchronize(s) != hipSuccess) return false;
  return hipMemcpyAsync(&seen, word + 1, sizeof seen, hipMemcpyDeviceToHost, ctx->stream) == hipSuccess && hipStreamSynchronize(ctx->stream) == hipSuccess && seen;
}

// Where the kernels that wait say how many uploads they gave up, behind the completion word on its cache line.
unsigned* missed(const gh_ctx* ctx) { return ctx->done_word + 4; }

// The stream, the event and the words, made for the first upload in pieces (which so waits for what is on the context's stream).
bool ready(gh_ctx* ctx, bool* fresh) {
  if (!ctx->done_word || (ctx->pieces && __atomic_load_n(missed(ctx), __ATOMIC_RELAXED) >= (unsigned)kMisses)) ctx->no_pieces = true;
  if (ctx->pieces || ctx->no_pieces) return !ctx->no_pieces;
  int before = ctx->device;
  (void)hipGetDevice(&before);
  bool ok = hipSetDevice(ctx->device) == hipSuccess && hipMalloc(&ctx->piece_words, sizeof(Words)) == hipSuccess &&
            hipEventCreateWithFlags(&ctx->pieces_after, hipEventDisableTiming) == hipSuccess;
  hipStream_t tried[kTries] = {};   // kept until one is found, or the next would have the same queue
  for (int k = 0; k < kTries && ok && !ctx->pieces; k++) {
    ok = hipStreamCreateWithFlags(&tried[k], hipStreamNonBlocking) == hipSuccess;
    if (ok && side_by_side(ctx, tried[k])) std::swap(ctx->pieces, tried[k]);
  }
  for (hipStream_t s : tried)
    if (s) hipStreamDestroy(s);
  if ((ok = ok && ctx->pieces)) {
    hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(kWordCount), 0, ctx->stream, (Words*)ctx->piece_words);
    ok = hipGetLastError() == hipSuccess;
  }
  if (!ok) {
    (void)hipGetLastError();
    gh_drop_pieces(ctx);
    ctx->no_pieces = true;
  }
  (void)hipSetDevice(before);
  *fresh = ok;
  return ok;
}

}  // namespace

void gh_drop_pieces(gh_ctx* ctx) {
  if (ctx->pieces) {
    hipStreamSynchronize(ctx->pieces);
    hipStreamDestroy(ctx->pieces);
  }
  if (ctx->pieces_after) hipEventDestroy(ctx->pieces_after);
  if (ctx->piece_words) hipFree(ctx->piece_words);
  ctx->pieces = nullptr;
  ctx->pieces_after = nullptr;
  ctx->piece_words = nullptr;
}

extern "C" int gh_pieces_layers(const gh_cmd* cmds, int n) {
  const int pieces = cmds ? pieces_of(cmds, n) : 0;
  Layer layers[kHead];
  return pieces ? layers_of(cmds, n, pieces, layers, kUnits, [](uint64_t) { return false; }) : 0;
}

int gh_submit_pieces(gh_ctx* ctx, const gh_cmd* cmds, int n, int* rc) {
  if (ctx->capturing || ctx->ws_strict) return 0;
  const int pieces = pieces_of(cmds, n);
  if (!pieces) return 0;
  const gh_cmd& up = cmds[0];
  const int64_t bytes = up.dim[0], B = cmds[1].dim[0];
  if (!gh_in_pinned_host(ctx, up.ptr[1]) || !gh_in_pinned_host(ctx, up.ptr[1] + (uint64_t)bytes - 1) || gh_in_pinned_host(ctx, up.ptr[0])) return 0;
  if (getenv("GORGONIA_HIP_NO_PIECES")) return 0;   // tuning switch: the upload first
  Layer layers[kHead];
  const int head = layers_of(cmds, n, pieces, layers, ctx->cu_count, [&](uint64_t p) { return gh_in_pinned_host(ctx, p); });
  bool fresh = false;
  if (head == 0 || !ready(ctx, &fresh)) return 0;
  hipError_t e = hipSuccess;
  if (!ctx->idle || fresh) {   // what is on the stream may read what the copy writes
    e = hipEventRecord(ctx->pieces_after, ctx->stream);
    if (e == hipSuccess) e = hipStreamWaitEvent(ctx->pieces, ctx->pieces_after, 0);
  }
  ctx->idle = false;
  int64_t last[kPieces];   // a piece's last image, and the 16-byte words to its end
  Ends ends;
  for (int p = 0; p < pieces; p++) {
    last[p] = (B * (p + 1) + pieces - 1) / pieces;
    ends.n16[p] = (int)(p == pieces - 1 ? bytes / 16 : (last[p] * (bytes / B) + 15) / 16);
  }
  int64_t begin = kBegin + bytes / 200, give_up = kGiveUp + bytes / 100;
  const char* const ticks = getenv("GORGONIA_HIP_PIECES_TICKS");   // tests: the waits given up early, which counts where the copy is late as well
  const bool late = getenv("GORGONIA_HIP_PIECES_LATE");            // tests: the copy behind the layers
  if (ticks)
    for (int64_t* limit : {&begin, &give_up}) *limit = std::max<int64_t>(0, std::min<int64_t>(*limit, atoll(ticks)));
  unsigned* const misses = ticks && !late ? nullptr : missed(ctx);
  void* const dst = (void*)(uintptr_t)up.ptr[0];
  const u32x4* const src = (const u32x4*)(uintptr_t)up.ptr[1];
  const int tail_words = (int)(bytes % 16 / 4);
  const unsigned long long seq = ++ctx->piece_seq;
  auto copy = [&] {
    hipLaunchKernelGGL(k_copy_pieces, dim3(kCopiers), dim3(kThreads), 0, ctx->pieces, dst, src, ends, pieces, tail_words, (Words*)ctx->piece_words, seq);
    return hipGetLastError();
  };
  if (e == hipSuccess && !late) e = copy();
  for (int p = 0; p < pieces && e == hipSuccess && !*rc; p++) {
    const int64_t first = p ? last[p - 1] : 0;
    hipLaunchKernelGGL(k_await_piece, dim3(1), dim3(kThreads), 0, ctx->stream, dst, src, (int)bytes, p ? ends.n16[p - 1] : 0, ends.n16[p],
                       p == pieces - 1 ? tail_words : 0, (Words*)ctx->piece_words, p, seq, begin, give_up, misses);
    if ((e = hipGetLastError()) != hipSuccess) break;
    gh_cmd part[kHead];
    for (int k = 0; k < head; k++) {
      part[k] = cmds[k + 1];
      part[k].dim[0] = last[p] - first;
      part[k].ptr[0] += (uint64_t)(first * layers[k].in_bytes);
      part[k].ptr[layers[k].out] += (uint64_t)(first * layers[k].out_bytes);
    }
    // The copy has kCopiers compute units, so a kernel of one workgroup to each of the device's would run in two rounds: while
    // it is under way the layers are planned without them (8 x 3 x 416 x 416 615 / 599 us, of which a 64 -> 128 convolution of
    // 256 workgroups on two images 28 / 16).
    ctx->whole_images = B;
    ctx->whole_units = ctx->cu_count;
    if (p + 1 < pieces) ctx->cu_count = units_beside(ctx->cu_count);
    *rc = gh_submit_each(ctx, part, head, 1);
    ctx->cu_count = ctx->whole_units;
    ctx->whole_images = 0;
  }
  if (e == hipSuccess && late) {
    e = hipEventRecord(ctx->pieces_after, ctx->stream);
    if (e == hipSuccess) e = hipStreamWaitEvent(ctx->pieces, ctx->pieces_after, 0);
    if (e == hipSuccess) e = copy();
  }
  if (e != hipSuccess && !*rc) *rc = gh_check_hip(ctx, e, "upload in pieces");
  if (*rc) (void)hipStreamSynchronize(ctx->pieces);   // nothing of it is under way behind an error
  ctx->joint[GH_JOINT_PIECES].launches++;
  ctx->joint[GH_JOINT_PIECES].form = pieces * 100 + head;
  return head + 1;
}
