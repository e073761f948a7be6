// Context, memory, submission and graph entry points of libgorgonia_hip.so.
// Replaces what Gorgonia's cuda.Engine gets from gorgonia.org/cu's
// BatchedContext: context creation (cuda/external.go:112-170), queued copies,
// kernel launch (cuda/arith.go:62) and DoWork/Signal (cuda/external.go:223).
#include <immintrin.h>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstring>

#include <mutex>

#include "gh_internal.h"

int gh_fail(gh_ctx* ctx, int code, const std::string& msg) {
  if (ctx && ctx->err == GH_OK) {
    ctx->err = code;
    ctx->errmsg = msg;
  }
  return code;
}

// Scratch of gh_submit_noalloc: part of the library's device image, so it exists
// on every GPU the library runs on from load time to process exit and no call
// has to allocate it.  In host code this name only stands for the symbol; the
// per-device address comes from hipGetSymbolAddress (static_scratch below) and
// is the only thing ever handed to a kernel.
static __device__ __align__(256) unsigned char scratch[GH_NOALLOC_SCRATCH_BYTES];

static constexpr int kMaxDevices = 64;
static void* g_scratch_ptr[kMaxDevices] = {};   // address of `scratch` on device i; filled by gh_init

// Address of the static scratch on `device`, which must be current.  Resolved
// once per device (every GPU holds its own copy at its own address).
static hipError_t static_scratch(int device, void** out) {
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  static std::mutex mu;   // contexts may be opened from several host threads at once
  std::lock_guard<std::mutex> lock(mu);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_ptr[device] = p;
  }
  *out = g_scratch_ptr[device];
  return hipSuccess;
}

int gh_ws_short(gh_ctx* ctx, int64_t need) {
  if (!ctx->ws_strict) return GH_OK;
  return gh_fail(ctx, GH_EINVAL,
                 "gh_submit_noalloc: operator needs " + std::to_string(need) + " bytes of scratch, the fixed scratch holds " +
                     std::to_string((int64_t)GH_NOALLOC_SCRATCH_BYTES) + " (use gh_submit)");
}

int gh_check_hip(gh_ctx* ctx, hipError_t e, const char* what) {
  if (e == hipSuccess) return GH_OK;
  std::string m = std::string(what) + ": " + hipGetErrorString(e);
  return gh_fail(ctx, GH_EDEVICE, m);
}

bool gh_in_pinned_host(const gh_ctx* ctx, uint64_t p) {
  for (const auto& r : ctx->host_ranges)
    if (p >= r.first && p < r.second) return true;
  return false;
}

// The contexts' completion words: 64 of them, 64 bytes apart, in one pinned page that lives as long as the process
// (allocating one costs more than the rest of a small context).  A context beyond the 64th has none and waits in
// the runtime.
static std::mutex g_words_mu;
static unsigned char* g_words_page = nullptr;
static uint64_t g_words_used = 0;

static uint32_t* take_word() {
  std::lock_guard<std::mutex> lock(g_words_mu);
  if (!g_words_page && hipHostMalloc((void**)&g_words_page, 4096, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
    (void)hipGetLastError();
    g_words_page = nullptr;
  }
  if (!g_words_page || ~g_words_used == 0) return nullptr;
  const int i = __builtin_ctzll(~g_words_used);
  g_words_used |= 1ull << i;
  uint32_t* const w = (uint32_t*)(g_words_page + 64 * i);
  *w = 0;
  ((uint64_t*)w)[1] = 0;
  w[4] = 0;
  return w;
}
static void give_word(uint32_t* w) {
  if (!w) return;
  std::lock_guard<std::mutex> lock(g_words_mu);
  g_words_used &= ~(1ull << (((unsigned char*)w - g_words_page) / 64));
}

// The contexts' pages for k_bn_held.hip, 64 on a device, part of the library's device image as `scratch` is: zero from load
// time on, and again whenever no kernel runs.  A context beyond the 64th has none and runs those commands apart.
static constexpr int kBnPages = 64;
static __device__ __align__(256) unsigned char bn_pages[kBnPages][kBnHeldPage];
static std::mutex g_pages_mu;
static unsigned char* g_pages[kMaxDevices] = {};
static uint64_t g_pages_used[kMaxDevices] = {};

static void* take_page(int device) {   // `device` is current
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_pages_mu);
  if (!g_pages[device]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(bn_pages)) != hipSuccess) (void)hipGetLastError();
    g_pages[device] = (unsigned char*)p;
  }
  if (!g_pages[device] || ~g_pages_used[device] == 0) return nullptr;
  const int i = __builtin_ctzll(~g_pages_used[device]);
  g_pages_used[device] |= 1ull << i;
  return g_pages[device] + i * kBnHeldPage;
}
static void give_page(const gh_ctx* ctx) {
  if (!ctx->bn_page || ctx->err == GH_EDEVICE) return;   // (a kernel that did not end may have left it as it was)
  std::lock_guard<std::mutex> lock(g_pages_mu);
  g_pages_used[ctx->device] &= ~(1ull << (((unsigned char*)ctx->bn_page - g_pages[ctx->device]) / kBnHeldPage));
}

static void drop_ctx(gh_ctx* ctx) {
  give_word(ctx->done_word);   // nothing is in flight any more
  give_page(ctx);
  if (ctx->workspace) hipFree(ctx->workspace);
  if (ctx->slab_space) hipFree(ctx->slab_space);
  if (ctx->arena) hipFree(ctx->arena);
  gh_drop_pieces(ctx);
  hipStreamDestroy(ctx->stream);
  delete ctx;
}

extern "C" {

const char* gh_version(void) { return "gorgonia_hip 0.1 (gfx950)"; }

int gh_device_count(int* out) {
  if (!out) return GH_EINVAL;
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) { *out = 0; return GH_EDEVICE; }
  *out = n;
  return GH_OK;
}

int gh_init(int device, int64_t arena_bytes, gh_ctx** out) {
  if (!out || arena_bytes < 0) return GH_EINVAL;
  *out = nullptr;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || device < 0 || device >= n) return GH_EDEVICE;
  if (hipSetDevice(device) != hipSuccess) return GH_EDEVICE;
  gh_ctx* ctx = new gh_ctx();
  ctx->device = device;
  // Default priority only: mixed stream priorities are not used anywhere.
  if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
    delete ctx;
    return GH_EDEVICE;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) ctx->cu_count = prop.multiProcessorCount;
  // tuning override: the launchers plan for so many compute units, never for more than there are
  if (const char* units = getenv("GORGONIA_HIP_COMPUTE_UNITS")) ctx->cu_count = std::max(1, std::min(ctx->cu_count, atoi(units)));
  if (const char* sm = getenv("GORGONIA_HIP_SYNC")) {
    ctx->sync_block = strcmp(sm, "block") == 0;
    ctx->sync_spin = strcmp(sm, "spin") == 0;
  }
  ctx->done_word = take_word();
  if (arena_bytes > 0) {
    size_t free_b = 0, total_b = 0;
    hipMemGetInfo(&free_b, &total_b);
    if ((size_t)arena_bytes >= free_b) {  // cuda/external.go:159-161
      drop_ctx(ctx);
      return GH_EOOM;
    }
    if (hipMalloc(&ctx->arena, (size_t)arena_bytes) != hipSuccess) {
      (void)hipGetLastError();
      drop_ctx(ctx);
      return GH_EOOM;
    }
    ctx->arena_bytes = arena_bytes;
  }
  // Context-owned scratch: split-K partial sums, reduction partials, mirrored
  // filters.  Mandatory: the launchers index it without asking again.
  ctx->workspace_bytes = 64ll << 20;
  void* fixed = nullptr;
  if (hipMalloc(&ctx->workspace, (size_t)ctx->workspace_bytes) != hipSuccess ||
      static_scratch(device, &fixed) != hipSuccess) {
    (void)hipGetLastError();
    drop_ctx(ctx);
    return GH_EOOM;
  }
  ctx->bn_page = take_page(device);
  *out = ctx;
  return GH_OK;
}

int gh_close(gh_ctx* ctx) {
  if (!ctx) return GH_EINVAL;
  hipSetDevice(ctx->device);
  hipStreamSynchronize(ctx->stream);
  for (auto& g : ctx->graphs) {
    if (g.exec) hipGraphExecDestroy(g.exec);
    if (g.graph) hipGraphDestroy(g.graph);
  }
  for (auto& e : ctx->events)
    if (e) hipEventDestroy(e);
  drop_ctx(ctx);
  return GH_OK;
}

int gh_device_info(gh_ctx* ctx, gh_devinfo* out) {
  if (!ctx || !out) return GH_EINVAL;
  hipDeviceProp_t p;
  int rc = gh_check_hip(ctx, hipGetDeviceProperties(&p, ctx->device), "hipGetDeviceProperties");
  if (rc) return rc;
  memset(out, 0, sizeof(*out));
  out->wavefront_size = p.warpSize;
  out->max_threads_per_block = p.maxThreadsPerBlock;
  out->max_grid_x = p.maxGridSize[0];
  out->max_grid_y = p.maxGridSize[1];
  out->max_grid_z = p.maxGridSize[2];
  out->max_block_x = p.maxThreadsDim[0];
  out->max_block_y = p.maxThreadsDim[1];
  out->max_block_z = p.maxThreadsDim[2];
  out->compute_units = p.multiProcessorCount;
  out->lds_bytes_per_block = (int32_t)p.sharedMemPerBlock;
  size_t f = 0, t = 0;
  hipMemGetInfo(&f, &t);
  out->free_mem = (int64_t)f;
  out->total_mem = (int64_t)t;
  snprintf(out->arch, sizeof(out->arch), "%s", p.gcnArchName);
  return GH_OK;
}

gh_devptr gh_arena_base(gh_ctx* ctx) { return ctx ? (gh_devptr)(uintptr_t)ctx->arena : 0; }
int64_t gh_arena_size(gh_ctx* ctx) { return ctx ? ctx->arena_bytes : 0; }

int gh_malloc(gh_ctx* ctx, int64_t bytes, gh_devptr* out) {
  if (!ctx || !out || bytes <= 0) return GH_EINVAL;
  void* p = nullptr;
  if (hipMalloc(&p, (size_t)bytes) != hipSuccess) {
    (void)hipGetLastError();
    return GH_EOOM;
  }
  *out = (gh_devptr)(uintptr_t)p;
  return GH_OK;
}

int gh_free(gh_ctx* ctx, gh_devptr p) {
  if (!ctx) return GH_EINVAL;
  if (!p) return GH_OK;
  return gh_check_hip(ctx, hipFree((void*)(uintptr_t)p), "hipFree");
}

int gh_host_alloc(gh_ctx* ctx, int64_t bytes, void** out) {
  if (!ctx || !out || bytes <= 0) return GH_EINVAL;
  if (hipHostMalloc(out, (size_t)bytes, hipHostMallocCoherent) != hipSuccess) {
    (void)hipGetLastError();
    return GH_EOOM;
  }
  ctx->host_ranges.emplace_back((uint64_t)(uintptr_t)*out, (uint64_t)(uintptr_t)*out + (uint64_t)bytes);
  return GH_OK;
}

int gh_host_free(gh_ctx* ctx, void* p) {
  if (!ctx) return GH_EINVAL;
  if (!p) return GH_OK;
  for (size_t i = 0; i < ctx->host_ranges.size(); i++)
    if (ctx->host_ranges[i].first == (uint64_t)(uintptr_t)p) {
      ctx->host_ranges.erase(ctx->host_ranges.begin() + (long)i);
      break;
    }
  return gh_check_hip(ctx, hipHostFree(p), "hipHostFree");
}

int gh_memcpy_h2d(gh_ctx* ctx, gh_devptr dst, const void* src, int64_t bytes) {
  if (!ctx || bytes < 0 || (bytes > 0 && (!dst || !src))) return GH_EINVAL;
  if (ctx->err) return ctx->err;
  if (bytes == 0) return GH_OK;
  ctx->idle = false;
  if (!gh_in_pinned_host(ctx, (uint64_t)(uintptr_t)src)) ctx->runtime_wait = true;
  return gh_check_hip(ctx,
                      hipMemcpyAsync((void*)(uintptr_t)dst, src, (size_t)bytes,
                                     hipMemcpyHostToDevice, ctx->stream),
                      "hipMemcpyAsync(H2D)");
}

int gh_memcpy_d2h(gh_ctx* ctx, void* dst, gh_devptr src, int64_t bytes) {
  if (!ctx || bytes < 0 || (bytes > 0 && (!dst || !src))) return GH_EINVAL;
  if (ctx->err) return ctx->err;
  if (bytes == 0) return GH_OK;
  ctx->idle = false;
  if (!gh_in_pinned_host(ctx, (uint64_t)(uintptr_t)dst)) ctx->runtime_wait = true;
  return gh_check_hip(ctx,
                      hipMemcpyAsync(dst, (const void*)(uintptr_t)src, (size_t)bytes,
                                     hipMemcpyDeviceToHost, ctx->stream),
                      "hipMemcpyAsync(D2H)");
}

// Copies done by a kernel: a kernel node costs less inside a captured graph than
// a copy-engine node, and either side may be pinned host memory (results staged
// out to the host, inputs staged in from it over PCIe).
__global__ __launch_bounds__(256) void k_copy_words(uint32_t* __restrict__ dst,
                                                    const uint32_t* __restrict__ src, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}
// 16 bytes per lane, two in flight; the tail (< 16 bytes, a multiple of 4) goes word by word.
__global__ __launch_bounds__(256) void k_copy_vec(uint4* __restrict__ dst, const uint4* __restrict__ src,
                                                  int64_t n16, int64_t tail_words) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (; i + stride < n16; i += 2 * stride) {
    const uint4 a = src[i], b = src[i + stride];
    dst[i] = a;
    dst[i + stride] = b;
  }
  if (i < n16) dst[i] = src[i];
  if (blockIdx.x == 0 && (int64_t)threadIdx.x < tail_words)
    ((uint32_t*)(dst + n16))[threadIdx.x] = ((const uint32_t*)(src + n16))[threadIdx.x];
}

static constexpr int64_t kKernelCopyLimit = 16 << 20;   // between device buffers
// Workgroups of a copy out of pinned host memory.  The bus needs few requests in flight and serves them the better
// the fewer workgroups interleave theirs: 16.6 MB take 355 us with 1024 workgroups, 308 with 64 to 128 (the copy
// engine: 301, and 5 us more for the kernel behind it to see its signal), 2 MB 62 and 51.
static constexpr int64_t kHostCopyBlocks = 96;

int gh_memcpy_d2d(gh_ctx* ctx, gh_devptr dst, gh_devptr src, int64_t bytes) {
  if (!ctx || bytes < 0 || (bytes > 0 && (!dst || !src))) return GH_EINVAL;
  if (ctx->err) return ctx->err;
  if (bytes == 0) return GH_OK;
  ctx->idle = false;
  const bool from_host = gh_in_pinned_host(ctx, src);
  if ((from_host || bytes <= kKernelCopyLimit) && ((dst | src | (uint64_t)bytes) & 3) == 0) {
    if (((dst | src) & 15) == 0 && bytes >= 4096) {
      const int64_t n16 = bytes / 16;
      int64_t blocks = (n16 + 511) / 512;
      const int64_t most = from_host ? kHostCopyBlocks : 1024;
      if (blocks > most) blocks = most;
      hipLaunchKernelGGL(k_copy_vec, dim3((int)blocks), dim3(256), 0, ctx->stream, (uint4*)(uintptr_t)dst,
                         (const uint4*)(uintptr_t)src, n16, (bytes % 16) / 4);
    } else {
      const int64_t n = bytes / 4;
      int64_t blocks = (n + 255) / 256;
      if (blocks > 1024) blocks = 1024;
      hipLaunchKernelGGL(k_copy_words, dim3((int)blocks), dim3(256), 0, ctx->stream,
                         (uint32_t*)(uintptr_t)dst, (const uint32_t*)(uintptr_t)src, n);
    }
    return gh_check_hip(ctx, hipGetLastError(), "copy launch");
  }
  return gh_check_hip(ctx,
                      hipMemcpyAsync((void*)(uintptr_t)dst, (const void*)(uintptr_t)src,
                                     (size_t)bytes, hipMemcpyDefault, ctx->stream),
                      "hipMemcpyAsync(D2D)");
}

// A value on its way from pageable memory: the host copies it into pinned memory and says after each `say` bytes how far it
// is, and the workgroups of one kernel, launched in front of that, read what is there.  Bound: the bus (56 GB/s) and the
// first bytes' way.  us with the wait: 392 KB 20 (24 copied, then moved), 2 MB 54 (70 in pieces of 512 KB, whose launches cost
// some 4 us each until their first bytes came), 4 MB 92 (123), 8 MB 173 (217), 16 MB 320 (385); the bus alone 7, 37, 74, 150
// and 296.  More workgroups read the host's word and the value against each other: 4 MB 97 with 96 of them, 108 with 192.
//
// A workgroup has ranges of kRange bytes and waits for the host's word to pass the end of the next one.  It gives up after
// kGiveUp of the device's clock: the host, which never waits for the kernel, then took longer than three quarters of that by
// its own clock (it looks at it before the launch and behind its last word) and enqueues an ordinary copy of everything.
static constexpr int64_t kRange = 16384, kFollowers = 32;
static constexpr int64_t kGiveUp = 400000;   // ticks of 10 ns (GORGONIA_HIP_STAGED_TICKS: fewer)
// A long value is copied in parts that memcpy stores past the host's caches: 16 MB 320 us, 358 in parts of 128 KB (which are
// quicker up to 12 MB: 253 for 261).
static int64_t say_after(int64_t bytes) { return bytes > (14 << 20) ? 1 << 20 : 128 << 10; }
__global__ __launch_bounds__(256) void k_copy_following(uint4* __restrict__ dst, const uint4* src, int64_t n16, int64_t tail_words, const uint64_t* said,
                                                        uint64_t base, int64_t give_up) {
  __shared__ uint64_t word;
  constexpr int kRange16 = kRange / 16;
  const int64_t t0 = wall_clock64();
  uint64_t known = base;
  bool there = true;
  // waits for `bytes` of the value, in all threads
  auto wait = [&](int64_t bytes) {
    if ((int64_t)(known - base) >= bytes) return;
    __syncthreads();
    if (threadIdx.x == 0) {
      uint64_t now;
      while ((int64_t)((now = __hip_atomic_load(said, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM)) - base) < bytes && (int64_t)wall_clock64() - t0 < give_up)
        __builtin_amdgcn_s_sleep(8);
      word = now;
    }
    __syncthreads();
    known = word;
    there = (int64_t)(known - base) >= bytes;
  };
  const int64_t ranges = (n16 + kRange16 - 1) / kRange16;
  for (int64_t r = blockIdx.x; r < ranges; r += gridDim.x) {
    const int64_t from = r * kRange16, to = from + kRange16 < n16 ? from + kRange16 : n16;
    wait(to * 16);
    if (!there) return;
    int64_t i = from + threadIdx.x;
    if (to - from == kRange16) {
      const uint4 a = src[i], b = src[i + 256], c = src[i + 512], d = src[i + 768];
      dst[i] = a;
      dst[i + 256] = b;
      dst[i + 512] = c;
      dst[i + 768] = d;
    } else {
      for (; i < to; i += 256) dst[i] = src[i];
    }
  }
  if (blockIdx.x == 0 && tail_words) {
    wait(n16 * 16 + tail_words * 4);
    if (there && (int64_t)threadIdx.x < tail_words) ((uint32_t*)(dst + n16))[threadIdx.x] = ((const uint32_t*)(src + n16))[threadIdx.x];
  }
}

int gh_memcpy_staged(gh_ctx* ctx, gh_devptr dst, void* stage, const void* src, int64_t bytes) {
  if (!ctx || bytes < 0 || (bytes > 0 && (!dst || !stage || !src))) return GH_EINVAL;
  if (ctx->err) return ctx->err;
  if (bytes == 0) return GH_OK;
  const uint64_t from = (uint64_t)(uintptr_t)stage;
  if (!gh_in_pinned_host(ctx, from) || !gh_in_pinned_host(ctx, from + (uint64_t)bytes - 1)) return gh_fail(ctx, GH_EINVAL, "gh_memcpy_staged: the staging memory is not of gh_host_alloc");
  if (!ctx->done_word || ctx->capturing || bytes < GH_STAGED_FROM || ((dst | from) & 15) || (bytes & 3)) {
    memcpy(stage, src, (size_t)bytes);
    return gh_memcpy_d2d(ctx, dst, from, bytes);
  }
  ctx->idle = false;
  uint64_t* const said = (uint64_t*)ctx->done_word + 1;   // behind the completion word, on its cache line
  const uint64_t base = *said;
  const int64_t ranges = (bytes / 16 + kRange / 16 - 1) / (kRange / 16), say = say_after(bytes);
  int64_t give_up = kGiveUp;
  if (const char* ticks = getenv("GORGONIA_HIP_STAGED_TICKS")) give_up = std::max<int64_t>(0, std::min<int64_t>(kGiveUp, atoll(ticks)));
  const auto before = std::chrono::steady_clock::now();
  hipLaunchKernelGGL(k_copy_following, dim3((unsigned)std::min(ranges, kFollowers)), dim3(256), 0, ctx->stream, (uint4*)(uintptr_t)dst, (const uint4*)stage, bytes / 16,
                     (bytes % 16) / 4, said, base, give_up);
  const hipError_t e = hipGetLastError();
  for (int64_t at = 0; at < bytes; at += say) {
    const int64_t len = std::min(say, bytes - at);
    memcpy((char*)stage + at, (const char*)src + at, (size_t)len);
    _mm_sfence();   // memcpy may have stored past the cache
    __atomic_store_n(said, base + (uint64_t)(at + len), __ATOMIC_RELEASE);
  }
  if (e != hipSuccess) return gh_check_hip(ctx, e, "copy launch");
  const auto took = std::chrono::steady_clock::now() - before;
  if (took >= std::chrono::nanoseconds(give_up * 10 * 3 / 4)) return gh_memcpy_d2d(ctx, dst, from, bytes);
  return GH_OK;
}

static int dispatch(gh_ctx* ctx, const gh_cmd& c) {
  // the streaming kernels keep their own account of what they touch; everything else marks its
  // operands as recently used (sizes unknown here: by start address), so that an elementwise
  // kernel behind a product or a convolution reads the result as the cache-resident data it is
  if (c.opcode != GH_OP_ELEM_BIN && c.opcode != GH_OP_ELEM_UNARY && c.opcode != GH_OP_BCAST_BIN && c.opcode != GH_OP_NOP)
    for (uint64_t p : c.ptr) ctx->llc.touch(p, 0, false);
  switch (c.opcode) {
    case GH_OP_NOP: return GH_OK;
    case GH_OP_ELEM_BIN: return gh_launch_elem_bin(ctx, c);
    case GH_OP_ELEM_UNARY: return gh_launch_elem_unary(ctx, c);
    case GH_OP_BCAST_BIN: return gh_launch_bcast_bin(ctx, c);
    case GH_OP_MEMCPY_D2D: return gh_memcpy_d2d(ctx, c.ptr[0], c.ptr[1], c.dim[0]);
    case GH_OP_GEMM: return gh_launch_gemm(ctx, c);
    case GH_OP_GEMV: return gh_launch_gemv(ctx, c);
    case GH_OP_OUTER: return gh_launch_outer(ctx, c);
    case GH_OP_CONV2D: return gh_launch_conv2d(ctx, c);
    case GH_OP_MAXPOOL2D: return gh_launch_maxpool2d(ctx, c);
    case GH_OP_BN_INFER: return gh_launch_bn_infer(ctx, c);
    case GH_OP_RELU: return gh_launch_relu(ctx, c);
    case GH_OP_LEAKY_RELU: return gh_launch_leaky_relu(ctx, c);
    case GH_OP_SOFTMAX: return gh_launch_softmax(ctx, c);
    case GH_OP_HAS_NAN:
    case GH_OP_HAS_INF: return gh_launch_has_nan_inf(ctx, c);
    case GH_OP_FILL: return gh_launch_fill(ctx, c);
    case GH_OP_MAXPOOL2D_BWD: return gh_launch_maxpool2d_bwd(ctx, c);
    case GH_OP_CONV2D_BWD_DATA: return gh_launch_conv2d_bwd_data(ctx, c);
    case GH_OP_CONV2D_BWD_FILTER: return gh_launch_conv2d_bwd_filter(ctx, c);
    case GH_OP_BN_TRAIN: return gh_launch_bn_train(ctx, c);
    case GH_OP_BN_BWD: return gh_launch_bn_bwd(ctx, c);
    case GH_OP_SOFTMAX_BWD: return gh_launch_softmax_bwd(ctx, c);
    case GH_OP_SOLVER_STEP: return gh_launch_solver_step(ctx, c);
    case GH_OP_RAND_UNIFORM: return gh_launch_rand_uniform(ctx, c);
    case GH_OP_DROPOUT: return gh_launch_dropout(ctx, c);
    case GH_OP_DROPOUT_BWD: return gh_launch_dropout_bwd(ctx, c);
    case GH_OP_RELU_BWD: return gh_launch_relu_bwd(ctx, c);
  }
  return GH_ENOFUNC;
}

int gh_validate(const gh_cmd* cmds, int n, char* msg, int msg_len) {
  if (n < 0 || (n > 0 && !cmds)) return GH_EINVAL;
  for (int i = 0; i < n; i++) {
    std::string m;
    int rc = gh_validate_cmd(cmds[i], m);
    if (rc) {
      if (msg && msg_len > 0) snprintf(msg, (size_t)msg_len, "cmd %d: %s", i, m.c_str());
      return rc;
    }
  }
  if (msg && msg_len > 0) msg[0] = 0;
  return GH_OK;
}

int gh_submit_each(gh_ctx* ctx, const gh_cmd* cmds, int n, int before) {
  ctx->idle = false;
  for (int i = 0; i < n; i++) {
    std::string m;
    int rc = gh_validate_cmd(cmds[i], m);
    if (rc) return gh_fail(ctx, rc, "cmd " + std::to_string(before + i) + ": " + m);
    // solver steps take the sums that wait along where they are their gradients
    if (ctx->pending && cmds[i].opcode == GH_OP_SOLVER_STEP) {
      const int steps = gh_solver_run_length(cmds + i, n - i);
      const bool copy = gh_solver_copy_rides(cmds + i, steps, n - i);
      bool valid = true;
      for (int j = 1; j < steps + copy; j++) valid = valid && gh_validate_cmd(cmds[i + j], m) == GH_OK;
      if (valid && (rc = gh_try_launch_solver_sums(ctx, cmds + i, steps, copy)) >= 0) {
        if (rc) return rc;
        i += steps + copy - 1;
        continue;
      }
    }
    if ((rc = gh_flush_sums_before(ctx, cmds[i]))) return rc;
    // a run of solver steps with the same settings (a model's weight tensors) is one launch, and so is a run of
    // elementwise commands on tensors of one size
    const int solver = gh_solver_run_length(cmds + i, n - i);
    const bool copy = solver && gh_solver_copy_rides(cmds + i, solver, n - i);
    const int run = solver > 1 || copy ? solver + copy : gh_chain_length(cmds + i, n - i);
    if (run > 1) {
      for (int j = 1; j < run; j++) {
        rc = gh_validate_cmd(cmds[i + j], m);
        if (rc) return gh_fail(ctx, rc, "cmd " + std::to_string(before + i + j) + ": " + m);
        if ((rc = gh_flush_sums_before(ctx, cmds[i + j]))) return rc;
      }
      rc = solver ? gh_launch_solver_steps(ctx, cmds + i, solver, copy) : gh_launch_chain(ctx, cmds + i, run);
      if (rc) return rc;
      i += run - 1;
      continue;
    }
    // a filter gradient and the image gradient beside it, in one launch where a kernel has both
    if (gh_gradient_pair(cmds + i, n - i)) {
      if ((rc = gh_flush_sums_before(ctx, cmds[i + 1]))) return rc;
      const bool first = cmds[i].opcode == GH_OP_CONV2D_BWD_FILTER;
      gh_unpool unpool;
      const int behind = gh_unpool_follows(cmds + i, n - i, &unpool);
      for (int j = 0; j < behind; j++)
        if ((rc = gh_flush_sums_before(ctx, cmds[i + 2 + j]))) return rc;
      if (behind) ctx->unpool = unpool;
      ctx->hold_filter = true;
      rc = dispatch(ctx, cmds[first ? i : i + 1]);
      ctx->hold_filter = false;
      if (!rc) rc = dispatch(ctx, cmds[first ? i + 1 : i]);
      const int alone = gh_launch_held(ctx);
      const bool unpooled = ctx->unpool.done;
      ctx->unpool = gh_unpool{};
      if (rc || alone) return rc ? rc : alone;
      for (int j = 0; unpooled && j < behind; j++, i++)
        for (uint64_t p : cmds[i + 2].ptr) ctx->llc.touch(p, 0, false);
      i++;
      continue;
    }
    // and so with a dense layer's two gradients
    if (gh_gemm_gradient_pair(cmds + i, n - i)) {
      if ((rc = gh_flush_sums_before(ctx, cmds[i + 1]))) return rc;
      const bool rectified = gh_rectify_gradient_follows(cmds + i, n - i);
      if (rectified && (rc = gh_flush_sums_before(ctx, cmds[i + 2]))) return rc;
      if ((rc = gh_try_launch_gemm_gradients(ctx, cmds + i, rectified)) >= 0) {
        if (rc) return rc;
        i += 1 + rectified;
        continue;
      }
    }
    // a product and its Rectify
    if (gh_rectify_follows(cmds + i, n - i)) {
      if ((rc = gh_flush_sums_before(ctx, cmds[i + 1]))) return rc;
      if ((rc = gh_try_launch_gemm_rectify(ctx, cmds + i)) >= 0) {
        if (rc) return rc;
        i++;
        continue;
      }
    }
    // a SoftMax, and the scaled tensor and the gradient behind it
    if (gh_softmax_gradient_follows(cmds + i, n - i)) {
      for (int j = 1; j < 3; j++)
        if ((rc = gh_flush_sums_before(ctx, cmds[i + j]))) return rc;
      if ((rc = (cmds[i].opcode == GH_OP_GEMM ? gh_try_launch_gemm_softmax_gradient : gh_try_launch_softmax_gradient)(ctx, cmds + i)) >= 0) {
        if (rc) return rc;
        i += 2;
        continue;
      }
    }
    // two commands of which the second reads what the first writes are one launch where a kernel takes both
    const bool held = gh_bn_held_pair(ctx, cmds + i, n - i), pair = held || gh_is_pair(cmds + i, n - i);
    if (cmds[i].opcode == GH_OP_MAXPOOL2D_BWD && (cmds[i].flags & GH_FLAG_BN_REMADE)) {
      if (!gh_bn_remade_follows(cmds + i, n - i)) return gh_fail(ctx, GH_EINVAL, "cmd " + std::to_string(before + i) + ": maxpool2d gradient: the batch normalisation's gradient does not follow");
      if ((rc = gh_flush_sums_before(ctx, cmds[i + 1]))) return rc;
      if (!held && (rc = gh_launch_bn_remake(ctx, cmds + i))) return rc;
    }
    if (pair && (rc = gh_flush_sums_before(ctx, cmds[i + 1]))) return rc;
    rc = held ? gh_launch_bn_held_pair(ctx, cmds + i) : pair ? gh_launch_pair(ctx, cmds + i) : dispatch(ctx, cmds[i]);
    if (rc) return rc;
    if (pair) i++;
  }
  return GH_OK;
}

// The memory for slabs whose sums wait: made for the first submission of several commands with a filter gradient among them
// (none while a graph is captured: the sums are then launched where they stand).
static bool slab_space(gh_ctx* ctx, const gh_cmd* cmds, int n) {
  if (ctx->slab_space || ctx->no_slab_space || ctx->capturing) return ctx->slab_space;
  bool any = false;
  for (int i = 0; i < n; i++) any = any || cmds[i].opcode == GH_OP_CONV2D_BWD_FILTER;
  if (!any) return false;
  int before = ctx->device;
  (void)hipGetDevice(&before);
  if (hipSetDevice(ctx->device) != hipSuccess || hipMalloc(&ctx->slab_space, (size_t)kSlabSpace) != hipSuccess) {
    (void)hipGetLastError();
    ctx->slab_space = nullptr;
    ctx->no_slab_space = true;
  }
  (void)hipSetDevice(before);
  return ctx->slab_space;
}

// Sums of filter-gradient slabs may wait for the commands behind them (k_slab_sums.hip); none waits past the submission.
static int submit_cmds(gh_ctx* ctx, const gh_cmd* cmds, int n) {
  ctx->defer_sums = n > 1 && !ctx->ws_strict && slab_space(ctx, cmds, n);
  int rc = GH_OK;
  const int ahead = gh_submit_pieces(ctx, cmds, n, &rc);
  if (!rc) rc = gh_submit_each(ctx, cmds + ahead, n - ahead, ahead);
  ctx->defer_sums = false;
  const int late = gh_flush_sums(ctx);
  return rc ? rc : late;
}

int64_t gh_joint_launches(const gh_ctx* ctx, int kind, int64_t* form) {
  if (!ctx || kind < 0 || kind >= GH_JOINT__COUNT) return -1;
  if (form) *form = ctx->joint[kind].form;
  return ctx->joint[kind].launches;
}

int gh_submit(gh_ctx* ctx, const gh_cmd* cmds, int n) {
  if (!ctx || n < 0 || (n > 0 && !cmds)) return GH_EINVAL;
  if (ctx->err) return ctx->err;
  return submit_cmds(ctx, cmds, n);
}

int gh_submit_noalloc(gh_ctx* ctx, const gh_cmd* cmds, int n) {
  if (!ctx || n < 0 || (n > 0 && !cmds)) return GH_EINVAL;
  if (ctx->err) return ctx->err;
  void* fixed = ctx->device >= 0 && ctx->device < kMaxDevices ? g_scratch_ptr[ctx->device] : nullptr;
  if (!fixed) return gh_fail(ctx, GH_ESTATE, "gh_submit_noalloc: the fixed scratch was not resolved on this device");
  // Same launchers, same plans: only the scratch they index changes, and a plan
  // that would not fit it is refused instead of shrunk (gh_ws_short).  Nothing
  // in the scratch has to start at zero: every slab and partial is written
  // before it is read.
  void* const keep = ctx->workspace;
  const int64_t keep_bytes = ctx->workspace_bytes;
  ctx->workspace = fixed;
  ctx->workspace_bytes = GH_NOALLOC_SCRATCH_BYTES;
  ctx->ws_strict = true;
  const int rc = submit_cmds(ctx, cmds, n);
  ctx->ws_strict = false;
  ctx->workspace = keep;
  ctx->workspace_bytes = keep_bytes;
  return rc;
}

// How long gh_sync polls its word before it leaves the wait to the runtime (and the core to others).
static constexpr auto kPollFor = std::chrono::microseconds(2000);
// The runtime frees what it keeps per launch when it is asked to wait: every so many waits it is.  At
// every 32nd the allocations of a new tape machine paid for the backlog (3.6 -> 5 to 6.8 ms for 37 tensors);
// at every 16th they do not, and the 3 us more of one wait in 16 cannot be told from noise.
static constexpr uint32_t kRuntimeWaitEvery = 16;

// The completion word of gh_sync.  What the kernels in front have stored is visible to this one when it begins, and its release
// takes that along to the host: results lie in coherent pinned memory, which no cache of the device holds back.  Bound: a
// launch behind the last kernel, 1.3 us; the runtime's own write to a word (hipStreamWriteValue32) sets a barrier of its own
// in front and begins 5 us after that kernel's end.  us with the runtime's / with this: 777 x 1543 x 1021 in float64 53.6 / 52.4,
// a convnet's forward step of four kernels 47.1 / 45.6, its training step 187.8 / 185.6.
__global__ void k_say_done(uint32_t* word, uint32_t seq) { __hip_atomic_store(word, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM); }

static bool say_done(gh_ctx* ctx, uint32_t seq) {
  hipLaunchKernelGGL(k_say_done, dim3(1), dim3(1), 0, ctx->stream, ctx->done_word, seq);
  return hipGetLastError() == hipSuccess;
}

// Waits for everything on the context's stream.  The runtime's own wait puts a barrier packet with a
// signal behind the last kernel and, where the work takes longer than some tens of microseconds, sleeps
// until an interrupt: one small kernel and hipStreamSynchronize take 11.3 us, ten take 47.  Here a
// kernel writes a sequence number to a pinned word behind the last one and the caller's thread polls
// that word (8.5 and 31 us where the runtime wrote it).  An idle stream is not waited for at all (a tape machine's run asks twice).
int gh_sync(gh_ctx* ctx) {
  if (!ctx) return GH_EINVAL;
  if (ctx->capturing) return gh_fail(ctx, GH_ESTATE, "gh_sync during graph capture");
  if (ctx->idle) return ctx->err;
  bool seen = false;
  const uint32_t seq = ctx->done_seq + 1;
  if (ctx->done_word && !ctx->sync_block && !ctx->runtime_wait && !ctx->err && seq % kRuntimeWaitEvery != 0 &&
      say_done(ctx, seq)) {
    const auto until = std::chrono::steady_clock::now() + kPollFor;
    for (int spins = 1; !(seen = __atomic_load_n(ctx->done_word, __ATOMIC_ACQUIRE) == seq); spins++) {
      _mm_pause();
      if (spins % 64 == 0 && std::chrono::steady_clock::now() > until) break;
    }
  }
  ctx->done_seq = seq;
  if (!seen) {
    hipError_t e;
    if (ctx->sync_spin) {   // the thread keeps its core however long it takes
      while ((e = hipStreamQuery(ctx->stream)) == hipErrorNotReady) {
      }
    } else {
      e = hipStreamSynchronize(ctx->stream);
    }
    if (e != hipSuccess) {
      gh_check_hip(ctx, e, "hipStreamSynchronize");
      return ctx->err;
    }
  }
  ctx->idle = true;
  ctx->runtime_wait = false;
  return ctx->err;
}

int gh_graph_begin(gh_ctx* ctx) {
  if (!ctx) return GH_EINVAL;
  if (ctx->err) return ctx->err;
  if (ctx->capturing) return gh_fail(ctx, GH_ESTATE, "graph capture already active");
  int rc = gh_check_hip(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal),
                        "hipStreamBeginCapture");
  if (rc) return rc;
  ctx->capturing = true;
  return GH_OK;
}

int gh_graph_end(gh_ctx* ctx, int* graph_id) {
  if (!ctx || !graph_id) return GH_EINVAL;
  if (!ctx->capturing) return gh_fail(ctx, GH_ESTATE, "no graph capture active");
  ctx->capturing = false;
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(ctx->stream, &g);
  if (e != hipSuccess) return gh_check_hip(ctx, e, "hipStreamEndCapture");
  if (ctx->err) {  // a submit failed while capturing: drop the graph
    if (g) hipGraphDestroy(g);
    return ctx->err;
  }
  hipGraphExec_t ex = nullptr;
  e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    hipGraphDestroy(g);
    return gh_check_hip(ctx, e, "hipGraphInstantiate");
  }
  int id = -1;
  for (size_t i = 0; i < ctx->graphs.size(); i++)
    if (!ctx->graphs[i].used) { id = (int)i; break; }
  if (id < 0) {
    ctx->graphs.emplace_back();
    id = (int)ctx->graphs.size() - 1;
  }
  ctx->graphs[id].graph = g;
  ctx->graphs[id].exec = ex;
  ctx->graphs[id].used = true;
  *graph_id = id;
  return GH_OK;
}

int gh_graph_launch(gh_ctx* ctx, int id) {
  if (!ctx) return GH_EINVAL;
  if (ctx->err) return ctx->err;
  if (id < 0 || id >= (int)ctx->graphs.size() || !ctx->graphs[id].used)
    return gh_fail(ctx, GH_EINVAL, "unknown graph id");
  ctx->idle = false;
  return gh_check_hip(ctx, hipGraphLaunch(ctx->graphs[id].exec, ctx->stream), "hipGraphLaunch");
}

int gh_graph_destroy(gh_ctx* ctx, int id) {
  if (!ctx) return GH_EINVAL;
  if (id < 0 || id >= (int)ctx->graphs.size() || !ctx->graphs[id].used) return GH_EINVAL;
  hipStreamSynchronize(ctx->stream);
  hipGraphExecDestroy(ctx->graphs[id].exec);
  hipGraphDestroy(ctx->graphs[id].graph);
  ctx->graphs[id] = gh_graph_slot();
  return GH_OK;
}

int gh_last_error(gh_ctx* ctx, char* buf, int len) {
  if (!ctx) return GH_EINVAL;
  if (buf && len > 0) snprintf(buf, (size_t)len, "%s", ctx->errmsg.c_str());
  return ctx->err;
}

int gh_clear_error(gh_ctx* ctx) {
  if (!ctx) return GH_EINVAL;
  ctx->err = GH_OK;
  ctx->errmsg.clear();
  (void)hipGetLastError();
  return GH_OK;
}

int gh_event_record(gh_ctx* ctx, int slot) {
  if (!ctx || slot < 0 || slot >= 64) return GH_EINVAL;
  if (ctx->err) return ctx->err;
  if (!ctx->events[slot]) {
    int rc = gh_check_hip(ctx, hipEventCreate(&ctx->events[slot]), "hipEventCreate");
    if (rc) return rc;
  }
  ctx->idle = false;
  return gh_check_hip(ctx, hipEventRecord(ctx->events[slot], ctx->stream), "hipEventRecord");
}

int gh_event_elapsed_ms(gh_ctx* ctx, int start, int stop, float* ms) {
  if (!ctx || !ms || start < 0 || start >= 64 || stop < 0 || stop >= 64) return GH_EINVAL;
  if (!ctx->events[start] || !ctx->events[stop]) return GH_ESTATE;
  int rc = gh_check_hip(ctx, hipEventSynchronize(ctx->events[stop]), "hipEventSynchronize");
  if (rc) return rc;
  return gh_check_hip(ctx, hipEventElapsedTime(ms, ctx->events[start], ctx->events[stop]),
                      "hipEventElapsedTime");
}

}  // extern "C"
