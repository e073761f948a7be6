// Batch statistics and the 2x2 pooling behind them in one launch, and their gradients in another.
//
// Training mode needs a channel's mean before its deviations and both before a value can be written, and a launch for each
// of these and for the pooling; the gradient needs two sums before it can be written.  Here C channels times G workgroups of
// up to 1024 threads, one workgroup on a compute unit, have a share of a channel each.  They pass their sums to each other
// through memory and wait for each other's.  A 22 MB tensor fits the chip's registers (128 MB): between its sums and the
// values it writes the gradient keeps what it has read, the forward its values between its two passes.
//
// Nobody waits for a workgroup that has not begun: a share belongs to the workgroup that claims it, its own at first, and one
// that has asked kPolls times for the missing sums claims shares that nobody has begun.  So a share that is waited for is being
// worked on, by a workgroup that waits for nothing meanwhile, however few of them the chip has room for; one that begins when
// its share is taken leaves.  The sums are added in the order of the shares, to the same bits whoever brings them.
// us of a forward pair in one context and in each of two, three and four at once, 8 x 16 x 208 x 208: 20, 35, 57 and 74 (the
// commands apart 33, 47, 61 and 77; waiting for every workgroup, with the missing shares added up again by all: 20, 61, 8900 and
// 13800); a training step of the four-block network 430, 660, 910 and 1310 (apart 500, 750, 990 and 1460).
//
// Bound: HBM and the caches for large planes, the launch and the waits (some 1.5 us each) for small ones.  us, four launches
// or three / one, forward and gradient: 8 x 16 x 208 x 208 30.9 / 19.6 and 33.8 / 22.5 (4.2 TB/s of the 94 MB that the
// gradient moves), 8 x 32 x 104 x 104 20.5 / 12.6 and 22.9 / 13.1, 8 x 128 x 26 x 26 14.2 / 9.8 and 13.4 / 7.7,
// 8 x 16 x 207 x 207 (single loads) 46.6 / 20.9 and 47.3 / 25.9, 2 x 3 x 4 x 4 12.1 / 8.9 and 10.0 / 5.7.  (The forward as the
// gradient is, its values kept as the pooling's windows lie: 14.8, 9.9 and 7.3, and other sums.)
// Where the normalised values are read by the pooling and its gradient only (GH_FLAG_BN_REMADE, a training step), the forward
// leaves them out and the gradient makes them again from what it reads anyway, and passes its own middle result on in registers:
// 44 MB less of 50 and 94 for 8 x 16 x 208 x 208.  In the step of the four-block network, traced, 21.3 -> 18.8 and 22.9 -> 18.1,
// 8 x 32 x 104 x 104 13.0 -> 11.9 and 14.5 -> 11.8, 8 x 64 x 52 x 52 10.0 -> 9.1 and 10.6 -> 8.8, 8 x 128 x 26 x 26 9.7 -> 9.4 and
// 8.1 -> 7.3; the step 408.6 -> 393.5.  What is left is the launch, the first loads and the two waits.
#include <algorithm>
#include <cfloat>

#include "gh_internal.h"

namespace {

constexpr int kThreads = 1024;
constexpr int kHeld = 6;   // groups of four values that a thread of the forward keeps
constexpr int kPolls = 8;   // some 5 us (GORGONIA_HIP_BN_POLLS: another number; 0: every second workgroup is taken to come too late)
constexpr int kGiveUp = 1 << 22;   // polls, seconds: never reached; the sums are NaN then
typedef unsigned long long u64;

__device__ __forceinline__ float relu_of(float v) { return v * (v >= 0.0f ? 1.0f : 0.0f); }
__device__ __forceinline__ float relu_mask(float v) { return v >= 0.0f ? 1.0f : 0.0f; }

template <int K> struct Vec { typedef float T __attribute__((ext_vector_type(K))); };

// B images of C planes of H x W; a unit is two rows of COLS columns (a last row or column alone where the size is odd),
// a workgroup has `per` of a channel's units.
struct Planes {
  int H, W, uw, plane_units, units, per, C, G;
  int polls;   // how often a workgroup asks for the others' sums before it claims shares
};

// Two rows of COLS values; EDGES: H or W is odd, or rows lie where only single values can be loaded.
template <int COLS, bool EDGES>
struct Unit {
  int b, uy, ux;
  bool right, below;   // the second column, the second row exist
  __device__ __forceinline__ Unit(const Planes& g, int u) {
    b = u / g.plane_units;
    const int r = u - b * g.plane_units;
    uy = r / g.uw;
    ux = r - uy * g.uw;
    right = !EDGES || 2 * ux + 1 < g.W;
    below = !EDGES || 2 * uy + 1 < g.H;
  }
  __device__ __forceinline__ int at(const Planes& g, int c) const { return ((b * g.C + c) * g.H + 2 * uy) * g.W + COLS * ux; }
  __device__ __forceinline__ int pooled(const Planes& g, int c) const { return ((b * g.C + c) * (g.H / 2) + uy) * (g.W / 2) + COLS / 2 * ux; }
  __device__ __forceinline__ bool has(int row, int col) const { return !EDGES || ((row == 0 || below) && (col == 0 || right)); }
  __device__ __forceinline__ void load(const Planes& g, const float* p, float (&v)[2][COLS]) const {
#pragma unroll
    for (int r = 0; r < 2; r++) {
      if constexpr (EDGES) {
#pragma unroll
        for (int e = 0; e < COLS; e++) v[r][e] = has(r, e) ? p[r * g.W + e] : 0.0f;
      } else {
        const auto t = *(const typename Vec<COLS>::T*)(p + r * g.W);
#pragma unroll
        for (int e = 0; e < COLS; e++) v[r][e] = t[e];
      }
    }
  }
  __device__ __forceinline__ void store(const Planes& g, float* p, const float (&v)[2][COLS]) const {
#pragma unroll
    for (int r = 0; r < 2; r++) {
      if constexpr (EDGES) {
#pragma unroll
        for (int e = 0; e < COLS; e++)
          if (has(r, e)) p[r * g.W + e] = v[r][e];
      } else {
        typename Vec<COLS>::T t;
#pragma unroll
        for (int e = 0; e < COLS; e++) t[e] = v[r][e];
        *(typename Vec<COLS>::T*)(p + r * g.W) = t;
      }
    }
  }
};

// The sum of v over the workgroup, in every thread: lanes, then wavefronts in order.
__device__ __forceinline__ float group_sum(float v, float* sh) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[wave] = v;
  __syncthreads();
  float r = 0.0f;
  for (int w = 0; w < waves; w++) r = r + sh[w];
  return r;
}

// One sum of a channel, passed between its workgroups: slot g holds a mark in its upper half and the share's sum in the
// lower one.
__device__ __forceinline__ void publish(u64* slots, int g, float v) {
  __hip_atomic_store(slots + g, (1ull << 32) | __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 look(const u64* slots, int g) { return __hip_atomic_load(slots + g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

struct Sums {
  float part[2][64];
  float waves[kThreads / 64];
  int mine;   // a claim came first
  int next;   // the share to do next, or -1
};

// What a channel's workgroups share: G sums of two kinds (forward: one after the other), a claim for each share, and a count.
struct Channel {
  u64* slots[2];
  unsigned *claims, *count;
  __device__ __forceinline__ Channel(u64* page, int c, int sums, int shares)
      : slots{page + c * sums, page + kBnHeldSlots + c * sums}, claims((unsigned*)(page + 2 * kBnHeldSlots) + c * shares), count((unsigned*)(page + 2 * kBnHeldSlots) + kBnHeldSlots + c) {}
};
__device__ __forceinline__ bool claim(const Channel& ch, int share) { return !__hip_atomic_exchange(ch.claims + share, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Waits for the G sums of kinds `first`..`last` and leaves them in LDS: -1.  Or the number of a share (of the first `shares`)
// that nobody has begun and that is this workgroup's now.
__device__ __forceinline__ int gather(const Channel& ch, int first, int last, int G, int shares, int polls, Sums& sh) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int next = -1;
    u64 v[2] = {1ull << 32, 1ull << 32};
    for (int asked = 0;; asked++) {
      if (lane < G)
        for (int k = first; k <= last; k++) v[k] = look(ch.slots[k], lane);
      if (!__ballot(!(v[0] >> 32) || !(v[1] >> 32)) || asked == kGiveUp) break;
      if (asked >= polls && shares) {
        const u64 open = __ballot(lane < shares && !__hip_atomic_load(ch.claims + (lane < shares ? lane : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (open) {
          const int s = __builtin_ctzll(open);
          const int got = lane == 0 && claim(ch, s);
          if (__shfl(got, 0, 64)) { next = s; break; }
          continue;
        }
      }
      __builtin_amdgcn_s_sleep(1);
    }
    for (int k = first; k <= last; k++) sh.part[k][lane] = v[k] >> 32 ? __builtin_bit_cast(float, (unsigned)v[k]) : __builtin_nanf("");
    if (lane == 0) sh.next = next;
  }
  __syncthreads();
  const int next = sh.next;
  __syncthreads();   // before the next one is written
  return next;
}
__device__ __forceinline__ float total(const Sums& sh, int kind, int G) {
  float s = 0.0f;
  for (int g = 0; g < G; g++) s = s + sh.part[kind][g];
  return s;
}

// Everything of the channel is zero again when its last workgroup is through.  (A workgroup that has published a sum has seen
// it, with all the others, before it comes here.  No order with the tensors' values is needed, and a release here would write
// the cache back: 16 us instead of 10 for 8 x 128 x 26 x 26.)
__device__ __forceinline__ void leave(const Channel& ch, int sums, int shares) {
  if (threadIdx.x == 0 && __hip_atomic_fetch_add(ch.count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)shares - 1) {
    for (int g = 0; g < sums; g++) {
      __hip_atomic_store(ch.slots[0] + g, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(ch.slots[1] + g, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    for (int g = 0; g < shares; g++) __hip_atomic_store(ch.claims + g, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ch.count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

struct BnOut {
  float *run_mean, *run_var, *save_mean, *save_var;
  float eps, momentum;
};

// How k_bn_reduce cuts a channel: `groups` groups of 256 threads, thread t of group k with the values k * 256 + t, then every
// groups * 256-th of a plane, of all images - or, in planes of fewer values than a group has threads, whole planes.  A
// workgroup here does the work of `own` of them.
struct Cut {
  int S, groups, own;
};

// The forward sums are k_bn_reduce's to the bit: where one order of additions sends a value to one side of a rectifier's
// step or a window's maximum and another order to the other, a whole gradient element goes with it.
// HELD: groups of four images that a thread keeps in registers between its two passes (0: it reads them again).
// y null: the normalised values are only pooled (GH_FLAG_BN_REMADE).
template <int COLS, bool EDGES, int HELD>
__global__ __launch_bounds__(kThreads) void k_bn_train_pool(const float* __restrict__ x, float* __restrict__ y, float* __restrict__ pooled, Planes g, Cut cut, int64_t n,
                                                            BnOut o, u64* page) {
  __shared__ Sums sh;
  const int c = blockIdx.x % g.C, w = blockIdx.x / g.C;
  const Channel ch(page, c, cut.groups, g.G);
  const int shares = (cut.groups + cut.own - 1) / cut.own;   // those with sums; the others only write
  bool claimed = false;
  if (threadIdx.x == 0 && !(g.polls == 0 && (w & 1) && w < shares)) claimed = claim(ch, w);
  const int quarter = threadIdx.x >> 8, t = threadIdx.x & 255, mine = w * cut.own + quarter;
  const bool works = quarter < cut.own && mine < cut.groups;
  const int B = (int)(n / cut.S), img = g.C * cut.S, step = cut.groups * 256;
  float v[HELD > 0 ? HELD : 1][4];
  auto term = [&](float x_, float mean, bool sq) {
    if (!sq) return x_;
    const float d = x_ - mean;
    return d * d;
  };
  // thread t's sum of group k: of values (mean 0) or of squared deviations
  auto walk = [&](int k, float mean, bool sq) {
    if (cut.S < 256) {
      float acc = 0.0f;
      for (int b = k * 256 + t; b < B; b += step) {
        const float* const p = x + (b * g.C + c) * cut.S;
        for (int d = 0; d < cut.S; d++) acc = acc + term(p[d], mean, sq);
      }
      return acc;
    }
    float a4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int d = k * 256 + t; d < cut.S; d += step) {
      const float* const p = x + c * cut.S + d;
      int b = 0;
      for (; b + 4 <= B; b += 4) {
        const float v0 = p[b * img], v1 = p[(b + 1) * img], v2 = p[(b + 2) * img], v3 = p[(b + 3) * img];
        a4[0] = a4[0] + term(v0, mean, sq);
        a4[1] = a4[1] + term(v1, mean, sq);
        a4[2] = a4[2] + term(v2, mean, sq);
        a4[3] = a4[3] + term(v3, mean, sq);
      }
      for (; b < B; b++) a4[0] = a4[0] + term(p[b * img], mean, sq);
    }
    return (a4[0] + a4[1]) + (a4[2] + a4[3]);
  };
  // the same from and to registers: whole groups of four images only, HELD of them at most
  const int fours = B >> 2;
  auto hold = [&](auto&& f) __attribute__((always_inline)) {   // f(slot, first value's place) for each group of four that thread t has
    int b4 = 0, d = mine * 256 + t;
#pragma unroll
    for (int j = 0; j < HELD; j++) {
      if (d < cut.S) f(j, c * cut.S + d + 4 * b4 * img);
      if (++b4 == fours) { b4 = 0; d += step; }
    }
  };
  auto held = [&](float mean, bool sq) __attribute__((always_inline)) {
    float a4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    hold([&](int j, int) {
#pragma unroll
      for (int e = 0; e < 4; e++) a4[e] = a4[e] + term(v[j][e], mean, sq);
    });
    return (a4[0] + a4[1]) + (a4[2] + a4[3]);
  };
  // a group's sum, in all of its threads: block_sum of k_bn_reduce
  auto group = [&](float acc) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh.waves[threadIdx.x >> 6] = acc;
    __syncthreads();
    const float* const four = sh.waves + 4 * quarter;
    return (four[0] + four[1]) + (four[2] + four[3]);
  };
  float mean = 0.0f, var = 0.0f;
  if constexpr (HELD > 0) {
    if (works)
      hold([&](int j, int at) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[j][e] = x[at + e * img];
      });
  }
  if (threadIdx.x == 0) sh.mine = claimed;   // (asked for in front of the loads)
  __syncthreads();
  if (!sh.mine) return leave(ch, cut.groups, g.G);
  u64 more = 0;   // shares that were claimed behind the first
  auto again = [&](int share, int pass) {   // from memory
    const int k = share * cut.own + quarter;
    const bool has = quarter < cut.own && k < cut.groups;
    const float s = group(has ? walk(k, mean, pass == 1) : 0.0f);
    if (has && t == 0) publish(ch.slots[pass], k, s);
  };
#pragma unroll
  for (int pass = 0; pass < 2; pass++) {
    const bool sq = pass == 1;
    float acc = 0.0f;
    if (works) acc = HELD > 0 ? held(mean, sq) : walk(mine, mean, sq);
    const float s = group(acc);
    if (works && t == 0) publish(ch.slots[pass], mine, s);
    if (sq)
      for (u64 left = more; left; left &= left - 1) again(__builtin_ctzll(left), pass);
    for (int share; (share = gather(ch, pass, pass, cut.groups, sq ? 0 : shares, g.polls, sh)) >= 0;) {
      more |= 1ull << share;
      again(share, pass);
    }
    const float sum = total(sh, pass, cut.groups);
    if (!sq) mean = sum / (float)n;
    else var = sum;
    __syncthreads();   // the sums have been read
  }
  more |= 1ull << w;
  if ((more & 1) && threadIdx.x == 0) {
    o.save_mean[c] = mean;
    o.save_var[c] = var;
    const float m1 = o.momentum * mean, m2 = (1.0f - o.momentum) * o.run_mean[c];
    o.run_mean[c] = m1 + m2;
    const float unb = var / (float)(n - 1);
    const float v1 = o.momentum * unb, v2 = (1.0f - o.momentum) * o.run_var[c];
    o.run_var[c] = v1 + v2;
  }
  const float a = 1.0f / sqrtf(var / (float)n + o.eps);
  const float b = -mean * a;
  // the values again, from the caches, as the pooling's windows lie
  for (; more; more &= more - 1) {
    const int from = __builtin_ctzll(more) * g.per, end = min(g.units, from + g.per);
#pragma unroll 2
    for (int u = from + threadIdx.x; u < end; u += blockDim.x) {
      const Unit<COLS, EDGES> q(g, u);
      float z[2][COLS];
      q.load(g, x + q.at(g, c), z);
#pragma unroll
      for (int r = 0; r < 2; r++)
#pragma unroll
        for (int e = 0; e < COLS; e++) {
          const float m = z[r][e] * a;
          z[r][e] = m + b;
        }
      if (y) q.store(g, y + q.at(g, c), z);
      if (EDGES && !(q.right && q.below)) continue;
      float best[COLS / 2];
#pragma unroll
      for (int e = 0; e < COLS / 2; e++) {
        best[e] = -FLT_MAX;
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const float r = relu_of(z[k >> 1][2 * e + (k & 1)]);
          if (r > best[e]) best[e] = r;
        }
      }
      float* const p = pooled + q.pooled(g, c);
      if constexpr (COLS == 4) *(Vec<2>::T*)p = Vec<2>::T{best[0], best[1]};
      else *p = best[0];
    }
  }
  leave(ch, cut.groups, g.G);
}

// x: the tensor that was rectified and pooled; dp: the pooled tensor's gradient; dx: the gradient of x; z: the tensor that was
// normalised; dz its gradient (which may take x's or z's place).  REMADE: x is z normalised with the saved statistics, made
// again here in the forward's two operations, and neither x nor dx is touched.
template <int COLS, bool EDGES, int N, bool REMADE>
__global__ __launch_bounds__(kThreads) void k_pool_bn_bwd(const float* x, const float* __restrict__ dp, float* __restrict__ dx, const float* z, float* dz, Planes g,
                                                          int64_t n, const float* __restrict__ save_mean, const float* __restrict__ save_var, float eps, u64* page) {
  __shared__ Sums sh;
  const int c = blockIdx.x % g.C, w = blockIdx.x / g.C;
  const Channel ch(page, c, g.G, g.G);
  bool claimed = false;
  if (threadIdx.x == 0 && !(g.polls == 0 && (w & 1))) claimed = claim(ch, w);
  const float mean = save_mean[c], vb = save_var[c] / (float)n;
  const float invstd = 1.0f / sqrtf(vb + eps), shift = -mean * invstd;
  float zv[N][2][COLS], gv[N][2][COLS];
  // unit k of a thread in share `who`
  auto has = [&](int who, int k) { return k * (int)blockDim.x + (int)threadIdx.x < g.per && who * g.per + k * (int)blockDim.x + (int)threadIdx.x < g.units; };
  auto unit = [&](int who, int k) { return Unit<COLS, EDGES>(g, who * g.per + k * (int)blockDim.x + (int)threadIdx.x); };
  auto load = [&](int who, int k, float (&hz)[2][COLS], float (&hg)[2][COLS], float (&d)[COLS / 2]) __attribute__((always_inline)) {
    if (!has(who, k)) return;
    const Unit<COLS, EDGES> t = unit(who, k);
    if constexpr (!REMADE) t.load(g, x + t.at(g, c), hg);
    t.load(g, z + t.at(g, c), hz);
    const float* const p = dp + t.pooled(g, c);
    if constexpr (COLS == 4) {
      const auto pv = *(const Vec<2>::T*)p;
      d[0] = pv[0];
      d[1] = pv[1];
    } else {
      d[0] = t.right && t.below ? *p : 0.0f;
    }
  };
  float s, dot;
  // a unit's gradient of x, where x was (REMADE: is made)
  auto gradient = [&](const Unit<COLS, EDGES>& t, const float (&hz)[2][COLS], float (&hg)[2][COLS], const float (&d)[COLS / 2]) __attribute__((always_inline)) {
    const bool whole = t.right && t.below;
    if constexpr (REMADE) {
#pragma unroll
      for (int r = 0; r < 2; r++)
#pragma unroll
        for (int e = 0; e < COLS; e++) {
          const float m = hz[r][e] * invstd;
          hg[r][e] = m + shift;
        }
    }
#pragma unroll
    for (int e = 0; e < COLS / 2; e++) {
      float best = -FLT_MAX;
      int arg = -1;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float r = relu_of(hg[q >> 1][2 * e + (q & 1)]);
        if (r > best) { best = r; arg = q; }
      }
      const float v = 0.0f + d[e];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        float& h = hg[q >> 1][2 * e + (q & 1)];
        const float o = arg == q ? v : 0.0f;
        h = whole ? o * relu_mask(h) : 0.0f;
      }
    }
  };
  auto add = [&](int who, int k, const float (&hz)[2][COLS], float (&hg)[2][COLS], const float (&d)[COLS / 2]) __attribute__((always_inline)) {
    if (!has(who, k)) return;
    const Unit<COLS, EDGES> t = unit(who, k);
    gradient(t, hz, hg, d);
    if constexpr (!REMADE) t.store(g, dx + t.at(g, c), hg);
    float s4[2][COLS], d4[2][COLS];
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int e = 0; e < COLS; e++) {
        const float t1 = hz[r][e] * hg[r][e], t2 = mean * hg[r][e];
        s4[r][e] = t.has(r, e) ? hg[r][e] : 0.0f;
        d4[r][e] = t.has(r, e) ? t1 - t2 : 0.0f;
      }
    float qs = 0.0f, qd = 0.0f;
#pragma unroll
    for (int e = 0; e < COLS; e += 2) {
      qs = qs + ((s4[0][e] + s4[0][e + 1]) + (s4[1][e] + s4[1][e + 1]));
      qd = qd + ((d4[0][e] + d4[0][e + 1]) + (d4[1][e] + d4[1][e + 1]));
    }
    s = s + qs;
    dot = dot + qd;
  };
  float sum[2];
  auto say = [&](int who) {
    sum[0] = group_sum(s, sh.waves);
    sum[1] = group_sum(dot, sh.waves);
    if (threadIdx.x == 0) {
      publish(ch.slots[0], who, sum[0]);
      publish(ch.slots[1], who, sum[1]);
    }
  };
  {
    // everything a thread needs is on its way before the first value is looked at
    float d[N][COLS / 2];
#pragma unroll
    for (int k = 0; k < N; k++) load(w, k, zv[k], gv[k], d[k]);
    if (threadIdx.x == 0) sh.mine = claimed;   // (asked for in front of the loads)
    __syncthreads();
    if (!sh.mine) return leave(ch, g.G, g.G);
    s = dot = 0.0f;
#pragma unroll
    for (int k = 0; k < N; k++) add(w, k, zv[k], gv[k], d[k]);
    say(w);
  }
  u64 more = 0;   // shares that were claimed behind the first
  for (int who; (who = gather(ch, 0, 1, g.G, g.G, g.polls, sh)) >= 0;) {
    more |= 1ull << who;
    s = dot = 0.0f;
#pragma unroll 1
    for (int k = 0; k < N; k++) {
      float hz[2][COLS], hg[2][COLS], d[COLS / 2];
      load(who, k, hz, hg, d);
      add(who, k, hz, hg, d);
    }
    say(who);
  }
  sum[0] = total(sh, 0, g.G);
  sum[1] = total(sh, 1, g.G);
  float f = sum[1] * invstd;
  f = f * invstd;
  f = f / (float)n;
  const float grad_mean = sum[0] / (float)n;
  auto finish = [&](const Unit<COLS, EDGES>& t, const float (&hz)[2][COLS], float (&hg)[2][COLS]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int e = 0; e < COLS; e++) {
        float m = hz[r][e] - mean;
        m = m * f;
        float q = hg[r][e] - grad_mean;
        q = q - m;
        hg[r][e] = q * invstd;
      }
    t.store(g, dz + t.at(g, c), hg);
  };
#pragma unroll
  for (int k = 0; k < N; k++) {
    if (!has(w, k)) break;
    finish(unit(w, k), zv[k], gv[k]);
  }
  for (; more; more &= more - 1) {   // (a thread reads the gradient that it has written, or makes it again)
    const int who = __builtin_ctzll(more);
#pragma unroll 1
    for (int k = 0; k < N && has(who, k); k++) {
      const Unit<COLS, EDGES> t = unit(who, k);
      float hz[2][COLS], hg[2][COLS], d[COLS / 2];
      if constexpr (REMADE) {
        load(who, k, hz, hg, d);
        gradient(t, hz, hg, d);
      } else {
        t.load(g, z + t.at(g, c), hz);
        t.load(g, dx + t.at(g, c), hg);
      }
      finish(t, hz, hg);
    }
  }
  leave(ch, g.G, g.G);
}

// ---- which commands ---------------------------------------------------------------------

bool apart(uint64_t p, int64_t bytes, uint64_t q, int64_t other) { return p + (uint64_t)bytes <= q || q + (uint64_t)other <= p; }

// a float32 2x2 / stride-2 pooling (or its gradient) without padding of the rectified input
bool pools(const gh_cmd& c) {
  if (gh_dtype_of(c.flags) != GH_F32 || !(c.flags & GH_FLAG_ACT_RELU)) return false;
  for (int i : {4, 5, 10, 11}) if (c.dim[i] != 2) return false;
  for (int i : {6, 7, 8, 9}) if (c.dim[i] != 0) return false;
  return c.dim[0] > 0 && c.dim[1] > 0 && c.dim[2] >= 2 && c.dim[3] >= 2;
}

constexpr int kMost = 3;   // units of a thread in the gradient, of four columns each: 24 values, and as many of the other tensor

struct Plan {
  Planes g;
  Cut cut;
  int cols, threads, N;   // N: units of a thread (the gradient)
  bool held;              // the forward's values stay in registers
};

// How the planes go to workgroups, one to a compute unit: false where a channel does not fit them.
bool plan(const gh_cmd& pool, bool fwd, uint64_t wide, uint64_t narrow, int cus, Plan& p) {
  const int64_t B = pool.dim[0], C = pool.dim[1], H = pool.dim[2], W = pool.dim[3], S = H * W, n = B * S;
  if (C > cus || B * C * S > INT32_MAX || n < 2) return false;
  p.cols = W % 4 == 0 && H % 2 == 0 && wide % 16 == 0 && narrow % 8 == 0 ? 4 : W % 2 == 0 && H % 2 == 0 && wide % 8 == 0 ? 2 : 1;
  const int64_t across = p.cols == 4 ? W / 4 : (W + 1) / 2, units = B * ((H + 1) / 2) * across;
  // half of a workgroup's threads have work at least: the gradient of 8 x 128 x 26 x 26 takes 7.9 us with one workgroup to a
  // channel, 6.7 with two
  int64_t G = std::min<int64_t>({(int64_t)cus / C, 64, (units + 511) / 512});
  p.cut = {(int)S, 0, 0};
  if (fwd) {
    const int64_t groups = gh_bn_groups(n, S);
    G = std::max(G, (groups + 3) / 4);
    if (C * G > cus || C * groups > kBnHeldSlots) return false;
    p.cut.groups = (int)groups;
    p.cut.own = (int)((groups + G - 1) / G);
  }
  const int64_t per = (units + G - 1) / G;
  p.g = {(int)H, (int)W, (int)across, (int)((H + 1) / 2 * across), (int)units, (int)per, (int)C, (int)G, kPolls};
  if (fwd) {
    p.N = 0;
    p.threads = (int)std::max<int64_t>(256 * p.cut.own, std::min<int64_t>(kThreads, (per + 255) / 256 * 256));
    // (a thread's strips of 256 values, of whole groups of four images)
    p.held = S >= 256 && B % 4 == 0 && ((S + 255) / 256 + p.cut.groups - 1) / p.cut.groups * (B / 4) <= kHeld;
  } else {
    p.g.G = (int)((units + per - 1) / per);
    p.N = (int)((per + kThreads - 1) / kThreads);
    if (C * p.g.G > kBnHeldSlots || p.N > kMost * (p.cols == 4 ? 1 : 2)) return false;
    p.threads = (int)(((per + p.N - 1) / p.N + 63) / 64 * 64);
  }
  if (const char* asks = getenv("GORGONIA_HIP_BN_POLLS")) p.g.polls = std::max(0, std::min(1000, atoi(asks)));
  return true;
}

// f(columns, edges, units of a thread): the gradient's form
template <class F>
void with_form(const Plan& p, F&& f) {
  auto of = [&](auto cols, auto edges, auto most) {
    if (p.N == 1) f(cols, edges, std::integral_constant<int, 1>());
    else if (p.N == 2) f(cols, edges, std::integral_constant<int, 2>());
    else f(cols, edges, most);
  };
  if (p.cols == 4) of(std::integral_constant<int, 4>(), std::false_type(), std::integral_constant<int, kMost>());
  else if (p.cols == 2) of(std::integral_constant<int, 2>(), std::false_type(), std::integral_constant<int, 2 * kMost>());
  else of(std::integral_constant<int, 2>(), std::true_type(), std::integral_constant<int, 2 * kMost>());
}
// f(columns, edges, held): the forward's
template <class F>
void with_held(const Plan& p, F&& f) {
  auto of = [&](auto cols, auto edges) {
    if (p.held) f(cols, edges, std::integral_constant<int, kHeld>());
    else f(cols, edges, std::integral_constant<int, 0>());
  };
  if (p.cols == 4) of(std::integral_constant<int, 4>(), std::false_type());
  else if (p.cols == 2) of(std::integral_constant<int, 2>(), std::false_type());
  else of(std::integral_constant<int, 2>(), std::true_type());
}

template <class T> T* at(uint64_t p) { return (T*)(uintptr_t)p; }

struct Tensors {
  uint64_t wide = 0, narrow = 0;   // addresses of the whole and of the pooled tensors, or-ed
};

// {BN_TRAIN, MAXPOOL2D} and {MAXPOOL2D_BWD, BN_BWD} in training mode; what is written lies apart from everything else, but
// the normalised tensor's gradient may take the place of a tensor that a thread has read where it writes.
bool fits(const gh_cmd* c, Tensors& t) {
  const bool fwd = c[0].opcode == GH_OP_BN_TRAIN;
  const gh_cmd &pool = fwd ? c[1] : c[0], &bn = fwd ? c[0] : c[1];
  if (!pools(pool) || gh_dtype_of(bn.flags) != GH_F32 || (bn.flags & GH_FLAG_BN_EVAL)) return false;
  if (bn.dim[0] != pool.dim[0] || bn.dim[1] != pool.dim[1] || bn.dim[2] != pool.dim[2] * pool.dim[3]) return false;
  const int64_t pooled = pool.dim[0] * pool.dim[1] * (pool.dim[2] / 2) * (pool.dim[3] / 2) * 4, whole = bn.dim[0] * bn.dim[1] * bn.dim[2] * 4, chan = bn.dim[1] * 4;
  struct Part { uint64_t p; int64_t bytes; };
  auto clear = [&](Part out, std::initializer_list<Part> all) {
    for (const Part& a : all)
      if (!apart(out.p, out.bytes, a.p, a.bytes)) return false;
    return true;
  };
  uint64_t every = pool.ptr[0] | pool.ptr[1];
  for (int i = 0; i < (fwd ? 6 : 5); i++) every |= bn.ptr[i];
  if (every & 3) return false;
  if (fwd) {
    const Part x{bn.ptr[0], whole}, y{bn.ptr[1], whole}, p{pool.ptr[1], pooled}, s[4] = {{bn.ptr[2], chan}, {bn.ptr[3], chan}, {bn.ptr[4], chan}, {bn.ptr[5], chan}};
    if (pool.ptr[0] != y.p || !clear(x, {y, p, s[0], s[1], s[2], s[3]}) || !clear(y, {p, s[0], s[1], s[2], s[3]}) || !clear(p, {s[0], s[1], s[2], s[3]})) return false;
    for (int i = 0; i < 4; i++)
      for (int j = 0; j < i; j++)
        if (!clear(s[i], {s[j]})) return false;
    t = {x.p | y.p, p.p};
    return true;
  }
  const Part x{pool.ptr[0], whole}, dp{pool.ptr[1], pooled}, dx{pool.ptr[2], whole}, z{bn.ptr[0], whole}, dz{bn.ptr[2], whole}, m{bn.ptr[3], chan}, v{bn.ptr[4], chan};
  if (bn.ptr[1] != dx.p || !clear(dx, {x, dp, z, dz, m, v}) || !clear(dz, {dp, m, v})) return false;
  if ((dz.p != x.p && !clear(dz, {x})) || (dz.p != z.p && !clear(dz, {z}))) return false;
  t = {x.p | dx.p | z.p | dz.p, dp.p};
  return true;
}

}  // namespace

// (c[0] is a valid command; c[1] is looked at where its opcode makes it a candidate)
bool gh_bn_held_pair(const gh_ctx* ctx, const gh_cmd* c, int n) {
  if (n < 2 || !ctx->bn_page) return false;
  const bool fwd = c[0].opcode == GH_OP_BN_TRAIN && c[1].opcode == GH_OP_MAXPOOL2D;
  if (!fwd && !(c[0].opcode == GH_OP_MAXPOOL2D_BWD && c[1].opcode == GH_OP_BN_BWD)) return false;
  std::string m;
  Tensors t;
  Plan p;
  return gh_validate_cmd(c[1], m) == GH_OK && fits(c, t) && plan(c[fwd ? 1 : 0], fwd, t.wide, t.narrow, ctx->cu_count, p);
}

int gh_launch_bn_held_pair(gh_ctx* ctx, const gh_cmd* c) {
  const bool fwd = c[0].opcode == GH_OP_BN_TRAIN;
  for (int k = 0; k < 2; k++)
    for (uint64_t p : c[k].ptr) ctx->llc.touch(p, 0, false);
  Tensors t;
  Plan p;
  if (!fits(c, t) || !plan(c[fwd ? 1 : 0], fwd, t.wide, t.narrow, ctx->cu_count, p)) return gh_fail(ctx, GH_EINVAL, "not a pair of commands that one launch takes");
  const gh_cmd &pool = fwd ? c[1] : c[0], &bn = fwd ? c[0] : c[1];
  const int64_t count = bn.dim[0] * bn.dim[2];
  const dim3 grid((unsigned)(p.g.C * p.g.G)), block((unsigned)p.threads);
  u64* const page = (u64*)ctx->bn_page;
  if (fwd) {
    const BnOut o{at<float>(bn.ptr[2]), at<float>(bn.ptr[3]), at<float>(bn.ptr[4]), at<float>(bn.ptr[5]), bn.f[0], bn.f[1]};
    float* const y = bn.flags & GH_FLAG_BN_REMADE ? nullptr : at<float>(bn.ptr[1]);
    with_held(p, [&](auto COLS, auto EDGES, auto HELD) {
      hipLaunchKernelGGL((k_bn_train_pool<COLS(), EDGES(), HELD()>), grid, block, 0, ctx->stream, at<const float>(bn.ptr[0]), y, at<float>(pool.ptr[1]), p.g, p.cut, count, o, page);
    });
  } else {
    const bool remade = pool.flags & GH_FLAG_BN_REMADE;
    with_form(p, [&](auto COLS, auto EDGES, auto UNITS) {
      const auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, ctx->stream, at<const float>(pool.ptr[0]), at<const float>(pool.ptr[1]), at<float>(pool.ptr[2]), at<const float>(bn.ptr[0]),
                           at<float>(bn.ptr[2]), p.g, count, at<const float>(bn.ptr[3]), at<const float>(bn.ptr[4]), bn.f[0], page);
      };
      if (remade) go(k_pool_bn_bwd<COLS(), EDGES(), UNITS(), true>);
      else go(k_pool_bn_bwd<COLS(), EDGES(), UNITS(), false>);
    });
  }
  return gh_check_hip(ctx, hipGetLastError(), fwd ? "batchnorm statistics launch" : "batchnorm backward launch");
}

namespace {

// y = z normalised with the saved statistics, one (image, channel) plane per blockIdx.y: the forward's two operations.
__global__ __launch_bounds__(256) void k_bn_remake(const float* __restrict__ z, float* __restrict__ y, const float* __restrict__ save_mean, const float* __restrict__ save_var, float eps,
                                                   int64_t BC, int C, int64_t S, int64_t n) {
  for (int64_t bc = blockIdx.y; bc < BC; bc += gridDim.y) {
    const int c = (int)(bc % C);
    const float a = 1.0f / sqrtf(save_var[c] / (float)n + eps), b = -save_mean[c] * a;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < S; i += (int64_t)gridDim.x * 256) {
      const float m = z[bc * S + i] * a;
      y[bc * S + i] = m + b;
    }
  }
}

}  // namespace

// (256 compute units, tensors at whole lines: what the tape's tensors have)
int gh_bn_can_remake(int64_t B, int64_t C, int64_t H, int64_t W) {
  gh_cmd pool{};
  pool.flags = GH_FLAG_DTYPE(GH_F32) | GH_FLAG_ACT_RELU;
  const int64_t dims[12] = {B, C, H, W, 2, 2, 0, 0, 0, 0, 2, 2};
  std::copy(dims, dims + 12, pool.dim);
  Plan p;
  return pools(pool) && plan(pool, true, 0, 0, 256, p) && plan(pool, false, 0, 0, 256, p);
}

// Whether c[1] is the batch normalisation's gradient that a MAXPOOL2D_BWD command with GH_FLAG_BN_REMADE needs behind it.
bool gh_bn_remade_follows(const gh_cmd* c, int n) {
  std::string m;
  return n >= 2 && c[1].opcode == GH_OP_BN_BWD && gh_dtype_of(c[1].flags) == GH_F32 && !(c[1].flags & GH_FLAG_BN_EVAL) && gh_validate_cmd(c[1], m) == GH_OK &&
         c[1].ptr[1] == c[0].ptr[2] && c[1].dim[0] == c[0].dim[0] && c[1].dim[1] == c[0].dim[1] && c[1].dim[2] == c[0].dim[2] * c[0].dim[3];
}

// The tensor that such a pair needs where no kernel takes it whole: into the place that the first command names.
int gh_launch_bn_remake(gh_ctx* ctx, const gh_cmd* c) {
  const gh_cmd& bn = c[1];
  const int64_t BC = bn.dim[0] * bn.dim[1], S = bn.dim[2];
  const dim3 grid((unsigned)std::min<int64_t>(1024, (S + 1023) / 1024), (unsigned)std::min<int64_t>(BC, 65535));
  hipLaunchKernelGGL(k_bn_remake, grid, dim3(256), 0, ctx->stream, at<const float>(bn.ptr[0]), at<float>(c[0].ptr[0]), at<const float>(bn.ptr[3]), at<const float>(bn.ptr[4]), bn.f[0], BC,
                     (int)bn.dim[1], S, bn.dim[0] * S);
  return gh_check_hip(ctx, hipGetLastError(), "batchnorm launch");
}
