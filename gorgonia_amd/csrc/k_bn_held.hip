// Batch statistics and the 2x2 pooling behind them in one launch, and their gradients in another.
//
// Training mode needs a channel's mean before its deviations and both before a value can be written, and a launch for each
// of these and for the pooling; the gradient needs two sums before it can be written.  Here C channels times G workgroups of
// up to 1024 threads, one workgroup on a compute unit, have a share of a channel each.  They pass their sums to each other
// through memory and wait for each other's.  A 22 MB tensor fits the chip's registers (128 MB): between its sums and the
// values it writes the gradient keeps what it has read, the forward its values between its two passes.
//
// A wait ends whether or not the others come: a workgroup that has asked kPolls times reads the missing shares and adds
// them up itself, in the same order, to the same bits.  Nothing depends on all workgroups being on the chip at once.
//
// Bound: HBM and the caches for large planes, the launch and the waits (some 1.5 us each) for small ones.  us, four launches
// or three / one, forward and gradient: 8 x 16 x 208 x 208 30.9 / 18.7 and 33.8 / 21.1 (4.4 TB/s of the 94 MB that the
// gradient moves), 8 x 32 x 104 x 104 20.5 / 11.8 and 22.9 / 12.3, 8 x 128 x 26 x 26 14.2 / 8.9 and 13.4 / 7.0,
// 8 x 16 x 207 x 207 (single loads) 46.6 / 20.8 and 47.3 / 25.8, 2 x 3 x 4 x 4 12.1 / 7.5 and 10.0 / 4.9.  (The forward as the
// gradient is, its values kept as the pooling's windows lie: 14.8, 9.9 and 7.3, and other sums.)
#include <algorithm>
#include <cfloat>

#include "gh_internal.h"

namespace {

constexpr int kThreads = 1024;
constexpr int kHeld = 6;   // groups of four values that a thread of the forward keeps
constexpr int kPolls = 2000;   // about a millisecond (GORGONIA_HIP_BN_POLLS: another number)
typedef unsigned long long u64;

__device__ __forceinline__ float relu_of(float v) { return v * (v >= 0.0f ? 1.0f : 0.0f); }
__device__ __forceinline__ float relu_mask(float v) { return v >= 0.0f ? 1.0f : 0.0f; }

template <int K> struct Vec { typedef float T __attribute__((ext_vector_type(K))); };

// B images of C planes of H x W; a unit is two rows of COLS columns (a last row or column alone where the size is odd),
// a workgroup has `per` of a channel's units.
struct Planes {
  int H, W, uw, plane_units, units, per, C, G;
  int polls;   // how often a workgroup asks for the others' sums
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
// the same, and back when every compute unit sees it
__device__ __forceinline__ void publish_and_wait(u64* slots, int g, float v) {
  const u64 old = __hip_atomic_exchange(slots + g, (1ull << 32) | __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("" ::"v"((unsigned)old) : "memory");
}
__device__ __forceinline__ u64 look(const u64* slots, int g) { return __hip_atomic_load(slots + g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

struct Sums {
  float part[2][64];
  u64 missing;
  float waves[kThreads / 64];
};

// Wavefront 0 waits for the G shares of `kinds` sums and leaves them in LDS; a share that has not come is in `missing`.
__device__ __forceinline__ void gather(u64* const (&slots)[2], int kinds, int G, int polls, Sums& sh) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    u64 v[2] = {1ull << 32, 1ull << 32};
    u64 miss = G < 64 ? (1ull << G) - 1 : ~0ull;
    for (int asked = 0; asked < polls; asked++) {
      if (lane < G)
        for (int k = 0; k < kinds; k++) v[k] = look(slots[k], lane);
      miss = __ballot(!(v[0] >> 32) || !(v[1] >> 32));
      if (!miss) break;
      __builtin_amdgcn_s_sleep(1);
    }
    for (int k = 0; k < kinds; k++) sh.part[k][lane] = __builtin_bit_cast(float, (unsigned)v[k]);
    if (lane == 0) sh.missing = miss;
  }
  __syncthreads();
}

// The G shares, the missing ones added up here by `share(g)`, in order.  A share that has come meanwhile is taken as it came:
// its workgroup may already be writing over what share(g) has read.
template <class F>
__device__ __forceinline__ void total(u64* const (&slots)[2], int kinds, int G, int polls, Sums& sh, float (&out)[2], F&& share) {
  gather(slots, kinds, G, polls, sh);
  u64 miss = sh.missing;
  while (miss) {
    const int g = __builtin_ctzll(miss);
    miss &= miss - 1;
    float v[2];
    share(g, v);
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0)
      for (int k = 0; k < kinds; k++) {
        const u64 now = look(slots[k], g);
        sh.part[k][g] = now >> 32 ? __builtin_bit_cast(float, (unsigned)now) : v[k];
      }
    __syncthreads();
  }
  for (int k = 0; k < kinds; k++) {
    float s = 0.0f;
    for (int g = 0; g < G; g++) s = s + sh.part[k][g];
    out[k] = s;
  }
}

// The channel's slots are zero again when its last workgroup is through.  (No order with the tensors' values is needed, and a
// release here would write the cache back: 16 us instead of 10 for 8 x 128 x 26 x 26.)
__device__ __forceinline__ void leave(u64* const (&slots)[2], unsigned* count, int shares, int workgroups) {
  if (threadIdx.x == 0 && __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)workgroups - 1) {
    for (int g = 0; g < shares; g++) {
      __hip_atomic_store(slots[0] + g, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(slots[1] + g, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
template <int COLS, bool EDGES, int HELD>
__global__ __launch_bounds__(kThreads) void k_bn_train_pool(const float* __restrict__ x, float* __restrict__ y, float* __restrict__ pooled, Planes g, Cut cut, int64_t n,
                                                            BnOut o, u64* page) {
  __shared__ Sums sh;
  const int c = blockIdx.x % g.C, w = blockIdx.x / g.C;
  u64* const slots[2] = {page + c * cut.groups, page + kBnHeldSlots + c * cut.groups};
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
  float mean = 0.0f, var = 0.0f, sum[2];
  if constexpr (HELD > 0) {
    if (works)
      hold([&](int j, int at) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[j][e] = x[at + e * img];
      });
  }
#pragma unroll
  for (int pass = 0; pass < 2; pass++) {
    const bool sq = pass == 1;
    float acc = 0.0f;
    if (works) acc = HELD > 0 ? held(mean, sq) : walk(mine, mean, sq);
    const float s = group(acc);
    if (works && t == 0) publish(slots[pass], mine, s);
    u64* const both[2] = {slots[pass], slots[pass]};
    total(both, 1, cut.groups, g.polls, sh, sum, [&](int k, float (&r)[2]) { r[0] = group(walk(k, mean, sq)); });
    if (!sq) mean = sum[0] / (float)n;
    else var = sum[0];
    __syncthreads();   // the sums have been read
  }
  if (w == 0 && threadIdx.x == 0) {
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
  const int end = min(g.units, (w + 1) * g.per);
#pragma unroll 2
  for (int u = w * g.per + threadIdx.x; u < end; u += blockDim.x) {
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
    q.store(g, y + q.at(g, c), z);
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
  leave(slots, (unsigned*)(page + 2 * kBnHeldSlots) + c, cut.groups, g.G);
}

// x: the tensor that was rectified and pooled; dp: the pooled tensor's gradient; dx: the gradient of x; z: the tensor that was
// normalised; dz its gradient (which may take x's or z's place).
template <int COLS, bool EDGES, int N>
__global__ __launch_bounds__(kThreads) void k_pool_bn_bwd(const float* x, const float* __restrict__ dp, float* __restrict__ dx, const float* z, float* dz, Planes g,
                                                          int64_t n, const float* __restrict__ save_mean, const float* __restrict__ save_var, float eps, u64* page) {
  __shared__ Sums sh;
  const int c = blockIdx.x % g.C, w = blockIdx.x / g.C;
  u64* const slots[2] = {page + c * g.G, page + kBnHeldSlots + c * g.G};
  const float mean = save_mean[c], vb = save_var[c] / (float)n;
  float zv[N][2][COLS], gv[N][2][COLS];
  auto share = [&](int who, bool own, float (&hz)[N][2][COLS], float (&hg)[N][2][COLS], float (&out)[2]) __attribute__((always_inline)) {
    float s = 0.0f, dot = 0.0f;
    // everything a thread needs is on its way before the first value is looked at
    float d[N][COLS / 2];
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int u = who * g.per + k * (int)blockDim.x + (int)threadIdx.x;
      const bool mine = k * (int)blockDim.x + (int)threadIdx.x < g.per && u < g.units;
      if (!mine) continue;
      const Unit<COLS, EDGES> t(g, u);
      t.load(g, x + t.at(g, c), hg[k]);
      t.load(g, z + t.at(g, c), hz[k]);
      const float* const p = dp + t.pooled(g, c);
      if constexpr (COLS == 4) {
        const auto pv = *(const Vec<2>::T*)p;
        d[k][0] = pv[0];
        d[k][1] = pv[1];
      } else {
        d[k][0] = t.right && t.below ? *p : 0.0f;
      }
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int u = who * g.per + k * (int)blockDim.x + (int)threadIdx.x;
      const bool mine = k * (int)blockDim.x + (int)threadIdx.x < g.per && u < g.units;
      if (!mine) continue;
      const Unit<COLS, EDGES> t(g, u);
      const bool whole = t.right && t.below;
#pragma unroll
      for (int e = 0; e < COLS / 2; e++) {
        float best = -FLT_MAX;
        int arg = -1;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const float r = relu_of(hg[k][q >> 1][2 * e + (q & 1)]);
          if (r > best) { best = r; arg = q; }
        }
        const float v = 0.0f + d[k][e];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          float& h = hg[k][q >> 1][2 * e + (q & 1)];
          const float o = arg == q ? v : 0.0f;
          h = whole ? o * relu_mask(h) : 0.0f;
        }
      }
      if (own) t.store(g, dx + t.at(g, c), hg[k]);
      float s4[2][COLS], d4[2][COLS];
#pragma unroll
      for (int r = 0; r < 2; r++)
#pragma unroll
        for (int e = 0; e < COLS; e++) {
          const float t1 = hz[k][r][e] * hg[k][r][e], t2 = mean * hg[k][r][e];
          s4[r][e] = t.has(r, e) ? hg[k][r][e] : 0.0f;
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
    }
    out[0] = group_sum(s, sh.waves);
    out[1] = group_sum(dot, sh.waves);
  };
  float sum[2];
  share(w, true, zv, gv, sum);
  if (threadIdx.x == 0) {
    // before dz is written (behind the barrier in total): a workgroup that adds up this share in this one's place and reads
    // values of dz finds the slots filled
    publish_and_wait(slots[0], w, sum[0]);
    publish_and_wait(slots[1], w, sum[1]);
  }
  total(slots, 2, g.G, g.polls, sh, sum, [&](int who, float (&r)[2]) {
    float oz[N][2][COLS], og[N][2][COLS];
    share(who, false, oz, og, r);
  });
  const float invstd = 1.0f / sqrtf(vb + eps);
  float f = sum[1] * invstd;
  f = f * invstd;
  f = f / (float)n;
  const float grad_mean = sum[0] / (float)n;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int u = w * g.per + k * (int)blockDim.x + (int)threadIdx.x;
    if (k * (int)blockDim.x + (int)threadIdx.x >= g.per || u >= g.units) break;
    const Unit<COLS, EDGES> t(g, u);
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int e = 0; e < COLS; e++) {
        float m = zv[k][r][e] - mean;
        m = m * f;
        float q = gv[k][r][e] - grad_mean;
        q = q - m;
        gv[k][r][e] = q * invstd;
      }
    t.store(g, dz + t.at(g, c), gv[k]);
  }
  leave(slots, (unsigned*)(page + 2 * kBnHeldSlots) + c, g.G, g.G);
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
  if (const char* asks = getenv("GORGONIA_HIP_BN_POLLS")) p.g.polls = std::max(0, std::min(kPolls, atoi(asks)));
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
    with_held(p, [&](auto COLS, auto EDGES, auto HELD) {
      hipLaunchKernelGGL((k_bn_train_pool<COLS(), EDGES(), HELD()>), grid, block, 0, ctx->stream, at<const float>(bn.ptr[0]), at<float>(bn.ptr[1]), at<float>(pool.ptr[1]), p.g,
                         p.cut, count, o, page);
    });
  } else {
    with_form(p, [&](auto COLS, auto EDGES, auto UNITS) {
      hipLaunchKernelGGL((k_pool_bn_bwd<COLS(), EDGES(), UNITS()>), grid, block, 0, ctx->stream, at<const float>(pool.ptr[0]), at<const float>(pool.ptr[1]),
                         at<float>(pool.ptr[2]), at<const float>(bn.ptr[0]), at<float>(bn.ptr[2]), p.g, count, at<const float>(bn.ptr[3]), at<const float>(bn.ptr[4]), bn.f[0], page);
    });
  }
  return gh_check_hip(ctx, hipGetLastError(), fwd ? "batchnorm statistics launch" : "batchnorm backward launch");
}
