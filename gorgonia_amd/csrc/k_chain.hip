// A run of elementwise operators in one pass.
//
// Elementwise commands that follow each other on tensors of one size read what the command before them wrote:
// each is a pass over memory (or, for small tensors, a launch) that exists only to hand a value on.  gh_submit
// gives such a run to this kernel: every thread takes its values through all the steps, reads each tensor
// where it is first needed, keeps intermediate values in registers and LDS, and stores only what is still
// there when the run ends - a tensor that a later step of the run overwrites is not stored twice.  The steps
// apply the functions of gh_elem_fn.h in the order of the commands, so the stored bits are theirs.
// Which commands make a run is decided by earns() and pays() below.
//
// Bound: HBM for large tensors (sigmoid, tanh and pow(., 2) of x * y + b on 4096 x 4096 float32: 336 MB instead
// of 738, 66 us instead of 117), for small ones the launch and a thread's walk from step to step (five launches become one).
#include <algorithm>
#include <cstring>

#include "gh_elem_fn.h"
#include "gh_internal.h"

namespace {

constexpr int kBlock = 256;
constexpr int kMaxSteps = 8;
constexpr int kSlots = 2;     // values kept past the step behind theirs

// Where a step finds an operand.
enum Src : uint8_t { kAcc, kSlot0, kSlot1, kMem, kScalar, kSmallVec, kSmallAny };
// Function codes: GH_BINFN, then GH_UNARYFN, then the activations.
constexpr int kUnary = 16, kRelu = 40, kLeaky = 41, kReluBwd = 42;

struct Step {
  const void* a;
  const void* b;
  void* store;        // null: the value is not stored
  double alpha;
  uint32_t mid, mid_mul, mid_sh, inner_mul, inner_sh;   // of a kSmall operand: its length and the divisors' reciprocals
  uint8_t fn, src_a, src_b, save;                       // save: slot + 1, or 0
};

struct Chain {
  int64_t n;
  int steps;
  Step step[kMaxSteps];
};

// n / d for n < 2^32 by multiplication (round-up reciprocal, Granlund & Montgomery 1994, figure 4.1).
__device__ __forceinline__ uint32_t fast_div(uint32_t n, uint32_t mul, uint32_t sh) {
  const uint32_t t = __umulhi(mul, n);
  return sh ? (t + ((n - t) >> 1)) >> (sh - 1) : n;
}

template <class T, bool STREAM, int N>
struct Lane {
  typedef T V __attribute__((ext_vector_type(N)));

  // vector i of a tensor of n elements: the last one may be partial
  static __device__ __forceinline__ V load(const void* p, int64_t i, int64_t n) {
    const T* q = (const T*)p;
    if ((i + 1) * N <= n) return ld_vec<V, STREAM>((const V*)p + i);
    V v = V{};
    for (int e = 0; e < N; e++)
      if (i * N + e < n) v[e] = q[i * N + e];
    return v;
  }
  static __device__ __forceinline__ void store(void* p, int64_t i, int64_t n, V v) {
    T* q = (T*)p;
    if ((i + 1) * N <= n) { st_vec<V, STREAM>((V*)p + i, v); return; }
    for (int e = 0; e < N; e++)
      if (i * N + e < n) q[i * N + e] = v[e];
  }
  static __device__ __forceinline__ V small_vec(const Step& s, const void* p, int64_t i) {   // inner 1, whole vectors
    const uint32_t x = (uint32_t)(i * N);
    return *(const V*)((const T*)p + (x - fast_div(x, s.mid_mul, s.mid_sh) * s.mid));
  }
  static __device__ __forceinline__ V small_any(const Step& s, const void* p, int64_t i) {
    V v;
#pragma unroll
    for (int e = 0; e < N; e++) {
      const uint32_t x = fast_div((uint32_t)(i * N + e), s.inner_mul, s.inner_sh);
      v[e] = ((const T*)p)[x - fast_div(x, s.mid_mul, s.mid_sh) * s.mid];
    }
    return v;
  }
};

template <class T>
__device__ __forceinline__ T relu_of(T x) { return x * (x >= (T)0 ? (T)1 : (T)0); }
template <class T>
__device__ __forceinline__ T leaky_of(T x, T alpha) {
  const T pos = x * (x >= (T)0 ? (T)1 : (T)0);
  const T neg = x * (x < (T)0 ? (T)1 : (T)0);
  const T na = neg * alpha;
  return pos + na;
}

template <int F, class T>
__device__ __attribute__((noinline)) T unary_call(T x) { return unary_apply<F>(x); }
template <int F, class T>
__device__ __attribute__((noinline)) T bin_call(T x, T y) { return bin_apply<F, T>(x, y); }

template <class T, bool STREAM, int N, int kU>
__global__ __launch_bounds__(kBlock) void k_chain(const Chain c) {
  typedef Lane<T, STREAM, N> L;
  typedef typename L::V V;
  // the arguments' lines into the scalar cache, all at once: a step's own loads would each wait for theirs
  uint32_t lines = 0;
#pragma unroll
  for (int l = 0; l < (int)(sizeof(Chain) / 64); l++) lines |= ((const uint32_t*)&c)[16 * l];
  asm volatile("" ::"s"(lines));
  __shared__ V slots[kSlots][kU][kBlock];
  __shared__ V scratch[2][kBlock];
  const int64_t nv = (c.n + N - 1) / N;
  const int64_t stride = (int64_t)gridDim.x * kBlock * kU;
  for (int64_t i0 = (int64_t)blockIdx.x * kBlock * kU + threadIdx.x; i0 < nv; i0 += stride) {
    V acc[kU] = {};
    int64_t at[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) at[u] = min(i0 + (int64_t)u * kBlock, nv);   // nv: past the end, loads and stores nothing
    for (int k = 0; k < c.steps; k++) {
      const Step& s = c.step[k];
      V a[kU], b[kU] = {};
      auto fetch = [&](V* v, uint8_t src, const void* p) {
#pragma unroll
        for (int u = 0; u < kU; u++) {
          if (src == kAcc) v[u] = acc[u];
          else if (src == kMem) v[u] = L::load(p, at[u], c.n);
          else if (src == kScalar) v[u] = V(*(const T*)p);
          else if (src == kSmallVec) v[u] = L::small_vec(s, p, at[u]);
          else if (src == kSmallAny) v[u] = L::small_any(s, p, at[u]);
          else v[u] = slots[src - kSlot0][u][threadIdx.x];
        }
      };
      fetch(a, s.src_a, s.a);
      if (s.fn < kUnary || s.fn == kReluBwd) fetch(b, s.src_b, s.b);
      switch (s.fn) {
#define GH_EACH(EXPR)                          \
  _Pragma("unroll") for (int u = 0; u < kU; u++) \
  _Pragma("unroll") for (int e = 0; e < N; e++) acc[u][e] = EXPR; \
  break;
// Functions of many instructions: one copy, looped over the elements in LDS.  Inlined per element they cost the
// kernel twice the registers (169 of float32 with all of them) and with that the waves that hide the loads.
#define GH_EACH_HEAVY(EXPR)                                     \
  _Pragma("unroll") for (int u = 0; u < kU; u++) {              \
    scratch[0][threadIdx.x] = a[u];                             \
    scratch[1][threadIdx.x] = b[u];                             \
    T* pe = (T*)&scratch[0][threadIdx.x];                       \
    const T* qe = (const T*)&scratch[1][threadIdx.x];           \
    _Pragma("unroll 1") for (int e = 0; e < N; e++) {           \
      const T x = pe[e], y = qe[e];                             \
      (void)y;                                                  \
      pe[e] = EXPR;                                             \
    }                                                           \
    acc[u] = scratch[0][threadIdx.x];                           \
  }                                                             \
  break;
#define GH_B(F) case F: GH_EACH((bin_apply<F, T>(a[u][e], b[u][e])))
        GH_B(GH_ADD) GH_B(GH_SUB) GH_B(GH_MUL) GH_B(GH_DIV) GH_B(GH_LT) GH_B(GH_LTE) GH_B(GH_GT) GH_B(GH_GTE) GH_B(GH_EQ)
        GH_B(GH_NE)
#undef GH_B
        case GH_MOD: GH_EACH_HEAVY((bin_call<GH_MOD, T>(x, y)))
        case GH_POW:
          // a scalar exponent of 2 is a product, as in the operator's own kernel
          if (s.src_b == kScalar && b[0][0] == (T)2) { GH_EACH(a[u][e] * a[u][e]) }
          GH_EACH_HEAVY((bin_call<GH_POW, T>(x, y)))
#define GH_U(F) case kUnary + F: GH_EACH(unary_apply<F>(a[u][e]))
        GH_U(GH_ABS) GH_U(GH_SIGN) GH_U(GH_CEIL) GH_U(GH_FLOOR) GH_U(GH_NEG) GH_U(GH_SQUARE) GH_U(GH_CUBE)
#undef GH_U
        // float32 tanh and sigmoid are some twenty instructions, the float64 ones library calls
#define GH_U(F) case kUnary + F: if constexpr (sizeof(T) == 4) { GH_EACH(unary_apply<F>(a[u][e])) } else { GH_EACH_HEAVY(unary_call<F>(x)) }
        GH_U(GH_TANH) GH_U(GH_SIGMOID)
#undef GH_U
#define GH_U(F) case kUnary + F: GH_EACH_HEAVY(unary_call<F>(x))
        GH_U(GH_SIN) GH_U(GH_COS) GH_U(GH_EXP) GH_U(GH_LN) GH_U(GH_LOG2) GH_U(GH_SQRT) GH_U(GH_INVERSE) GH_U(GH_INVSQRT)
        GH_U(GH_LOG1P) GH_U(GH_EXPM1) GH_U(GH_SOFTPLUS)
#undef GH_U
        case kRelu: GH_EACH(relu_of(a[u][e]))
        case kLeaky: GH_EACH(leaky_of(a[u][e], (T)s.alpha))
        case kReluBwd: GH_EACH(b[u][e] * (a[u][e] >= (T)0 ? (T)1 : (T)0))
#undef GH_EACH
#undef GH_EACH_HEAVY
      }
      if (s.save) {
#pragma unroll
        for (int u = 0; u < kU; u++) slots[s.save - 1][u][threadIdx.x] = acc[u];   // read back by this thread only
      }
      if (s.store) {
#pragma unroll
        for (int u = 0; u < kU; u++) L::store(s.store, at[u], c.n, acc[u]);
      }
    }
  }
}

// ---- what can be one run -------------------------------------------------------------

// One command's part in a run: a value computed from a and b, element by element, and written to d.
struct Elem {
  uint64_t a, b, d;       // b is 0 where there is one operand
  int64_t n, mid, inner;  // mid, inner: of a small b (or a, where small_a)
  int fn;
  double alpha;
  bool scalar_a, scalar_b, small_a, small_b;
};

bool as_elem(const gh_cmd& c, Elem* e) {
  *e = Elem{};
  const bool f64 = gh_dtype_of(c.flags) == GH_F64;
  if (gh_dtype_of(c.flags) > GH_F64) return false;
  switch (c.opcode) {
    case GH_OP_ELEM_BIN: {
      const uint32_t mode = gh_mode(c.flags);
      if (mode > GH_SV || gh_fn(c.flags) >= GH_BINFN__COUNT) return false;
      e->fn = (int)gh_fn(c.flags);
      e->a = c.ptr[0]; e->b = c.ptr[1];
      e->scalar_a = mode == GH_SV; e->scalar_b = mode == GH_VS;
      e->d = c.ptr[2] ? c.ptr[2] : e->scalar_a ? c.ptr[1] : c.ptr[0];
      e->n = c.dim[0];
      break;
    }
    case GH_OP_ELEM_UNARY:
      if (gh_fn(c.flags) >= GH_UNARYFN__COUNT) return false;
      e->fn = kUnary + (int)gh_fn(c.flags);
      e->a = c.ptr[0]; e->d = c.ptr[1] ? c.ptr[1] : c.ptr[0];
      e->n = c.dim[0];
      break;
    case GH_OP_BCAST_BIN: {
      if (gh_fn(c.flags) >= GH_BINFN__COUNT || c.dim[0] < 0 || c.dim[1] <= 0 || c.dim[2] <= 0) return false;
      const bool left = c.flags & GH_FLAG_SMALL_LEFT;
      e->fn = (int)gh_fn(c.flags);
      e->a = left ? c.ptr[2] : c.ptr[1]; e->b = left ? c.ptr[1] : c.ptr[2];
      e->small_a = left; e->small_b = !left;
      e->d = c.ptr[0];
      e->mid = c.dim[1]; e->inner = c.dim[2];
      e->n = c.dim[0] * c.dim[1] * c.dim[2];
      break;
    }
    case GH_OP_RELU:
    case GH_OP_LEAKY_RELU:
      e->fn = c.opcode == GH_OP_RELU ? kRelu : kLeaky;
      e->a = c.ptr[0]; e->d = c.ptr[1];
      e->n = c.dim[0];
      if (f64) memcpy(&e->alpha, &c.dim[1], 8);
      else e->alpha = c.f[0];
      break;
    case GH_OP_RELU_BWD:
      e->fn = kReluBwd;
      e->a = c.ptr[0]; e->b = c.ptr[1]; e->d = c.ptr[2];
      e->n = c.dim[0];
      break;
    default: return false;
  }
  if (!e->a || !e->d || ((e->fn < kUnary || e->fn == kReluBwd) && !e->b)) return false;
  // whole vectors from the first element on; element numbers in 32 bits
  if (e->n <= 0 || e->n > INT32_MAX || (e->d & 15)) return false;
  if (!e->scalar_a && !e->small_a && (e->a & 15)) return false;
  if (e->b && !e->scalar_b && !e->small_b && (e->b & 15)) return false;
  return true;
}

// Memory one operand covers.
struct Range { uint64_t lo, hi; bool tensor, written; };

// Adds an operand to the run's ranges; false where the run cannot hold it: what a run writes is either one
// whole tensor of the run (then every thread sees its own elements in order) or apart from all it touches.
bool add_range(Range* r, int* count, uint64_t lo, int64_t bytes, bool tensor, bool written) {
  const uint64_t hi = lo + (uint64_t)bytes;
  int same = -1;
  for (int i = 0; i < *count; i++) {
    if (hi <= r[i].lo || r[i].hi <= lo) continue;
    if (r[i].lo == lo && r[i].tensor && tensor) { same = i; continue; }
    if (written || r[i].written) return false;
  }
  if (same >= 0) { r[same].written |= written; return true; }
  r[(*count)++] = Range{lo, hi, tensor, written};
  return true;
}

void reciprocal(uint32_t d, uint32_t* mul, uint32_t* sh) {   // of fast_div
  uint32_t l = 0;
  while (l < 32 && (1ull << l) < d) l++;
  *sh = l;
  *mul = (uint32_t)(((1ull << 32) * ((1ull << l) - d)) / d + 1);
}

// The run's steps: where each operand comes from, what is kept for later and what is stored.  False where a
// value would have to be kept and no slot is free.
bool plan(const Elem* e, int count, int item, Chain* c) {
  const int N = 16 / item;
  uint64_t slot_of[kSlots] = {};   // the tensor whose value a slot holds
  uint64_t acc_of = 0;
  c->n = e[0].n;
  c->steps = count;
  for (int k = 0; k < count; k++) {
    const Elem& x = e[k];
    Step& s = c->step[k];
    s = Step{};
    s.a = (const void*)(uintptr_t)x.a;
    s.b = (const void*)(uintptr_t)x.b;
    s.alpha = x.alpha;
    s.fn = (uint8_t)x.fn;
    auto source = [&](uint64_t p, bool scalar, bool small) -> uint8_t {
      if (scalar) return kScalar;
      if (small) return x.inner == 1 && x.mid % N == 0 && (p & 15) == 0 ? kSmallVec : kSmallAny;
      if (p == acc_of) return kAcc;
      for (int i = 0; i < kSlots; i++)
        if (slot_of[i] == p) return (uint8_t)(kSlot0 + i);
      return kMem;
    };
    s.src_a = source(x.a, x.scalar_a, x.small_a);
    s.src_b = x.b ? source(x.b, x.scalar_b, x.small_b) : (uint8_t)kAcc;
    if (x.small_a || x.small_b) {
      s.mid = (uint32_t)x.mid;
      reciprocal((uint32_t)x.mid, &s.mid_mul, &s.mid_sh);
      reciprocal((uint32_t)x.inner, &s.inner_mul, &s.inner_sh);
    }
    for (int i = 0; i < kSlots; i++)
      if (slot_of[i] == x.d) slot_of[i] = 0;   // overwritten
    // is this value read past the next step, and is it still there when the run ends?
    auto reads = [&](const Elem& y, uint64_t p) {
      return (y.a == p && !y.scalar_a && !y.small_a) || (y.b == p && !y.scalar_b && !y.small_b);
    };
    bool later = false, over = false;
    for (int j = k + 1; j < count && !over; j++) {
      if (j > k + 1 && reads(e[j], x.d)) later = true;
      if (e[j].d == x.d) over = true;
    }
    if (!over) s.store = (void*)(uintptr_t)x.d;
    for (int i = 0; i < kSlots; i++) {   // slots nothing reads any more
      if (!slot_of[i]) continue;
      bool live = false;
      for (int j = k + 1; j < count && !live; j++) {
        if (reads(e[j], slot_of[i])) live = true;
        else if (e[j].d == slot_of[i]) break;
      }
      if (!live) slot_of[i] = 0;
    }
    if (later) {
      int free_slot = -1;
      for (int i = 0; i < kSlots; i++)
        if (!slot_of[i]) free_slot = i;
      if (free_slot < 0) return false;
      slot_of[free_slot] = x.d;
      s.save = (uint8_t)(free_slot + 1);
    }
    acc_of = x.d;
  }
  return true;
}

// Whether the run is quicker than its commands one by one.  Up to 16 MiB a tensor the launches it saves decide, and
// commands that have nothing to do with each other gain as well (eight multiplications on their own tensors, float32: 14
// against 30 us at 2 MiB a tensor, 68 against 77 at 16 MiB); of four and more commands up to 32 MiB (float64, four
// negations 47 against 52 us, eight 91 against 104, but two multiplications 36 against 34).  Larger tensors are bound by
// memory, which more streams in one kernel only slow down (eight multiplications at 64 MiB: 287 against 263 us; eight
// exponentials 223 against 187): there a run has to save a tenth of the passes over memory (two commands, one reading
// what the other wrote, save a quarter: 36 against 45 us; two that only read the same tensor: 42 against 41).
constexpr int64_t kLaunchBound = 16 << 20;

// What a command earns by joining a run, in percent of the launch (of large tensors: the pass over memory) that a run
// costs.  A function of few instructions earns the whole of its own launch or pass.  One of many costs more in the run than
// by itself, a call for each of a thread's elements in turn, and the long ones as much as they save: two in one launch
// against two launches, float32, 2^10 to 2^24 elements: sin, cos, ln, log2 0.87 to 1.0 times as fast, log1p 0.80 to 1.0,
// softplus 0.65 to 1.06, pow 0.52 to 0.96, exp and expm1 1.14 to 1.07 below 4 MiB and 0.90 to 1.0 from there;
// float64: pow 0.79 to 0.98, softplus 0.90 to 1.15, tanh 0.98 to 1.1, the others above 1.06.  With one command of few
// instructions all gain (1.0 to 1.7) but float32 pow below 16 MiB (x * y, then pow: 0.81 to 0.95), which two of them carry.
// A scalar exponent is 2 more often than not, which makes pow a product: only the kernel knows.
int earns(const Elem& x, int item) {
  const bool f64 = item == 8, small = x.n * item < (4 << 20), large = x.n * item >= (16 << 20);
  switch (x.fn) {
    case GH_POW: return x.scalar_b ? 50 : f64 ? 10 : large ? 27 : -55;
    case kUnary + GH_SOFTPLUS: return f64 ? (small ? 45 : 55) : large ? 55 : small ? 0 : 45;
    case kUnary + GH_TANH: return f64 ? 55 : 105;
    case kUnary + GH_EXP: case kUnary + GH_EXPM1: return f64 ? 105 : small ? 75 : 45;
    case kUnary + GH_LOG1P: return f64 ? 60 : small ? 28 : 45;
    case kUnary + GH_SIN: case kUnary + GH_COS: case kUnary + GH_LN: case kUnary + GH_LOG2: return f64 ? 105 : 45;
    default: return 105;
  }
}

bool pays(const Elem* e, int count, int item, const Chain& c) {
  int earned = 0;
  for (int k = 0; k < count; k++) earned += earns(e[k], item);
  if (earned <= 100) return false;
  if (e[0].n * item <= (count >= 4 ? 2 : 1) * kLaunchBound) return true;
  int apart = 0, together = 0;   // tensors read and written
  for (int k = 0; k < count; k++) {
    apart += 1 + (!e[k].scalar_a && !e[k].small_a) + (e[k].b && !e[k].scalar_b && !e[k].small_b);
    together += (c.step[k].src_a == kMem) + (e[k].b && c.step[k].src_b == kMem) + (c.step[k].store != nullptr);
  }
  return 10 * together <= 9 * apart;
}

// The longest run at the front of cmds that one pass can take and pays for; its plan in *c.
int find_run(const gh_cmd* cmds, int n, Chain* c) {
  Elem e[kMaxSteps];
  Range r[3 * kMaxSteps];
  int count = 0, ranges = 0;
  const uint32_t dtype = gh_dtype_of(cmds[0].flags);
  const int item = dtype == GH_F64 ? 8 : 4;
  for (; count < n && count < kMaxSteps; count++) {
    Elem& x = e[count];
    if (gh_dtype_of(cmds[count].flags) != dtype || !as_elem(cmds[count], &x) || x.n != e[0].n) break;
    const int64_t whole = x.n * item;
    const bool ok = add_range(r, &ranges, x.a, x.scalar_a ? item : x.small_a ? x.mid * item : whole, !x.scalar_a && !x.small_a, false) &&
                    (!x.b || add_range(r, &ranges, x.b, x.scalar_b ? item : x.small_b ? x.mid * item : whole, !x.scalar_b && !x.small_b, false)) &&
                    add_range(r, &ranges, x.d, whole, true, true);
    if (!ok) break;
  }
  while (count >= 2 && !(plan(e, count, item, c) && pays(e, count, item, *c))) count--;
  return count >= 2 ? count : 0;
}

template <class T, bool STREAM, int N, int U>
void launch_as(gh_ctx* ctx, const Chain& c, int64_t most) {
  const int64_t nv = (c.n + N - 1) / N, blocks = (nv + kBlock * U - 1) / (kBlock * U);
  hipLaunchKernelGGL((k_chain<T, STREAM, N, U>), dim3((unsigned)std::min(blocks, most)), dim3(kBlock), 0, ctx->stream, c);
}

// A thread's share.  What a run of few elements takes is a thread's way through the steps, so as long as that leaves a compute
// unit no more than five workgroups a thread has one element; above, one vector, and the whole run a launch of that many
// workgroups.  The pow-free chain at the head of this file, us with the wait, two vectors a thread and at most sixteen
// workgroups to a compute unit / as here: float32 1024 values 20.1 / 15.1, 131072 21.1 / 15.8, 262144 21.2 / 17.0, 524288
// 17.8 / 17.0 (one element 19.8, one vector 19.5 where the power is no product), 2097152 21.6 / 20.8, 16777216 74.3 / 71.2,
// 33554432 138 / 128.  float64 keeps two vectors and the bounded launch for tensors beyond 16 MiB (8388608 values 106, one
// vector 114 to 124; 2097152 36 either way, 524288 21.4 / 20.0, 10001 20.0 / 15.6).
template <class T>
void launch(gh_ctx* ctx, const Chain& c, bool stream) {
  constexpr int N = VecOf<T>::N;
  if (c.n <= 5 * (int64_t)ctx->cu_count * kBlock) return launch_as<T, false, 1, 1>(ctx, c, INT32_MAX);
  if constexpr (sizeof(T) == 8) {
    const int64_t most = 16 * (int64_t)ctx->cu_count;
    if (stream) return launch_as<T, true, N, 2>(ctx, c, most);
    if (c.n * (int64_t)sizeof(T) > (16 << 20)) return launch_as<T, false, N, 2>(ctx, c, most);
  } else if (stream) {
    return launch_as<T, true, N, 1>(ctx, c, INT32_MAX);
  }
  launch_as<T, false, N, 1>(ctx, c, INT32_MAX);
}

}  // namespace

int gh_chain_length(const gh_cmd* cmds, int n) {
  Chain c;
  return n >= 2 ? find_run(cmds, n, &c) : 0;
}

extern "C" int gh_elementwise_run(const gh_cmd* cmds, int n) {
  return n > 0 && cmds ? std::max(1, gh_chain_length(cmds, n)) : 0;
}

int gh_launch_chain(gh_ctx* ctx, const gh_cmd* cmds, int count) {
  Chain c;
  if (find_run(cmds, count, &c) != count) return gh_fail(ctx, GH_EINVAL, "not a run of elementwise commands");
  const bool f64 = gh_dtype_of(cmds[0].flags) == GH_F64;
  const int64_t tensor = c.n * (f64 ? 8 : 4);
  int64_t bytes = 0;
  bool cold = true;
  for (int k = 0; k < count; k++) {
    const Step& s = c.step[k];
    const void* in[2] = {s.src_a == kMem ? s.a : nullptr, s.src_b == kMem ? s.b : nullptr};
    for (const void* p : in)
      if (p) { bytes += tensor; cold = cold && gh_llc_cold(ctx, (uint64_t)(uintptr_t)p); }
    if (s.store) bytes += tensor;
  }
  const bool stream = gh_llc_stream(bytes, cold);
  for (int k = 0; k < count; k++) {
    const Step& s = c.step[k];
    if (s.src_a == kMem) ctx->llc.touch((uint64_t)(uintptr_t)s.a, tensor, true);
    if (s.src_b == kMem) ctx->llc.touch((uint64_t)(uintptr_t)s.b, tensor, true);
    if (s.store) ctx->llc.touch((uint64_t)(uintptr_t)s.store, tensor, true);
  }
  if (f64) launch<double>(ctx, c, stream);
  else launch<float>(ctx, c, stream);
  return gh_check_hip(ctx, hipGetLastError(), "elementwise run launch");
}
