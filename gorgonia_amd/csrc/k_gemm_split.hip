// Large float32 products on the bf16 matrix instructions (gh_split.h): eight of their instructions do the work of eight
// float32 ones that take nearly twice the time.
//
// A workgroup owns a tile of the result; the operands' values are split into their bf16 parts on the way from memory to
// LDS, once per workgroup that needs them.  That is what the tile's size buys: at 128 x 128 a lane converts 16 values
// (104 vector instructions) for 32 matrix instructions, at 64 x 64 for 16.  A wavefront issues a vector instruction every
// five cycles under its matrix instructions, if it does not wait for the one before: the stages of several pairs of values
// are interleaved, one to a matrix instruction.  (256 x 256 has no registers for the two sums of a result; 256 x 128 with
// one wavefront to a SIMD takes 1023 us for 4096 x 4096 x 4096, 128 x 128 843.)
// Smaller products have too few such tiles for the compute units: theirs are smaller, and K is cut into parts inside the
// workgroup, each with wavefronts and LDS buffers of its own, whose sums are added in LDS at the end.  Which form runs
// depends on the shape only.
//
// Error against 64-bit sums, of normal / of uniform values in [0, 1), next to the float32 kernel that the shape would run
// on: 4096 x 4096 x 4096 4.0e-7 / 3.0e-7 (k_sgemm 1.14e-6 / 8.4e-7); 2321 x 3480, K = 2049 1.9e-7 / 1.2e-7 (k_gemm_direct in
// four slices 4.1e-7 / 1.6e-7); 1000 x 1000, K = 4000 1.9e-7 / 8.3e-8 (in eight 4.0e-7 / 1.1e-7).  One, two and sixteen
// products to a result 2.53e-8, 2.56e-8 and 3.4e-8 (2.53e-8, 3.1e-8 and 6.0e-8).
//
// Values that the split cannot hold: a workgroup whose sums are not finite computes its tile on the float32 instructions, from
// the step on where it finds that out.  It looks in its third step, every 32 steps, and at the end.  us, beside k_sgemm or
// k_gemm_direct: 4096 x 4096 x 4096 of NaN 1230 (1102), with one row of -FLT_MAX 1372 (1157), with a triangle of it or infinities
// in the last k 2010 and 2131 (1138); 1024 x 1024 x 1024 31, 33, 44 and 45 (25); 64 of 512 x 512 x 512 180, 200, 274 and 304 (160).
#include <algorithm>
#include <type_traits>

#include "gh_conv_common.h"
#include "gh_internal.h"
#include "gh_split.h"

namespace {

using namespace gh_split;

struct Args {
  const float* A; const float* B; float* C;
  int M, N, K, lda, ldb, ldc;
  int64_t sA, sB, sC;
  const float* bias;
  int act; float alpha;
};

constexpr int kStep = 16;   // k of one step: one MFMA's

// An operand's way from memory through registers into LDS: R rows (of A; columns of B) by 16 k.  A unit is eight
// k of one row, 16 bytes a part; a part lies in LDS as [8 k][row], the second half 64 bytes further than it would follow, so
// that the writes of a wavefront, which alternate between the halves, fall into different banks.
template <int R, int NT, bool ALONG_K>
struct Operand {
  static constexpr int kHalf = R + 4, kPart = 2 * kHalf, kUnits = 3 * kPart;   // in 16-byte units
  static constexpr int kPer = 2 * R / NT;
  static_assert(2 * R % NT == 0, "whole units per thread");
  const float* base; int ld;
  uint32_t off[kPer];
  int k_at[kPer], slot[kPer];
  float reg[kPer][8];
  __device__ __forceinline__ void prep(const float* p, int ld_, int r0, int rmax, int tid) {
    ld = ld_;
    base = ALONG_K ? p + (int64_t)r0 * ld : p + r0;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
      const int u = tid + j * NT;
      const int row = ALONG_K ? u >> 1 : u % R, half = ALONG_K ? u & 1 : u / R;
      const int r = min(row, rmax - 1 - r0);   // rows past the end are the last one again and not stored
      k_at[j] = 8 * half;
      off[j] = ALONG_K ? (uint32_t)(r * ld + 8 * half) : (uint32_t)(8 * half * ld + r);
      slot[j] = half * kHalf + row;
    }
  }
  // unit j of the step at k0; k0 ... k0 + 15 are all there
  __device__ __forceinline__ void load(int j, int k0) {
    const float* const b = base + (ALONG_K ? (int64_t)k0 : (int64_t)k0 * ld);
    if constexpr (ALONG_K) {
      const f32x4 lo = *(const f32x4_a4*)(b + off[j]), hi = *(const f32x4_a4*)(b + off[j] + 4);
#pragma unroll
      for (int e = 0; e < 4; e++) { reg[j][e] = lo[e]; reg[j][4 + e] = hi[e]; }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) reg[j][e] = (b + (int64_t)e * ld)[off[j]];
    }
  }
  // those from kmax on are zero (and read from the last one's place)
  __device__ __forceinline__ void load_end(int j, int k0, int kmax) {
    const float* const b = base + (ALONG_K ? (int64_t)k0 : (int64_t)k0 * ld);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int past = max(k0 + k_at[j] + e - (kmax - 1), 0);
      const float v = b[(int64_t)off[j] + (int64_t)(e - past) * (ALONG_K ? 1 : ld)];
      reg[j][e] = past ? 0.0f : v;
    }
  }
  // the values as they are, as [k][row] with rows kRows floats long
  static constexpr int kRows = R + 4;
  __device__ __forceinline__ void put32(float* lds) const {
#pragma unroll
    for (int j = 0; j < kPer; j++) {
      float* const p = lds + k_at[j] * kRows + slot[j] - k_at[j] / 8 * kHalf;
#pragma unroll
      for (int e = 0; e < 8; e++) p[e * kRows] = reg[j][e];
    }
  }
  // stage K of pair I of a thread's values; the last stage of a unit's last pair stores the unit
  static constexpr int kPairs = 4 * kPer;
  u32x4 part[kPer][3];
  Pair pairs[kPairs];
  template <int I, int K>
  __device__ __forceinline__ void convert(u32x4* lds) {
    constexpr int j = I / 4, e = I % 4;
    pairs[I].template stage<K>(reg[j][2 * e], reg[j][2 * e + 1]);
    if constexpr (K == 1 || K == 4 || K == 7) {
      part[j][K / 3][e] = pairs[I].part[K / 3];
      if constexpr (e == 3) lds[(K / 3) * kPart + slot[j]] = part[j][K / 3];
    }
  }
};

// sixteen results of a 32 x 32 tile: the rows i, i + 1, i + 2, i + 3, i + 8, ... of column j
__device__ __forceinline__ void put(const Args& g, float* C, int i, int j, f32x16 v, float scale, float bias) {
#pragma unroll
  for (int e = 0; e < 16; e++) v[e] = v[e] * scale + bias;
  if (g.act == 1) {
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = act_apply(v[e], 1, g.alpha);
  } else if (g.act == 2) {
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = act_apply(v[e], 2, g.alpha);
  }
  if (j >= g.N) return;
  float* const p = C + (int64_t)i * g.ldc + j;
#pragma unroll
  for (int e = 0; e < 16; e++)
    if (i + 8 * (e / 4) + e % 4 < g.M) p[(int64_t)(8 * (e / 4) + e % 4) * g.ldc] = v[e];
}

template <int WM, int WN, int TM, int TN, int KS, bool TA, bool TB>
__global__ __launch_bounds__(WM * WN * KS * 64, 2) void k_gemm_split(Args g) {
  constexpr int NT = WM * WN * 64, BM = WM * TM * 32, BN = WN * TN * 32;
  using OA = Operand<BM, NT, !TA>;
  using OB = Operand<BN, NT, TB>;
  constexpr int kBuf = OA::kUnits + OB::kUnits;
  __shared__ u32x4 shared[3 * kBuf * KS];

  // tiles in groups of eight tile rows, each XCD one contiguous run of the whole launch
  const int gx = (g.N + BN - 1) / BN, gy = (g.M + BM - 1) / BM, all = (int)gridDim.x;
  int id = (int)blockIdx.x;
  if (all % 8 == 0) id = (id % 8) * (all / 8) + id / 8;
  const int bz = id / (gx * gy);
  id -= bz * gx * gy;
  const int first = id / (8 * gx) * 8, gsz = min(gy - first, 8), in = id % (8 * gx);
  const int m0 = (first + in % gsz) * BM, n0 = (in / gsz) * BN;

  const int tid = (int)threadIdx.x % NT, part = KS > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT) : 0;
  const int lane = tid & 63, wave = tid >> 6;
  u32x4* const lds = shared + part * (3 * kBuf);
  const int wm = (wave / WN) * (TM * 32), wn = (wave % WN) * (TN * 32);
  const int lr = lane & 31, lh = lane >> 5;
  const float* const pa = g.A + bz * g.sA;
  const float* const pb = g.B + bz * g.sB;

  OA oa; OB ob;
  oa.prep(pa, g.lda, m0, g.M, tid);
  ob.prep(pb, g.ldb, n0, g.N, tid);

  f32x16 acc[TM][TN], low[TM][TN];   // the products of the first parts; the seven smaller ones
  auto clear = [&](f32x16 (&v)[TM][TN]) {
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) v[a][b] = f32x16{};
  };
  auto fold = [&] {
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) acc[a][b] += low[a][b];
  };
  clear(acc);
  clear(low);
  // whether a sum of this wavefront is infinite or NaN, for the whole workgroup behind its next barrier
  __shared__ int lost;
  if (threadIdx.x == 0) lost = 0;
  auto look = [&] {
    float zero = 0.0f;   // stays 0 where every sum is finite
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int v = 0; v < 16; v++) zero = __builtin_fmaf(acc[a][b][v], 0.0f, zero);
    if (__any(zero != 0.0f) && lane == 0) lost = 1;
  };

  // the parts take the steps in turn: this one's step s is the product's step s KS + part (zeros behind the last one)
  const int full = g.K / kStep / KS, steps = (g.K + kStep * KS - 1) / (kStep * KS);
  auto k_of = [&](int s) { return (s * KS + part) * kStep; };
  auto load = [&](int s) {
#pragma unroll
    for (int j = 0; j < OA::kPer; j++) s < full ? oa.load(j, k_of(s)) : oa.load_end(j, k_of(s), g.K);
#pragma unroll
    for (int j = 0; j < OB::kPer; j++) s < full ? ob.load(j, k_of(s)) : ob.load_end(j, k_of(s), g.K);
  };
  for (int s = 0; s < 2 && s < steps; s++) {
    load(s);
    each<OA::kPairs * kStages>([&](auto i) { oa.template convert<decltype(i)::value / kStages, decltype(i)::value % kStages>(lds + s * kBuf); });
    each<OB::kPairs * kStages>([&](auto i) { ob.template convert<decltype(i)::value / kStages, decltype(i)::value % kStages>(lds + s * kBuf + OA::kUnits); });
  }
  if (steps > 2) load(2);
  __syncthreads();

  // One step: the products of LDS buffer s mod 3.  Its first operands were read at the end of the step before; the step
  // reads the next one's, converts the values of the step after that, which were loaded a step ago, and loads into the
  // registers that this leaves free the step behind those.  So a load has the time of a whole step, one barrier a step is
  // enough, and no wavefront waits for LDS behind it.  The order is pinned: what is not a matrix instruction goes in
  // small pieces behind them.
  const int at_a = lh * OA::kHalf + wm + lr, at_b = OA::kUnits + lh * OB::kHalf + wn + lr;
  u32x4 fa[3][TM], fb[3][TN], na[TM], nb[TN];   // part 2 of A comes first, part 0 of both last: na, nb
  auto read_a = [&](const u32x4* buf, int p, int a) { return buf[at_a + p * OA::kPart + a * 32]; };
  auto read_b = [&](const u32x4* buf, int p, int b) { return buf[at_b + p * OB::kPart + b * 32]; };
#pragma unroll
  for (int a = 0; a < TM; a++) na[a] = read_a(lds, 2, a);
#pragma unroll
  for (int b = 0; b < TN; b++) { nb[b] = read_b(lds, 0, b); fb[1][b] = read_b(lds, 1, b); fb[2][b] = read_b(lds, 2, b); }
  u32x4 *cur = lds, *next = lds + kBuf, *then = lds + 2 * kBuf;
  // LOAD: 0 nothing, 1 a whole step, 2 the ragged end of K; CONV: there is a step s + 2
  auto step = [&](int s, auto load_kind, auto conv) {
    constexpr int LOAD = decltype(load_kind)::value;
    constexpr bool CONV = decltype(conv)::value;
    constexpr int T = TM * TN, NM = 8 * T, kPairs = OA::kPairs + OB::kPairs;
#pragma unroll
    for (int a = 0; a < TM; a++) fa[2][a] = na[a];
#pragma unroll
    for (int b = 0; b < TN; b++) fb[0][b] = nb[b];
    each<NM>([&](auto at) {
      constexpr int i = decltype(at)::value;
      // smaller products first: part 2 of A with 1 and 0 of B, 1 with 2, 1 and 0, 0 with 2, 1 and 0
      constexpr int p = i < 2 * T ? 2 : i < 5 * T ? 1 : 0, in = i - (p == 2 ? 0 : p == 1 ? 2 * T : 5 * T), q = (p == 2 ? 1 : 2) - in / T, t = in % T, a = t / TN, b = t % TN;
      if constexpr (p + q > 0) low[a][b] = mfma(fa[p][a], fb[q][b], low[a][b]);
      else acc[a][b] = mfma(fa[p][a], fb[q][b], acc[a][b]);
      if constexpr (i < TM) fa[1][i] = read_a(cur, 1, i);
      if constexpr (i >= T && i < T + TM) fa[0][i - T] = read_a(cur, 0, i - T);
      // operands of the next step as their registers fall free (behind the last step: whatever LDS holds, unused)
      if constexpr (i >= 4 * T && i < 4 * T + TM) na[i - 4 * T] = read_a(next, 2, i - 4 * T);
      if constexpr (i >= 6 * T && i < 6 * T + TN) fb[2][i - 6 * T] = read_b(next, 2, i - 6 * T);
      if constexpr (i >= 7 * T && i < 7 * T + TN) { fb[1][i - 7 * T] = read_b(next, 1, i - 7 * T); nb[i - 7 * T] = read_b(next, 0, i - 7 * T); }
      if constexpr (CONV) {
        // pair c begins behind instruction c kLast / (kPairs - 1), a stage to an instruction; the last stores have some
        // instructions to go before the barrier waits for them
        constexpr int kLast = NM - kStages - (NM >= 24 ? 4 : 0);
        each<kPairs>([&](auto n) {
          constexpr int c = decltype(n)::value, k = i - c * kLast / (kPairs - 1), d = c - OA::kPairs;
          if constexpr (k >= 0 && k < kStages) {
            if constexpr (c < OA::kPairs) oa.template convert<c, k>(then);
            else ob.template convert<d, k>(then + OA::kUnits);
          }
          if constexpr (k == 0 && c % 4 == 3) {   // a unit's values are taken: the loads of the step behind
            if constexpr (c < OA::kPairs && LOAD == 1) oa.load(c / 4, k_of(s + 3));
            if constexpr (c < OA::kPairs && LOAD == 2) oa.load_end(c / 4, k_of(s + 3), g.K);
            if constexpr (c >= OA::kPairs && LOAD == 1) ob.load(d / 4, k_of(s + 3));
            if constexpr (c >= OA::kPairs && LOAD == 2) ob.load_end(d / 4, k_of(s + 3), g.K);
          }
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    __syncthreads();
    u32x4* const was = cur;
    cur = next; next = then; then = was;
  };
  using Yes = std::true_type; using No = std::false_type;
  int s = 0;
  bool again = false;
  for (; s + 3 < full && !again; s++) {
    // (early, for operands that are infinite or NaN throughout, and now and then; 1 % of the time)
    const bool looks = s % 32 == 2;
    if (looks) look();
    step(s, std::integral_constant<int, 1>{}, Yes{});
    if (looks) again = lost;
  }
  if (!again) {
    for (; s + 3 < steps; s++) step(s, std::integral_constant<int, 2>{}, Yes{});
    for (; s + 2 < steps; s++) step(s, std::integral_constant<int, 0>{}, Yes{});
    for (; s < steps; s++) step(s, std::integral_constant<int, 0>{}, No{});
  }

  // the parts' sums, in the order of the parts, to those of part 0
  static_assert((KS - 1) * BM * BN * 4 <= (int)sizeof(shared), "the parts' sums fit");
  auto gather = [&] {
    if constexpr (KS > 1) {
      __syncthreads();   // LDS is free
      float* const sums = (float*)shared;
      if (part) {
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
          for (int b = 0; b < TN; b++)
#pragma unroll
            for (int v = 0; v < 16; v++) sums[((((part - 1) * TM + a) * TN + b) * 16 + v) * NT + tid] = acc[a][b][v];
      }
      __syncthreads();
      if (!part) {
#pragma unroll
        for (int p = 0; p < KS - 1; p++)
#pragma unroll
          for (int a = 0; a < TM; a++)
#pragma unroll
            for (int b = 0; b < TN; b++)
#pragma unroll
              for (int v = 0; v < 16; v++) acc[a][b][v] += sums[(((p * TM + a) * TN + b) * 16 + v) * NT + tid];
      }
    }
  };
  if (!again) {
    fold();
    gather();
    look();
    __syncthreads();
    again = lost;
  }
  float scale = kDown;
  if (again) {
    // The tile with the float32 instructions, its operands staged as they are, in two buffers; a chain of 256 k at a time.
    constexpr int kTile = kStep * (OA::kRows + OB::kRows);
    static_assert(2 * kTile <= 4 * 3 * kBuf, "two steps of float32 operands fit");
    float* const mine = (float*)lds;
    scale = 1.0f;
    clear(acc);
    clear(low);
    load(0);
    for (int r = 0; r < steps; r++) {
      float* const buf = mine + (r & 1) * kTile;
      oa.put32(buf);
      ob.put32(buf + kStep * OA::kRows);
      if (r + 1 < steps) load(r + 1);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < kStep; k += 2) {
        float xa[TM], xb[TN];
#pragma unroll
        for (int a = 0; a < TM; a++) xa[a] = buf[(k + lh) * OA::kRows + wm + a * 32 + lr];
#pragma unroll
        for (int b = 0; b < TN; b++) xb[b] = buf[(kStep * OA::kRows) + (k + lh) * OB::kRows + wn + b * 32 + lr];
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
          for (int b = 0; b < TN; b++) low[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[a], xb[b], low[a][b], 0, 0, 0);
      }
      if (r % 16 == 15) { fold(); clear(low); }
    }
    fold();
    gather();
  }
  if (part) return;

  float* const C = g.C + bz * g.sC;
#pragma unroll
  for (int b = 0; b < TN; b++) {
    const int j = n0 + wn + b * 32 + lr;
    const float bias = g.bias && j < g.N ? g.bias[j] : -0.0f;
#pragma unroll
    for (int a = 0; a < TM; a++) put(g, C, m0 + wm + a * 32 + 4 * lh, j, acc[a][b], scale, bias);
  }
}

template <int WM, int WN, int TM, int TN, int KS>
void launch(hipStream_t stream, const Args& g, int batch, bool ta, bool tb) {
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
  const dim3 grid((unsigned)((int64_t)((g.N + BN - 1) / BN) * ((g.M + BM - 1) / BM) * batch)), block(WM * WN * KS * 64);
  if (ta && tb) hipLaunchKernelGGL((k_gemm_split<WM, WN, TM, TN, KS, true, true>), grid, block, 0, stream, g);
  else if (ta) hipLaunchKernelGGL((k_gemm_split<WM, WN, TM, TN, KS, true, false>), grid, block, 0, stream, g);
  else if (tb) hipLaunchKernelGGL((k_gemm_split<WM, WN, TM, TN, KS, false, true>), grid, block, 0, stream, g);
  else hipLaunchKernelGGL((k_gemm_split<WM, WN, TM, TN, KS, false, false>), grid, block, 0, stream, g);
}

}  // namespace

// The forms: rows and columns of a workgroup's tile, parts of K inside the workgroup, workgroups that share a compute
// unit, and their times in us: per tile and step of 16 k (of each part) with a compute unit full of workgroups, the
// same for those that do not fill one (per_odd once, and for each of them), per tile, and once.  Fitted to 318 products of 64 to
// 4096 a side and batches of up to 64, each run for 12 ms; nine in ten of the estimates are between 0.87 and 1.11 of the times,
// those above 200 us, where the clock comes down, between 0.81 and 0.99.  4096 x 4096 x 4096 takes 843 us on 128 x 128 tiles
// (float32 instructions 1202) and 1082 on 64 x 64, where every wavefront converts more of what it multiplies; 2048 x 2048 x 2048
// 115 with K in two parts, 123 in one (float32 153); 64 of 512 x 512 x 512 116 (151); 1024 x 1024 x 1024 22 with K in four parts (26).
struct Form { int rows, cols, parts, share; double per_step, per_odd, per_tile, start; };
static const Form kForms[] = {{128, 128, 1, 2, 0.69, 0.38, 2.8, 3.5}, {128, 128, 2, 1, 1.41, 0, 7.3, 0}, {64, 64, 2, 2, 0.495, 0.34, 1.75, 2.6},
                              {64, 64, 4, 1, 1.01, 0, 4.6, 1.0}};

// The form for a float32 product whose quickest kernel on the float32 instructions takes other_us by its estimate and cuts K
// into other_slices sums, or -1.
//
// A sum of n roundings is off by about sqrt(n) of one, cut into p parts by sqrt(n) / p: 2.0e-8 sqrt(n) / p for uniform values
// on either kind of instruction.  Here n is K / 16, there K / 2, so that p has to be 0.35 of the other's slices at least for an
// error below the other kernel's (2321 x 3480, K = 2049 of uniform values: 2.2e-7 in one part, 1.2e-7 in two, 1.6e-7 on
// k_gemm_direct in four).
//
// Below 9 us the launch and the first loads are what either kernel takes, and the estimates no help (1241 x 199,
// K = 90 6.4 us against 6.0).  Of 318 products offered to the rule it takes 214, together in 0.75 of the time; at 0.95 of the other
// estimate and less eight of them are slower, by 1 to 4 %.
int gh_gemm_split_form(const gh_cmd& c, int cus, double other_us, int other_slices) {
  const int64_t M = c.dim[0], N = c.dim[1], K = c.dim[2], batch = c.dim[6] <= 0 ? 1 : c.dim[6];
  // at least one whole step; offsets inside a tile in 32 bits; a launch of one dimension
  if (K < kStep || std::max(c.dim[3], c.dim[4]) >= (int64_t)1 << 21 || std::max(M, N) >= (int64_t)1 << 30 || (M + 63) / 64 * ((N + 63) / 64) * batch >= (int64_t)1 << 30) return -1;
  int best = -1;
  double us = 0.95 * other_us;
  if (us < 9.0) return -1;
  for (int i = 0; i < (int)(sizeof(kForms) / sizeof(kForms[0])); i++) {
    const Form& f = kForms[i];
    if (8 * f.parts * f.parts < other_slices * other_slices) continue;
    const int64_t tiles = (M + f.rows - 1) / f.rows * ((N + f.cols - 1) / f.cols) * batch, steps = (K + kStep * f.parts - 1) / (kStep * f.parts);
    const int64_t each = (tiles + cus - 1) / cus, odd = each % f.share, whole = each - odd;
    const double est = f.start + (double)steps * ((double)whole * f.per_step + (odd ? (1.0 + (double)odd) * f.per_odd : 0.0)) + (double)each * f.per_tile;
    if (est < us) { us = est; best = i; }
  }
  return best;
}

int gh_launch_gemm_split(gh_ctx* ctx, const gh_cmd& c, int form) {
  Args g;
  g.A = (const float*)(uintptr_t)c.ptr[0]; g.B = (const float*)(uintptr_t)c.ptr[1]; g.C = (float*)(uintptr_t)c.ptr[2];
  g.M = (int)c.dim[0]; g.N = (int)c.dim[1]; g.K = (int)c.dim[2];
  g.lda = (int)c.dim[3]; g.ldb = (int)c.dim[4]; g.ldc = (int)c.dim[5];
  const int batch = c.dim[6] <= 0 ? 1 : (int)c.dim[6];
  g.sA = batch > 1 ? c.dim[7] : 0; g.sB = batch > 1 ? c.dim[8] : 0; g.sC = batch > 1 ? c.dim[9] : 0;
  g.bias = (c.flags & GH_FLAG_GEMM_BIAS) ? (const float*)(uintptr_t)c.ptr[3] : nullptr;
  g.act = (c.flags & GH_FLAG_ACT_RELU) ? 1 : (c.flags & GH_FLAG_ACT_LEAKY) ? 2 : 0;
  g.alpha = c.f[0];
  const bool ta = c.flags & GH_FLAG_TRANS_A, tb = c.flags & GH_FLAG_TRANS_B;
  switch (form) {
    case 0: launch<2, 2, 2, 2, 1>(ctx->stream, g, batch, ta, tb); break;
    case 1: launch<2, 2, 2, 2, 2>(ctx->stream, g, batch, ta, tb); break;
    case 2: launch<1, 2, 2, 1, 2>(ctx->stream, g, batch, ta, tb); break;
    default: launch<1, 2, 2, 1, 4>(ctx->stream, g, batch, ta, tb); break;
  }
  return gh_check_hip(ctx, hipGetLastError(), "gemm launch");
}
