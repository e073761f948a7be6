// Sums of slabs of partial results, for the launch that adds them up (k_slab_sums.hip) and the solver steps that take the sums
// they need along (k_solver.hip).
#pragma once
#include "gh_internal.h"

namespace slab_sums {

struct Batch {
  const void* ws[kSlabSums];
  void* out[kSlabSums];
  int64_t total[kSlabSums];
  int slabs[kSlabSums], how[kSlabSums], first[kSlabSums + 1];   // sum t has the workgroups [first[t], first[t + 1])
};

// RW results to a workgroup; its 256 / RW thread groups take every G-th slab (reads of a slab are RW values wide), and the
// groups' sums are added pairwise, neighbours first.
template <class T, int RW, class Put>
__device__ __forceinline__ void by_groups(const T* __restrict__ ws, int slabs, int64_t total, int block, T* sh, Put&& put) {
  constexpr int G = 256 / RW;
  const int grp = threadIdx.x / RW;
  const int64_t e = (int64_t)block * RW + threadIdx.x % RW;
  T sum = (T)0;
  if (e < total) {
    int s = grp;
    for (; s + 3 * G < slabs; s += 4 * G) {   // four loads in flight
      T v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) v[u] = ws[(int64_t)(s + u * G) * total + e];
#pragma unroll
      for (int u = 0; u < 4; u++) sum = sum + v[u];
    }
    for (; s < slabs; s += G) sum = sum + ws[(int64_t)s * total + e];
  }
  sh[threadIdx.x] = sum;
  for (int d = 1; d < G; d <<= 1) {
    __syncthreads();
    T v = (T)0;
    const bool mine = grp % (2 * d) == 0;
    if (mine) v = sh[threadIdx.x] + sh[threadIdx.x + d * RW];
    __syncthreads();
    if (mine) sh[threadIdx.x] = v;
  }
  if (grp == 0 && e < total) put(e, sh[threadIdx.x]);
}

// Many slabs, few results: L lanes share one result.  Lane q adds slabs q, q + L, q + 2 L, ... in that order, then the L
// sums are combined pairwise, neighbours first.
template <int L, class Put>
__device__ __forceinline__ void by_lanes(const float* __restrict__ ws, int slabs, int64_t total, int block, Put&& put) {
  const int q = threadIdx.x & (L - 1);
  const int64_t e = ((int64_t)block * 256 + threadIdx.x) / L;
  float acc = 0.f;
  if (e < total) {
    const float* p = ws + (int64_t)q * total + e;
    int s = q;
    for (; s + 3 * L < slabs; s += 4 * L) {   // four loads in flight
      const float v0 = p[0], v1 = p[(int64_t)L * total], v2 = p[2 * (int64_t)L * total], v3 = p[3 * (int64_t)L * total];
      acc = acc + v0; acc = acc + v1; acc = acc + v2; acc = acc + v3;
      p += 4 * (int64_t)L * total;
    }
    for (; s < slabs; s += L) { acc = acc + p[0]; p += (int64_t)L * total; }
  }
  float sum = acc;
#pragma unroll
  for (int d = 1; d < L; d <<= 1) sum = sum + __shfl_xor(sum, d, 64);   // commutative per level: every lane ends with the total
  if (e < total && q == 0) put(e, sum);
}

// A workgroup of 256 threads' part of sum t: put(e, result e), by the thread that has it.  sh: 2 KB.
template <class T, class Put>
__device__ __forceinline__ void workgroup(const Batch& b, int t, int block, double* sh, Put&& put) {
  const int slabs = b.slabs[t];
  const int64_t total = b.total[t];
  const T* const ws = (const T*)b.ws[t];
  if constexpr (sizeof(T) == 8) {
    if (b.how[t] == kSumGroups64F64) by_groups<double, 64>(ws, slabs, total, block, sh, put);
    else by_groups<double, 16>(ws, slabs, total, block, sh, put);
  } else {
    switch (b.how[t]) {
      case kSumGroups64: by_groups<float, 64>(ws, slabs, total, block, (float*)sh, put); break;
      case kSumGroups16: by_groups<float, 16>(ws, slabs, total, block, (float*)sh, put); break;
      case kSumLanes16: by_lanes<16>(ws, slabs, total, block, put); break;
      case kSumLanes4: by_lanes<4>(ws, slabs, total, block, put); break;
      default: {
        const int64_t e = (int64_t)block * 256 + threadIdx.x;
        if (e >= total) break;
        float acc = ws[e];
        for (int s = 1; s < slabs; s++) acc = acc + ws[(int64_t)s * total + e];
        put(e, acc);
      }
    }
  }
}

inline int64_t item(int how) { return how == kSumGroups64F64 || how == kSumGroups16F64 ? 8 : 4; }

inline int results_of_block(int how) {
  switch (how) {
    case kSumGroups64: case kSumGroups64F64: case kSumLanes4: return 64;
    case kSumGroups16: case kSumGroups16F64: case kSumLanes16: return 16;
    default: return 256;
  }
}

// The batch of n sums, and its workgroups.
inline int batch_of(const gh_slab_sum* sums, int n, Batch* b) {
  *b = Batch{};
  int blocks = 0;
  for (int i = 0; i < n; i++) {
    b->ws[i] = sums[i].ws;
    b->out[i] = sums[i].out;
    b->total[i] = sums[i].total;
    b->slabs[i] = sums[i].slabs;
    b->how[i] = sums[i].how;
    b->first[i] = blocks;
    const int r = results_of_block(sums[i].how);
    blocks += (int)((sums[i].total + r - 1) / r);
  }
  for (int i = n; i <= kSlabSums; i++) b->first[i] = blocks;
  return blocks;
}

}  // namespace slab_sums
