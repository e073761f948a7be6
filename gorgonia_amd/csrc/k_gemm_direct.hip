// Matrix products with operands taken from memory straight into the lanes of the 16x16x4 MFMA.
//
// A workgroup owns a tile of 16 TM x 16 TN results and its wavefronts, four or eight (waves_of), each sum their share of K
// over the whole tile: chunks 2 w and 2 w + 1 of every 8 or 16, of KC = 4 KQ consecutive k.  Lane (i, q) holds, of every row of A and column of B it
// feeds, the KQ values k0 + KQ q ... - one 16-byte load where k runs along memory - and MFMA step t takes element
// t of both, so it does not matter that a step's four k are KQ apart.  Where k does not run along memory, a lane
// takes V = KQ neighbouring rows (columns) per k instead, also 16 bytes, and its V tiles are interleaved: tile e
// of a group holds every V-th row.  Nothing is staged and no barrier stands in the loop; the loads of a chunk
// stand among the MFMAs of the chunk in front of it.  The wavefronts' sums meet in LDS in wavefront order.
//
// Against the LDS-tiled kernels: no tile staging to hide with a second workgroup, so one large tile per compute
// unit runs at the rate of many, any tile height in steps of 16 is to be had, and a product is cut so that its
// tiles come out just under a multiple of the compute units (gemm_direct_tile).
#include <algorithm>

#include "gh_gemm_direct.h"

namespace {

using gemm_direct::Gemm;

template <class T, int kWaves, int TM, int TN, bool kSplitK, bool kTA, bool kTB>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(kWaves == 8 || TM * TN * sizeof(T) <= 160 ? 2 : 1))) void k_gemm_direct(const Gemm<T> g) {
  __shared__ __attribute__((aligned(16))) char lds[gemm_direct::lds_of<T, kWaves, TN, kSplitK>()];
  gemm_direct::workgroup<T, kWaves, TM, TN, kSplitK, kTA, kTB>(g, (int)(blockIdx.y * gridDim.x + blockIdx.x), (int)gridDim.x, (int)gridDim.y, (int)blockIdx.z, lds);
}

template <class T, int W, int TM, int TN, bool kSplitK>
void launch_along_k(gh_ctx* ctx, const Gemm<T>& g, dim3 grid) {
  if constexpr (sizeof(T) == 4 || W == 4) hipLaunchKernelGGL((k_gemm_direct<T, W, TM, TN, kSplitK, false, true>), grid, dim3(W * 64), 0, ctx->stream, g);
}

template <class T, int W, int TM, int TN, bool kSplitK = true>
void launch(gh_ctx* ctx, const Gemm<T>& g, int batch, bool ta, bool tb) {
  constexpr int rows = 16 * TM * (kSplitK ? 1 : W);
  const dim3 grid((unsigned)((g.N + 16 * TN - 1) / (16 * TN)), (unsigned)((g.M + rows - 1) / rows), (unsigned)batch);
  if (ta && tb) hipLaunchKernelGGL((k_gemm_direct<T, W, TM, TN, kSplitK, true, true>), grid, dim3(W * 64), 0, ctx->stream, g);
  else if (ta) hipLaunchKernelGGL((k_gemm_direct<T, W, TM, TN, kSplitK, true, false>), grid, dim3(W * 64), 0, ctx->stream, g);
  else if (tb) launch_along_k<T, W, TM, TN, kSplitK>(ctx, g, grid);
  else hipLaunchKernelGGL((k_gemm_direct<T, W, TM, TN, kSplitK, false, false>), grid, dim3(W * 64), 0, ctx->stream, g);
}

}  // namespace

// The forms: rows x columns of a workgroup's tile in sixteens, whether its wavefronts split K, and what a multiple of
// the compute units' worth of such tiles takes: us per 16 x 16 results and 1000 of K, and per 16 x 16 results
// (measured over square and ragged products of 100 to 4096; the estimates are within 10 % of the times).
struct Form { int tm, tn; bool split; double per_k, per_tile; };
static const Form kForms32[] = {{2, 4, true, 1.40, 0.12}, {3, 4, true, 1.28, 0.12}, {4, 4, true, 1.25, 0.12},
                                {5, 4, true, 1.22, 0.12}, {4, 4, false, 1.45, 0.06}, {8, 4, false, 1.25, 0.06}};
static const Form kForms64[] = {{2, 2, true, 2.28, 0.17}, {2, 4, true, 2.00, 0.17}, {3, 4, true, 1.92, 0.17}, {4, 4, true, 1.94, 0.17},
                                {5, 4, true, 1.90, 0.17}};

// Whether k_gemm_direct takes a product - at least one whole group of rows and columns, a tile's offsets in 32 bits -
// and the quickest form for it: its number, its time in *us and its rounds of tiles over the compute units.
int gh_gemm_direct_form(const gh_cmd& c, int cus, double* us, int* rounds) {
  const bool f64 = gh_dtype_of(c.flags) == GH_F64;
  const int64_t M = c.dim[0], N = c.dim[1], K = c.dim[2], batch = c.dim[6] <= 0 ? 1 : c.dim[6];
  const int v = f64 ? 2 : 4;
  if (M < v || N < v || batch > 65535 || std::max(c.dim[3], c.dim[4]) * (f64 ? 8 : 4) >= ((int64_t)1 << 31) / 160) return -1;
  const bool along_k = !(c.flags & GH_FLAG_TRANS_A) && (c.flags & GH_FLAG_TRANS_B);   // both operands: half lines per load
  const Form* forms = f64 ? kForms64 : kForms32;
  const int n = f64 ? 5 : 6;
  int best = -1;
  for (int i = 0; i < n; i++) {
    const Form& f = forms[i];
    if (!f64 && f.split && K <= 128) continue;   // four pairs of chunks: half of eight wavefronts would have none
    const int64_t tiles = (M + 16 * f.tm - 1) / (16 * f.tm) * ((N + 16 * f.tn - 1) / (16 * f.tn)) * batch;
    const double per_k = f.per_k * (f64 && along_k && f.tm == 2 ? (f.tn == 2 ? 1.5 : 1.3) : 1.0);
    const double est = 4.0 + (double)((tiles + cus - 1) / cus) * f.tm * f.tn * ((double)K * 1e-3 * per_k + f.per_tile);
    if (best >= 0 && est >= *us) continue;
    *us = est;
    best = i;
    if (rounds) *rounds = (int)((tiles + cus - 1) / cus);
  }
  return best;
}

// K slices of a form: the wavefronts' shares.  One tile per compute unit has eight wavefronts: with four, a chunk's MFMAs are over
// before the next chunk's loads are.  float64, whose MFMAs take twice as long, gains from K = 640 on (us, four / eight: 113 x 1444,
// K = 1480 21.4 / 14.4, 370 x 661, K = 860 13.3 / 10.5, 1061 x 281, K = 1180 22.1 / 21.5; 777 x 1543, K = 1021 equal) and below loses to the
// longer meeting (1863 x 388, K = 458 20.6 / 21.2, 764 x 1563, K = 152 13.4 / 14.1).  Both operands along K, an input gradient's form,
// stay with four: 97 x 1954, K = 713 12.1 / 11.8, but 20.0 / 21.5 beside the weight gradient in one launch.
static int waves_of(const gh_cmd& c, const Form& f, int cus) {
  if (!f.split) return 1;
  const int64_t tiles = (c.dim[0] + 16 * f.tm - 1) / (16 * f.tm) * ((c.dim[1] + 16 * f.tn - 1) / (16 * f.tn)) * std::max<int64_t>(1, c.dim[6]);
  const bool along_k = !(c.flags & GH_FLAG_TRANS_A) && (c.flags & GH_FLAG_TRANS_B);
  return tiles <= cus && (gh_dtype_of(c.flags) != GH_F64 || (c.dim[2] >= 640 && !along_k)) ? 8 : 4;
}
int gh_gemm_direct_slices(const gh_cmd& c, int form, int cus) {
  return waves_of(c, (gh_dtype_of(c.flags) == GH_F64 ? kForms64 : kForms32)[form], cus);
}

int gh_launch_gemm_direct(gh_ctx* ctx, const gh_cmd& c, int form) {
  const bool ta = c.flags & GH_FLAG_TRANS_A, tb = c.flags & GH_FLAG_TRANS_B;
  int batch;
  if (gh_dtype_of(c.flags) == GH_F64) {
    const Gemm<double> g = gemm_direct::gemm_of<double>(c, &batch);
    const bool eight = waves_of(c, kForms64[form], ctx->cu_count) == 8;
    switch (form) {
      case 0: eight ? launch<double, 8, 2, 2>(ctx, g, batch, ta, tb) : launch<double, 4, 2, 2>(ctx, g, batch, ta, tb); break;
      case 1: eight ? launch<double, 8, 2, 4>(ctx, g, batch, ta, tb) : launch<double, 4, 2, 4>(ctx, g, batch, ta, tb); break;
      case 2: eight ? launch<double, 8, 3, 4>(ctx, g, batch, ta, tb) : launch<double, 4, 3, 4>(ctx, g, batch, ta, tb); break;
      case 3: eight ? launch<double, 8, 4, 4>(ctx, g, batch, ta, tb) : launch<double, 4, 4, 4>(ctx, g, batch, ta, tb); break;
      default: eight ? launch<double, 8, 5, 4>(ctx, g, batch, ta, tb) : launch<double, 4, 5, 4>(ctx, g, batch, ta, tb); break;
    }
  } else {
    const Gemm<float> g = gemm_direct::gemm_of<float>(c, &batch);
    const bool eight = waves_of(c, kForms32[form], ctx->cu_count) == 8;
    switch (form) {
      case 0: eight ? launch<float, 8, 2, 4>(ctx, g, batch, ta, tb) : launch<float, 4, 2, 4>(ctx, g, batch, ta, tb); break;
      case 1: eight ? launch<float, 8, 3, 4>(ctx, g, batch, ta, tb) : launch<float, 4, 3, 4>(ctx, g, batch, ta, tb); break;
      case 2: eight ? launch<float, 8, 4, 4>(ctx, g, batch, ta, tb) : launch<float, 4, 4, 4>(ctx, g, batch, ta, tb); break;
      case 3: eight ? launch<float, 8, 5, 4>(ctx, g, batch, ta, tb) : launch<float, 4, 5, 4>(ctx, g, batch, ta, tb); break;
      case 4: launch<float, 4, 1, 4, false>(ctx, g, batch, ta, tb); break;
      default: launch<float, 4, 2, 4, false>(ctx, g, batch, ta, tb); break;
    }
  }
  return gh_check_hip(ctx, hipGetLastError(), "gemm launch");
}
