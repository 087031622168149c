// Argument block and helpers shared by the GEMM kernels (gemm.hip,
// gemm_stream.hip).
#pragma once

#include "svla_common.h"

namespace svla_gemm {

enum AMode { A_DENSE = 0, A_PSHUF = 1, A_PATCH = 2 };
// EPI_PART: fp32 partial tiles of a K split (gemm_stream.hip)
enum Epi { EPI_STORE = 0, EPI_ROPE = 1, EPI_SILU = 2, EPI_EULER = 3, EPI_PART = 4 };

struct GemmArgs {
  const bf16* a;
  long lda;
  // A_PSHUF: source [n_img, grid*grid, hidden], shuffle factor `scale`
  int g_grid, g_hidden, g_scale;
  // A_PATCH: images [n_img, chans, img, img], patch size
  int p_chans, p_img, p_patch;
  const bf16* b;
  long ldb;
  void* c;
  long ldc;
  int M, N, K;
  float alpha;
  const bf16* bias;
  const float* bias_f32;
  const bf16* res;
  long ldr;
  const bf16* rowadd;  // added after rounding: rowadd[(m % rowadd_period) * N + n]
  int rowadd_period;
  int out_f32;
  const float* rope_cos;
  const float* rope_sin;
  int rope_cols;
  int rope_period;
  bf16* c_lo;  // ROPE (optional): o - bf16(o) of every rotated column, layout of c
  float* x_f32;
  long ldx;
  bf16* x_bf16;
  long ldxb;
  float dt;
  // output row remap: row m is stored at (m / c_rpg) * c_gstride + m % c_rpg
  // (c_rpg == 0: identity).  Lets the connector write each sample's image
  // tokens straight into its slot of the [B, prefix_len, H] prefix buffer.
  int c_rpg;
  long c_gstride;
  // fused RMSNorm of the A rows: a = bf16((x * r) * w[k]), r = 1 / sqrt(mean(x^2) + eps)
  const bf16* norm_w;
  float norm_eps;
  // skinny split-K (gridDim.z > 1): fp32 partial tiles [tile][split][BM * BN]
  // and one arrival counter per output tile (zero between calls)
  float* ws;
  unsigned* ws_cnt;
  // persistent wide kernel: the tile grid (its launch grid is one workgroup per
  // CU); w_cn > 0: each XCD keeps w_cn column blocks (see xcd_tile), else the
  // grouped order of tile_coords
  int tiles_m, tiles_n, w_cn;
  // slab-blocked operands / output of the wide kernel: element (row, k) of a
  // blocked [rows, K] matrix sits at (k / 32) * rows * 32 + row * 32 + k % 32,
  // so the 16 rows x 32 columns an LDS-DMA instruction fetches are one
  // contiguous kilobyte (the row-major layout gives 16 separate 64-byte pieces)
  int a_blk, b_blk, c_blk;
  // second product of a pair (gemm_small_kernel, blockIdx.z == 1)
  const bf16 *a2, *b2;
  void* c2;
};

__device__ __forceinline__ long crow(const GemmArgs& p, int m) {
  if (p.c_rpg <= 0) return m;
  const int g = m / p.c_rpg;
  return (long)g * p.c_gstride + (m - g * p.c_rpg);
}

template <int ACT>
__device__ __forceinline__ float apply_act(float v) {
  if constexpr (ACT == SVLA_ACT_GELU_TANH) return gelu_tanh_f(v);
  else if constexpr (ACT == SVLA_ACT_GELU_ERF) return gelu_erf_f(v);
  else if constexpr (ACT == SVLA_ACT_SILU) return silu_f(v);
  else return v;
}

__device__ __forceinline__ void store_bf16x4(bf16* dst, const float v[4]) {
  bf16x4 o;
  o[0] = f2bf(v[0]); o[1] = f2bf(v[1]); o[2] = f2bf(v[2]); o[3] = f2bf(v[3]);
  *reinterpret_cast<bf16x4*>(dst) = o;
}

__device__ __forceinline__ void load_bf16x4(const bf16* src, float v[4]) {
  bf16x4 t = *reinterpret_cast<const bf16x4*>(src);
  v[0] = bf2f(t[0]); v[1] = bf2f(t[1]); v[2] = bf2f(t[2]); v[3] = bf2f(t[3]);
}

constexpr int kNumXCD = 8;

// Maps the hardware workgroup id so that consecutive logical tiles share an
// XCD (the hardware deals workgroups round-robin over the 8 XCDs).
__device__ __forceinline__ int xcd_remap(int bid, int total) {
  const int per = total / kNumXCD;
  const int full = per * kNumXCD;
  if (bid >= full) return bid;
  return (bid % kNumXCD) * per + bid / kNumXCD;
}

// Logical tile -> (row block, column block) in groups of kGroupRows row
// blocks: consecutive tiles walk down a group's rows, then across its
// columns, so the workgroups that run together on one XCD cover a compact
// rows x columns patch and share both their A row panels and their weight
// column panels in that XCD's L2.  (Row-major order makes a concurrent set
// span every column block, i.e. the whole weight matrix, which does not fit.)
constexpr int kGroupRows = 8;
__device__ __forceinline__ void tile_coords(int t, int gm, int gn, int& tm, int& tn) {
  const int per_group = kGroupRows * gn;
  const int group = t / per_group;
  const int first = group * kGroupRows;
  const int rows = min(gm - first, kGroupRows);
  const int r = t - group * per_group;
  tm = first + r % rows;
  tn = r / rows;
}

// gemm_stream.hip: the K-split line-DMA kernels for mid-size dense problems.
// stream_takes: whether they can serve a problem (no launch); stream_tile: the
// tile they choose (rows * 1000 + columns); stream_run: the launch (SVLA_OK or
// an error).
__attribute__((visibility("hidden"))) bool stream_takes(const GemmArgs& p, int epi);
__attribute__((visibility("hidden"))) int stream_tile(int M, int N, int K, int epi);
__attribute__((visibility("hidden"))) int stream_run(const GemmArgs& p, int epi, int act,
                                                     hipStream_t s);

// The gathers (pixel shuffle, patches) on the same kernels: tile and K splits of
// a problem with room for ws_floats floats of split-K partial tiles (0: no
// split; force > 0: that many splits, as far as K and the room allow), the
// tile's sizes (rows * 1000 + columns), and the launch (p.ws: the room).
struct GatherPlan {
  int cfg, splits;
};
__attribute__((visibility("hidden"))) bool gather_takes(const GemmArgs& p);
__attribute__((visibility("hidden"))) GatherPlan gather_plan(int M, int N, int K, long ws_floats,
                                                             int force);
__attribute__((visibility("hidden"))) int gather_tile(const GatherPlan& g);
__attribute__((visibility("hidden"))) int gather_run(const GemmArgs& p, int amode,
                                                     const GatherPlan& g, hipStream_t s);

}  // namespace svla_gemm
