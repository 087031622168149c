// Mid-size bf16 MFMA GEMM for gfx950: K-split workgroups on a line-DMA ring.
//
//   C[M, N] = epilogue(alpha * A[M, K] . W[N, K]^T)     (dense A, W)
//
// For the problems between the skinny tiles and the 256x256 kernel (the
// expert and prefix at batch > 1, the ViT up to a few images, single layers):
// tens to hundreds of microsecond-sized tiles, where a workgroup's fixed costs
// weigh as much as its K loop.
//
// What bounds it (MI355X, measured with copies of the loop that leave out the
// DMA, the LDS reads or the MFMAs): a CU's LDS-DMA path moves about 57
// bytes/clock from L2 in 128-byte pieces of line-aligned rows, 27 in 64-byte
// pieces and 30 when the rows straddle lines (K = 720, rows of 1440 bytes: the
// expert's Q, QKV and gate|up operands, about 1 us each).  Per 64-deep
// K stage a 128x128 tile needs 575 clocks of DMA and 512 of MFMA; 4 waves that
// each do both halves of a stage in turn (reads, wait, MFMAs) take 1100, since
// one wave per SIMD cannot overlap its own chain.  So:
//  * 8 waves: 4 along the rows x 2 K groups.  Group k takes the k-th 32-deep
//    half of every stage, so a SIMD always has two independent waves and a
//    128x128 stage takes 740-760 clocks.
//  * every wave covers all BN columns of its BM / 4 rows: each activation
//    fragment is read from LDS once, each weight fragment by four waves.
//  * the fragments of stage s + 1 are read into a second register set between
//    the MFMAs of stage s, and the DMA that refills stage s's slot is spread
//    over them; one barrier per stage.  Nothing is fetched past K (a ring that
//    reloads its last stage to keep its counts moves 4 / 12 more bytes at
//    K = 720), and a ragged K is one masked stage in the ring, not a tail of
//    direct loads (a memory round trip, 1 us).
//  * residual tiles are requested before the K loop, bias and RoPE operands
//    before the K groups' partial sums meet in LDS; both groups finish half the
//    columns each, and the output leaves through LDS in whole 16-byte pieces
//    of consecutive columns.
#include <type_traits>

#include "gemm_args.h"

using namespace svla_gemm;

namespace {

constexpr int GK = 64;                     // K per stage
constexpr int GW = 8;                      // waves: 4 row groups x 2 K groups
__device__ __forceinline__ int gswz(int r, int c) { return c ^ (r & 7); }

constexpr int g_waitcnt(int vm, int lgkm) {
  return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8);
}

template <int I, int N, class F>
__device__ __forceinline__ void g_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    g_for<I + 1, N>(f);
  }
}

// Packed weight row (= output column) of column j of a paired problem in unit
// order: unit U = j / 32 holds 16 first-half columns of a 64-column block and
// their 16 partners 32 columns on, so that MFMA tiles 2u, 2u + 1 pair up and
// BN can be any multiple of 32.
__device__ __forceinline__ int pair_col(int j) {
  const int u = j >> 5, q = j & 31;
  return 64 * (u >> 1) + 16 * (u & 1) + (q & 15) + 32 * (q >> 4);
}

// Element offset of A[m][k] = a_row(m) + a_col(k): both gathers separate (k in
// chunks of 8, which neither map splits; the maps are those of a_ptr in
// gemm.hip).  Pixel shuffle: the s tokens of one patch row are adjacent, so
// k runs through s * E contiguous elements, then jumps a token row.  Patches:
// 8 adjacent patches give the 8-row DMA block 4 runs of 256 bytes per stage.
template <int AMODE>
__device__ __forceinline__ long a_row(const GemmArgs& p, int m) {
  if constexpr (AMODE == A_DENSE) {
    return (long)m * p.lda;
  } else if constexpr (AMODE == A_PSHUF) {
    const int gs = p.g_grid / p.g_scale, per = gs * gs;
    const int img = m / per, i = m - img * per, hp = i / gs, wp = i - hp * gs;
    return ((long)img * p.g_grid * p.g_grid + (long)p.g_scale * hp * p.g_grid + p.g_scale * wp) *
           p.g_hidden;
  } else {
    const int P = p.p_patch, H = p.p_img, G = H / P, per = G * G;
    const int img = m / per, t = m - img * per, pr = t / G, pc = t - pr * G;
    return ((long)img * p.p_chans * H + pr * P) * H + pc * P;
  }
}
template <int AMODE>
__device__ __forceinline__ long a_col(const GemmArgs& p, int k) {
  if constexpr (AMODE == A_DENSE) {
    return k;
  } else if constexpr (AMODE == A_PSHUF) {
    const int sE = p.g_scale * p.g_hidden, t = k / sE;
    return (long)t * p.g_grid * p.g_hidden + (k - t * sE);
  } else {
    const int P = p.p_patch, P2 = P * P, ch = k / P2, r = k - ch * P2, ky = r / P;
    return ((long)ch * p.p_img + ky) * p.p_img + (r - ky * P);
  }
}

template <int BM, int BN, int WMW, int KG, int ST, int MINB, int AMODE, int EPI, int ACT>
__global__ __launch_bounds__(GW * 64, 2 * MINB) void gemm_stream_kernel(GemmArgs p) {
  constexpr bool PAIRED = EPI == EPI_ROPE || EPI == EPI_SILU;
  static_assert(AMODE == A_DENSE || (BM % 64 == 0 && (EPI == EPI_STORE || EPI == EPI_PART)), "gathers");
  constexpr int WNW = GW / WMW / KG;                 // waves along the columns
  constexpr int WM = BM / WMW, WN = BN / WNW;        // wave tile
  constexpr int TM = WM / 16, TN = WN / 16, NF = TM + TN, NM = TM * TN;
  constexpr int STAGE = (BM + BN) * GK;              // bf16 per stage
  constexpr int TD = (BM + BN) / 8;                  // 1 KB (8-row) DMA blocks per stage
  constexpr int ND = (TD + GW - 1) / GW;             // per wave; the last may be missing
  // column tiles K group 0 finishes (all without a K split)
  constexpr int H0 = KG == 1 ? TN : PAIRED ? (TN / 2 + 1) / 2 * 2 : (TN + 1) / 2;
  constexpr int BNO = EPI == EPI_SILU ? BN / 2 : BN;  // output columns
  constexpr int LDO = BNO + 8;                        // staged output row
  constexpr int PPR = BNO / 8, NP = (BM * PPR + GW * 64 - 1) / (GW * 64);  // 16-byte pieces
  static_assert(WMW * WNW * KG == GW && BM % (16 * WMW) == 0 && BN % (16 * WNW) == 0 &&
                    (!PAIRED || WN % 32 == 0),
                "tile shape");
  static_assert(ST >= 2 && ST <= 5 && (ST - 1) * ND < 63, "ring");
  constexpr int RING = ST * STAGE;
  constexpr int EX = KG == 1 ? 0 : BM * BN * 2;       // fp32 exchange, in bf16 elements
  constexpr int OUT = BM * LDO * (EPI == EPI_ROPE ? 2 : 1);
  constexpr int LDS = RING > EX ? (RING > OUT ? RING : OUT) : (EX > OUT ? EX : OUT);
  __shared__ __attribute__((aligned(1024))) bf16 sh[LDS];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = KG == 1 ? 0 : wave / (WMW * WNW);
  const int wm = wave / WNW % WMW, wn = wave % WNW;
  const int fr = lane & 15, g = lane >> 4;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  int tm_idx, tn_idx;
  tile_coords(tile, p.tiles_m, p.tiles_n, tm_idx, tn_idx);
  const int m0 = tm_idx * BM, n0 = tn_idx * BN;
  // this workgroup's K stages: all, or split blockIdx.z of gridDim.z (EPI_PART)
  const int nk_all = (p.K + GK - 1) / GK;
  const int kt0 = EPI == EPI_PART ? (int)((long)nk_all * blockIdx.z / gridDim.z) : 0;
  const int nk = EPI == EPI_PART ? (int)((long)nk_all * (blockIdx.z + 1) / gridDim.z) - kt0 : nk_all;

  // residual pieces of this thread's stores: requested before the K loop at one
  // workgroup per CU, after it at two (registers; the other workgroup covers)
  bf16x8 rsd[NP];
  auto load_res = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int q = tid + i * GW * 64, r = q / PPR, c = q - r * PPR;
      const int m = min(m0 + r, p.M - 1), n = min(n0 + c * 8, p.N - 8);
      rsd[i] = ld8(AMODE == A_PATCH ? p.rowadd + (long)(m % p.rowadd_period) * p.N + n
                                    : p.res + (long)m * p.ldr + n);
    }
  };
  // (the patch embedding's addend is its position table)
  const bool addend = EPI == EPI_STORE && (AMODE == A_PATCH ? p.rowadd : p.res) != nullptr;
  if (MINB == 1 && addend) load_res();

  // DMA block j * 8 + wave of a stage: rows 8 blk .. + 7 of [A | W], 8 lanes
  // per 128-byte row piece, chunk c of row r in slot gswz(r, c)
  const bool all = TD % GW == 0 || wave < TD % GW;  // wave-uniform: ND or ND - 1 blocks
  const bf16* src[ND];
  const int chunk = gswz(lane >> 3, lane & 7) * 8;  // (8-row blocks: r & 7 = lane / 8)
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    const int r = min(j * GW + wave, TD - 1) * 8 + (lane >> 3);
    if (r < BM) {
      src[j] = p.a + a_row<AMODE>(p, min(m0 + r, p.M - 1));
    } else {
      const int c = n0 + r - BM;
      src[j] = p.b + (long)min(PAIRED ? pair_col(c) : c, p.N - 1) * p.ldb;
    }
  }
  auto dma = [&](int slot, int kt, int j) __attribute__((always_inline)) {
    if (TD % GW != 0 && j == ND - 1 && !all) return;  // wave-uniform
    // chunks past K reload the row's last one (masked before the MFMAs)
    const int k = min((kt0 + kt) * GK + chunk, p.K - 8);
    const long off = AMODE != A_DENSE && j < BM / 64 ? a_col<AMODE>(p, k) : k;  // (blocks < BM / 8: A)
    __builtin_amdgcn_global_load_lds((void*)(src[j] + off),
                                     (lds_ptr_t)(sh + slot * STAGE + (j * GW + wave) * 512), 16, 0,
                                     0);
  };

  bf16x8 fr_[2][NF];  // two register sets; fragment f < TN: weight tile, else activation tile
  // half h (32 deep) of the stage in `slot`
  auto read = [&](auto RC, auto FC, int slot, int h) __attribute__((always_inline)) {
    constexpr int R = decltype(RC)::value, f = decltype(FC)::value;
    const int row = f < TN ? BM + wn * WN + f * 16 + fr : wm * WM + (f - TN) * 16 + fr;
    fr_[R][f] = *reinterpret_cast<const bf16x8*>(sh + slot * STAGE + row * GK +
                                                 gswz(fr, 4 * h + g) * 8);
  };
  f32x4 acc[NM];  // column tile i % TN, row tile i / TN
#pragma unroll
  for (int i = 0; i < NM; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mma = [&](auto RC, auto IC) __attribute__((always_inline)) {
    constexpr int R = decltype(RC)::value, i = decltype(IC)::value;
    acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fr_[R][i % TN], fr_[R][TN + i / TN], acc[i], 0,
                                                     0, 0);
  };

  // wait until all but the `newer` most recent stages have landed and this
  // wave's LDS reads are complete (a slot refilled after the barrier must not
  // be overwritten under a pending read), then the barrier
  auto wait = [&](int newer) __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    g_for<0, ST>([&](auto NC) __attribute__((always_inline)) {
      constexpr int n = decltype(NC)::value;
      if (newer == n) {
        if (all) __builtin_amdgcn_s_waitcnt(g_waitcnt(n * ND, 0));
        else __builtin_amdgcn_s_waitcnt(g_waitcnt(n * (ND - 1), 0));
      }
    });
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // MFMAs on set R; between them the reads of half h of the stage in slot sn
  // into the other set and, FILL, the DMA of stage kt into slot s
  auto segment = [&](auto RC, int sn, int h, auto FILL, int s, int kt) __attribute__((always_inline)) {
    constexpr int R = decltype(RC)::value;
    constexpr int RM = NM > 1 ? (NM + 1) / 2 : 1;  // reads spread over the first half
    g_for<0, NM>([&](auto IC) __attribute__((always_inline)) {
      constexpr int i = decltype(IC)::value;
      mma(RC, IC);
      constexpr int r0 = i * NF / RM < NF ? i * NF / RM : NF;
      constexpr int r1 = (i + 1) * NF / RM < NF ? (i + 1) * NF / RM : NF;
      g_for<r0, r1>([&](auto FC) __attribute__((always_inline)) {
        read(std::integral_constant<int, 1 - R>{}, FC, sn, h);
      });
      if constexpr (decltype(FILL)::value) {
        g_for<i * ND / NM, (i + 1) * ND / NM>(
            [&](auto JC) __attribute__((always_inline)) { dma(s, kt, decltype(JC)::value); });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  using Y = std::true_type;
  using N = std::false_type;
  // the last stage: fragments past K are zero in both operands
  auto mask = [&](auto RC, int h) __attribute__((always_inline)) {
    constexpr int R = decltype(RC)::value;
    if ((kt0 + nk - 1) * GK + (4 * h + g) * 8 >= p.K) {
#pragma unroll
      for (int f = 0; f < NF; ++f) fr_[R][f] = bf16x8{};
    }
  };
  auto mma_all = [&](auto RC) __attribute__((always_inline)) {
    g_for<0, NM>([&](auto IC) __attribute__((always_inline)) { mma(RC, IC); });
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  auto nxt = [](int s) __attribute__((always_inline)) { return s == ST - 1 ? 0 : s + 1; };

#pragma unroll
  for (int s = 0; s < ST; ++s) {
    if (s >= nk) break;
#pragma unroll
    for (int j = 0; j < ND; ++j) dma(s, s, j);
  }
  wait(min(ST, nk) - 1);
  g_for<0, NF>([&](auto FC) __attribute__((always_inline)) { read(I0{}, FC, 0, kg); });
  int kt = 0, s = 0;
  if constexpr (KG == 1) {
    // both halves of a stage in turn: half 0 is in set 0 on entry
    for (; kt + 1 < nk; ++kt) {
      asm volatile("" ::: "memory");
      segment(I0{}, s, 1, N{}, 0, 0);
      wait(min(ST - 2, nk - 2 - kt));
      const int sn = nxt(s);
      if (kt + ST < nk) segment(I1{}, sn, 0, Y{}, s, kt + ST);
      else segment(I1{}, sn, 0, N{}, 0, 0);
      s = sn;
    }
    mask(I0{}, 0);
    segment(I0{}, s, 1, N{}, 0, 0);
    mask(I1{}, 1);
    mma_all(I1{});
  } else {
    // one half of every stage: the register sets alternate by stage
    auto step = [&](auto RC, int kt, int s, int sn) __attribute__((always_inline)) {
      wait(min(ST - 2, nk - 2 - kt));
      if (kt + ST < nk) segment(RC, sn, kg, Y{}, s, kt + ST);
      else segment(RC, sn, kg, N{}, 0, 0);
    };
    for (; kt + 2 < nk; kt += 2) {
      const int s1 = nxt(s), s2 = nxt(s1);
      step(I0{}, kt, s, s1);
      step(I1{}, kt + 1, s1, s2);
      s = s2;
    }
    if (kt + 2 == nk) {
      step(I0{}, kt, s, nxt(s));
      mask(I1{}, kg);
      mma_all(I1{});
    } else {
      mask(I0{}, kg);
      mma_all(I0{});
    }
  }

  // ---- epilogue -------------------------------------------------------------
  // operands of the column tiles this K group finishes, [t0, t1)
  const int t0 = kg == 0 ? 0 : H0;  // (uniform)
  constexpr int HT = H0 > TN - H0 ? H0 : TN - H0;
  auto ccol = [&](int t) __attribute__((always_inline)) {  // first column of tile t, this lane
    const int j = n0 + wn * WN + t * 16 + 4 * g;
    return PAIRED ? pair_col(j) : j;
  };
  f32x4 eu[PAIRED ? (HT / 2) * TM : HT], ew[EPI == EPI_ROPE ? (HT / 2) * TM : 1];
  if constexpr (EPI == EPI_STORE) {
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      const int n = min(ccol(t0 + h), p.N - 4);
      eu[h] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (p.bias) {
        const bf16x4 b = *reinterpret_cast<const bf16x4*>(p.bias + n);
#pragma unroll
        for (int i = 0; i < 4; ++i) eu[h][i] = bf2f(b[i]);
      }
      if (p.bias_f32) eu[h] += *reinterpret_cast<const f32x4*>(p.bias_f32 + n);
    }
  } else if constexpr (EPI == EPI_ROPE) {
#pragma unroll
    for (int h = 0; h < HT / 2; ++h)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        const int pos = min(m0 + wm * WM + tm * 16 + fr, p.M - 1) % p.rope_period;
        const int d = ccol(t0 + 2 * h) & 31;
        eu[h * TM + tm] = *reinterpret_cast<const f32x4*>(p.rope_cos + pos * 32 + d);
        ew[h * TM + tm] = *reinterpret_cast<const f32x4*>(p.rope_sin + pos * 32 + d);
      }
  }
  __syncthreads();  // every wave is done with the ring
  if constexpr (KG == 2) {
    // the K groups' partial sums meet: each hands the other's column tiles over
    float* ex = reinterpret_cast<float*>(sh) + wave % (WMW * WNW) * (NM * 256);
#pragma unroll
    for (int i = 0; i < NM; ++i)
      if ((i % TN < H0) == (kg == 1))
        *reinterpret_cast<f32x4*>(ex + i * 256 + lane * 4) = acc[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NM; ++i)
      if ((i % TN < H0) == (kg == 0))
        acc[i] += *reinterpret_cast<const f32x4*>(ex + i * 256 + lane * 4);
    __syncthreads();  // exchange read: the space takes the output
  }
  if constexpr (EPI == EPI_PART) {
    // fp32 partial tile of this split, [split][M][N]
    float* part = p.ws + (long)blockIdx.z * p.M * p.N;
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      const int t = i % TN, m = m0 + wm * WM + i / TN * 16 + fr, n = ccol(t);
      if ((KG == 2 && (t < H0) != (kg == 0)) || m >= p.M || n >= p.N) continue;
      *reinterpret_cast<f32x4*>(part + (long)m * p.N + n) = acc[i];
    }
    return;
  }
  auto stage = [&](int row, int col, const float (&v)[4], int half) __attribute__((always_inline)) {
    bf16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = f2bf(v[i]);
    *reinterpret_cast<bf16x4*>(sh + half * (BM * LDO) + row * LDO + col) = o;
  };
  auto finish = [&](auto KC) __attribute__((always_inline)) {
    constexpr int T0 = decltype(KC)::value == 0 ? 0 : H0, T1 = decltype(KC)::value == 0 ? H0 : TN;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const int row = wm * WM + tm * 16 + fr;
#pragma unroll
      for (int t = T0; t < T1; t += PAIRED ? 2 : 1) {
        const f32x4 a = acc[tm * TN + t];
        float v[4];
        if constexpr (EPI == EPI_STORE) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[i] = a[i] * p.alpha + eu[t - T0][i];
            if constexpr (ACT != SVLA_ACT_NONE) v[i] = apply_act<ACT>(rbf(v[i]));
          }
          stage(row, wn * WN + t * 16 + 4 * g, v, 0);
        } else {
          const f32x4 b = acc[tm * TN + t + 1];
          if constexpr (EPI == EPI_SILU) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              v[i] = rbf(silu_f(rbf(a[i] * p.alpha))) * rbf(b[i] * p.alpha);
            stage(row, wn * (WN / 2) + t * 8 + 4 * g, v, 0);
          } else {
            // as epi_apply<EPI_ROPE>: fp32 rotation of the bf16 projection,
            // columns past rope_cols as projected, remainders for the rotated
            const bool rot = ccol(t) < p.rope_cols;
            float o2[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float x1 = rbf(a[i] * p.alpha), x2 = rbf(b[i] * p.alpha);
              const float c = eu[(t - T0) / 2 * TM + tm][i], sn = ew[(t - T0) / 2 * TM + tm][i];
              const float r1 = __fsub_rn(__fmul_rn(x1, c), __fmul_rn(x2, sn));
              const float r2 = __fadd_rn(__fmul_rn(x2, c), __fmul_rn(x1, sn));
              v[i] = rot ? r1 : x1;
              o2[i] = rot ? r2 : x2;
            }
            stage(row, wn * WN + t * 16 + 4 * g, v, 0);
            stage(row, wn * WN + t * 16 + 16 + 4 * g, o2, 0);
            if (p.c_lo) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                v[i] = __fsub_rn(v[i], rbf(v[i]));
                o2[i] = __fsub_rn(o2[i], rbf(o2[i]));
              }
              stage(row, wn * WN + t * 16 + 4 * g, v, 1);
              stage(row, wn * WN + t * 16 + 16 + 4 * g, o2, 1);
            }
          }
        }
      }
    }
  };
  if (KG == 1 || kg == 0) finish(I0{});
  else finish(I1{});
  if (MINB > 1 && addend) load_res();
  __syncthreads();
  // whole 16-byte pieces of consecutive columns, row by row
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int q = tid + i * GW * 64, r = q / PPR, c = q - r * PPR;
    const int m = m0 + r;
    const int n = EPI == EPI_SILU ? n0 / 2 + c * 8 : EPI == EPI_ROPE ? pair_col(n0 + c * 8) : n0 + c * 8;
    if (q >= BM * PPR || m >= p.M || n0 * BNO / BN + c * 8 >= p.N * BNO / BN) continue;
    bf16x8 o = *reinterpret_cast<const bf16x8*>(sh + r * LDO + c * 8);
    if (addend) {
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = f2bf(bf2f(o[e]) + bf2f(rsd[i][e]));
    }
    st8(reinterpret_cast<bf16*>(p.c) + (AMODE == A_PSHUF ? crow(p, m) : (long)m) * p.ldc + n, o);
    if (EPI == EPI_ROPE && p.c_lo && n < p.rope_cols)
      st8(p.c_lo + (long)m * p.ldc + n,
          *reinterpret_cast<const bf16x8*>(sh + BM * LDO + r * LDO + c * 8));
  }
}

// Sums the K splits' partial tiles in split order and finishes the rows: bias,
// one rounding, the position table, the row remap.  One thread per 8 columns.
__global__ __launch_bounds__(256) void stream_reduce_kernel(GemmArgs p, int splits) {
  const int per = p.N / 8;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= p.M * per) return;
  const int m = i / per, n = (i - m * per) * 8;
  const float* src = p.ws + (long)m * p.N + n;
  const long step = (long)p.M * p.N;
  f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll 4
  for (int z = 0; z < splits; ++z) {
    a += *reinterpret_cast<const f32x4*>(src + z * step);
    b += *reinterpret_cast<const f32x4*>(src + z * step + 4);
  }
  bf16x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float v = (e < 4 ? a[e & 3] : b[e & 3]) * p.alpha;
    if (p.bias) v += bf2f(p.bias[n + e]);
    if (p.rowadd) v = rbf(v) + bf2f(p.rowadd[(long)(m % p.rowadd_period) * p.N + n + e]);
    o[e] = f2bf(v);
  }
  st8(reinterpret_cast<bf16*>(p.c) + crow(p, m) * p.ldc + n, o);
}

template <int BM, int BN, int WMW, int KG, int ST, int MINB>
int launch_stream(GemmArgs p, int epi, int act, hipStream_t s) {
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  const dim3 grid(p.tiles_m * p.tiles_n), block(GW * 64);
#define SVLA_STREAM(E, A) \
  hipLaunchKernelGGL((gemm_stream_kernel<BM, BN, WMW, KG, ST, MINB, A_DENSE, E, A>), grid, block, 0, s, p)
  if (epi == EPI_STORE) {
    if (act == SVLA_ACT_GELU_TANH) SVLA_STREAM(EPI_STORE, SVLA_ACT_GELU_TANH);
    else if (act == SVLA_ACT_GELU_ERF) SVLA_STREAM(EPI_STORE, SVLA_ACT_GELU_ERF);
    else if (act == SVLA_ACT_SILU) SVLA_STREAM(EPI_STORE, SVLA_ACT_SILU);
    else SVLA_STREAM(EPI_STORE, SVLA_ACT_NONE);
  } else if constexpr (BN / (GW / WMW / KG) % 32 == 0) {
    if (epi == EPI_ROPE) SVLA_STREAM(EPI_ROPE, 0);
    else SVLA_STREAM(EPI_SILU, 0);
  } else {
    return SVLA_EINVAL;
  }
#undef SVLA_STREAM
  SVLA_CHECK_LAUNCH();
  return 0;
}

// The gathers, K split over `splits` workgroups per tile (1: none).
template <int BM, int BN, int WMW, int KG, int ST, int MINB>
int launch_gather(GemmArgs p, int amode, int splits, hipStream_t s) {
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  const dim3 grid(p.tiles_m * p.tiles_n, 1, splits), block(GW * 64);
#define SVLA_GATHER(A, E) \
  hipLaunchKernelGGL((gemm_stream_kernel<BM, BN, WMW, KG, ST, MINB, A, E, 0>), grid, block, 0, s, p)
  if (amode == A_PSHUF) {
    if (splits > 1) SVLA_GATHER(A_PSHUF, EPI_PART);
    else SVLA_GATHER(A_PSHUF, EPI_STORE);
  } else {
    if (splits > 1) SVLA_GATHER(A_PATCH, EPI_PART);
    else SVLA_GATHER(A_PATCH, EPI_STORE);
  }
#undef SVLA_GATHER
  SVLA_CHECK_LAUNCH();
  if (splits > 1) {
    hipLaunchKernelGGL(stream_reduce_kernel, dim3((p.M * (p.N / 8) + 255) / 256), dim3(256), 0, s, p,
                       splits);
    SVLA_CHECK_LAUNCH();
  }
  return 0;
}

// The configurations and what they cost (microseconds): a launch, one round of
// workgroups over the chip's slots (256 CUs x MINB), and each 64-deep stage of
// a round -- with both workgroups of a CU busy, or (two-workgroup tiles) with
// at most one.  Least-squares fits of 40 to 68 problems each (50 to 9127 rows,
// K 320 to 3072, graph replay on MI355X), 6-13% rms; over those 67 problems
// the choice they make costs 0.8% on average against the best configuration
// (9% at worst).
struct StreamCfg {
  int bm, bn, wg;        // tile, workgroups per CU
  bool paired;           // has the RoPE / SiLU epilogues
  float launch, round, stage, stage1;
  int (*run)(GemmArgs, int, int, hipStream_t);
};
const StreamCfg kStream[] = {
    {64, 64, 1, true, 3.46f, 0.87f, 0.193f, 0.f, launch_stream<64, 64, 4, 2, 4, 1>},
    {64, 80, 1, false, 4.14f, 0.83f, 0.232f, 0.f, launch_stream<64, 80, 4, 2, 4, 1>},
    {64, 96, 2, true, 2.67f, 2.26f, 0.507f, 0.270f, launch_stream<64, 96, 4, 2, 3, 2>},
    {64, 160, 1, true, 1.90f, 3.79f, 0.375f, 0.f, launch_stream<64, 160, 4, 2, 4, 1>},
    {128, 64, 1, true, 1.68f, 3.15f, 0.287f, 0.f, launch_stream<128, 64, 4, 2, 4, 1>},
    {128, 64, 2, true, 1.94f, 2.37f, 0.613f, 0.313f, launch_stream<128, 64, 4, 1, 3, 2>},
    {128, 96, 1, true, 1.86f, 4.29f, 0.357f, 0.f, launch_stream<128, 96, 4, 2, 3, 1>},
    {128, 128, 1, true, 0.95f, 5.89f, 0.388f, 0.f, launch_stream<128, 128, 4, 2, 4, 1>},
    {128, 192, 1, false, 0.00f, 5.94f, 0.520f, 0.f, launch_stream<128, 192, 2, 1, 3, 1>},
    {192, 128, 1, true, 0.60f, 6.27f, 0.531f, 0.f, launch_stream<192, 128, 4, 1, 3, 1>},
    {256, 128, 1, true, 0.42f, 7.68f, 0.635f, 0.f, launch_stream<256, 128, 4, 1, 3, 1>},
};

// microseconds of a problem on configuration c, K split over `splits`
template <class C>
double stream_cost(const C& c, int M, int N, int K, int splits) {
  const long nk = ((K + GK - 1) / GK + splits - 1) / splits;
  const long tiles = (long)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * splits;
  const long full = tiles / (256L * c.wg), rest = tiles % (256L * c.wg);
  const bool single = c.wg == 2 && rest > 0 && rest <= 256;
  return c.launch + c.round * (full + (rest > 0)) +
         nk * ((double)c.stage * (full + (rest > 0 && !single)) + (single ? c.stage1 : 0.f));
}

const StreamCfg& pick_stream(int M, int N, int K, int epi) {
  const bool paired = epi == EPI_ROPE || epi == EPI_SILU;
  const StreamCfg* best = nullptr;
  double best_us = 0;
  for (const StreamCfg& c : kStream) {
    if (paired && !c.paired) continue;
    const double us = stream_cost(c, M, N, K, 1);
    if (!best || us < best_us) {
      best = &c;
      best_us = us;
    }
  }
  return *best;
}

// The gathers' configurations (costs as kStream's).
struct GatherCfg {
  int bm, bn, wg;
  float launch, round, stage, stage1;
  int (*run)(GemmArgs, int, int, hipStream_t);
};
const GatherCfg kGather[] = {
    {64, 64, 1, 3.46f, 0.87f, 0.193f, 0.f, launch_gather<64, 64, 4, 2, 4, 1>},
    {64, 96, 2, 2.67f, 2.26f, 0.507f, 0.270f, launch_gather<64, 96, 4, 2, 3, 2>},
    {64, 160, 1, 1.90f, 3.79f, 0.375f, 0.f, launch_gather<64, 160, 4, 2, 4, 1>},
    {128, 128, 1, 0.95f, 5.89f, 0.388f, 0.f, launch_gather<128, 128, 4, 2, 4, 1>},
    {128, 192, 1, 0.00f, 5.94f, 0.520f, 0.f, launch_gather<128, 192, 2, 1, 3, 1>},
    {192, 128, 1, 0.60f, 6.27f, 0.531f, 0.f, launch_gather<192, 128, 4, 1, 3, 1>},
    {256, 128, 1, 0.42f, 7.68f, 0.635f, 0.f, launch_gather<256, 128, 4, 1, 3, 1>},
};
constexpr int kMaxSplits = 12;
// A split's partial tiles: the reduction launch, and their fp32 write and read
// (connector at 1 to 32 images, measured beyond the tiles' own cost: 6.4 us for
// 6 MB, 8.3 for 12, 16-20 for 32).
double split_cost(int M, int N, int splits) {
  return splits == 1 ? 0.0 : 4.0 + 8e-6 * M * N * splits / 2.3;
}

}  // namespace

namespace svla_gemm {

// Plain, RoPE or SiLU epilogue on bf16 rows that 16-byte pieces can address
// (the other preconditions are run_gemm's).
bool stream_takes(const GemmArgs& p, int epi) {
  if (epi == EPI_EULER || p.norm_w || p.out_f32 || p.rowadd || p.c_rpg > 0 || p.K < 8) return false;
  if (p.N % 8 || p.ldc % 8) return false;
  if (p.c_lo && !svla_aligned16(p.c_lo)) return false;
  if (p.res && (p.ldr % 8 || !svla_aligned16(p.res))) return false;
  return true;
}

int stream_tile(int M, int N, int K, int epi) {
  const StreamCfg& c = pick_stream(M, N, K, epi);
  return c.bm * 1000 + c.bn;
}

bool gather_takes(const GemmArgs& p) {
  return p.M >= 64 && p.K >= GK && p.N % 8 == 0 && p.ldc % 8 == 0 && !p.out_f32 && !p.bias_f32 &&
         !p.res && !p.norm_w;
}

// Unsplit without a workspace; a few images' connector has tens of tiles and
// K = 12288, so with one its K is split over workgroups as far as `ws_floats`
// floats hold the partial tiles.  MI355X, graph replay, before (64x64 line
// tile, register-staged 128x128 or split skinny tiles) / now: connector of 1
// image 22.0 / 13.9 us, 3 images 38.4 / 19.4, 4 images 42.1 / 23.8 (split), 9
// images 103 / 60, 32 images 133 / 89 (unsplit; 32 and 64 split, but these
// never shared the workspace), 96 images 225 / 144; patch embedding of 1 image
// 12.3 / 8.7, 7 images 26.7 / 16.6, 96 images 235 / 171.  The connector's K lies
// past that of the fits: for 96 images they say 106 us.
// Under four K stages a tile is mostly its fixed cost, which the fits (K from
// 320) do not hold apart: 64x64 tiles up to two per CU, past that the choice
// among those of 128 rows and more.  MI355X, graph replay, register-staged
// 128x128 / 64x64 at every size / now: 8-pixel patches of 3 channels (K = 192,
// N = 768), 1 image 12.0 / 10.1 / 9.1 us, 12 images 65.4 / 76.3 / 52.0, 48
// images 263 / 311 / 193; K = 64, N = 200, 48 images of 784 patches 17.1 / 19.1
// / 14.2; a pixel shuffle of 2048x960x128 (480 tiles) 7.1 / 6.0 / 6.0 (128x192
// 7.2), of 16384x960x128 20.7 / 26.1 / 17.0.
GatherPlan gather_plan(int M, int N, int K, long ws_floats, int force) {
  const int nk = (K + GK - 1) / GK;
  const bool brief = nk < 4;
  if (force <= 0 && brief && (long)((M + 63) / 64) * ((N + 63) / 64) <= 512) return {0, 1};
  int lo = 1, hi = force > 0 ? min(force, nk) : min(kMaxSplits, max(nk / 4, 1));
  hi = (int)max(min((long)hi, ws_floats / ((long)M * N)), 1L);
  if (force > 0) lo = hi;
  GatherPlan best{0, 1};
  double best_us = -1;
  for (int i = 0; i < (int)(sizeof(kGather) / sizeof(kGather[0])); ++i) {
    if (force <= 0 && brief && kGather[i].bm < 128) continue;
    for (int z = lo; z <= hi; ++z) {
      const double us = stream_cost(kGather[i], M, N, K, z) + split_cost(M, N, z);
      if (best_us < 0 || us < best_us) {
        best = {i, z};
        best_us = us;
      }
    }
  }
  return best;
}

int gather_tile(const GatherPlan& g) { return kGather[g.cfg].bm * 1000 + kGather[g.cfg].bn; }

int gather_run(const GemmArgs& p, int amode, const GatherPlan& g, hipStream_t s) {
  return kGather[g.cfg].run(p, amode, g.splits, s);
}

int stream_run(const GemmArgs& p, int epi, int act, hipStream_t s) {
  return pick_stream(p.M, p.N, p.K, epi).run(p, epi, act, s);
}

}  // namespace svla_gemm
