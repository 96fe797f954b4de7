// GEMM for 16-bit inputs (bf16 / f16) with f32 accumulation on the gfx950 matrix cores and
// the fused bias / activation / conversion epilogue of the matmul payload
// (emit_mlp_layer, lighthouse/ingress/mlir_gen/gpu_mlp_payload.py:110-156).
//
// Fast kernel (shapes that are multiples of the tile): workgroup tile BM x BN x 64, A and B
// panels double-buffered in LDS, v_mfma_f32_32x32x16 tiles, one barrier per k-step.  The MFMA
// is issued with the B panel as its first operand and the A panel as its second, so the
// accumulator of a lane holds 4 consecutive columns n of one row m and the epilogue stores
// 8 or 16 contiguous bytes per lane.  A row-major B ([K,N], n contiguous) is transposed in
// registers (v_perm_b32) on its way into LDS so both LDS panels are k-contiguous and every
// MFMA operand is a single 16-byte LDS read.
//
// Generic kernel: any shape, stride and transpose combination, 64 x 64 x 32 tiles with
// bounds-checked scalar loads.
#include <algorithm>

#include "gemm16.h"

namespace lh {

constexpr int kBK = 64;
constexpr int kLdsStride = kBK + 8;  // elements; 144-byte rows keep 16-byte reads of 16 rows conflict free

template <int BM, int BN>
constexpr size_t gemm16_lds_bytes() {
  return (size_t)2 * (BM + BN) * kLdsStride * sizeof(uint16_t);
}

template <int DT, int BM, int BN, int WAVES_M, int WAVES_N, bool B_KC>
__global__ void __launch_bounds__(WAVES_M* WAVES_N * 64) gemm16_fast(GemmArgs g) {
  constexpr int NT = WAVES_M * WAVES_N * 64;
  constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int A_CH = BM * (kBK / 8) / NT;  // 16-byte chunks of the A panel per thread
  constexpr int B_CH = BN * (kBK / 8) / NT;  // same for a k-contiguous B panel
  constexpr int B_UN = (kBK / 8) * (BN / 4) / NT;  // 8k x 4n units per thread for a row-major B
  static_assert(A_CH >= 1 && B_CH >= 1 && B_UN >= 1, "tile too small for the thread count");

  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  uint16_t* As = smem;
  uint16_t* Bs = smem + 2 * BM * kLdsStride;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm0 = (wave / WAVES_N) * WTM;
  const int wn0 = (wave % WAVES_N) * WTN;

  // Tile assignment: XCD-contiguous ids, then groups of 4 tile rows.
  const int tiles_m = g.M / BM, tiles_n = g.N / BN;
  int id = xcd_remap(blockIdx.x, gridDim.x);
  constexpr int GROUP_M = 4;
  const int group_size = GROUP_M * tiles_n;
  const int first_m = (id / group_size) * GROUP_M;
  const int gm = min(tiles_m - first_m, GROUP_M);
  const int tile_m = first_m + (id % group_size) % gm;
  const int tile_n = (id % group_size) / gm;
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  const uint16_t* A = reinterpret_cast<const uint16_t*>(g.a);
  const uint16_t* B = reinterpret_cast<const uint16_t*>(g.b);

  u32x4 ra[A_CH];
  u32x4 rbk[B_KC ? B_CH : 1];
  u32x2 rbn[B_KC ? 1 : B_UN][8];

  auto load_global = [&](int k0) {
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      int c = tid + i * NT;
      int row = c >> 3, kc = c & 7;
      ra[i] = *reinterpret_cast<const u32x4*>(A + (int64_t)(m0 + row) * g.lda + k0 + kc * 8);
    }
    if constexpr (B_KC) {
#pragma unroll
      for (int i = 0; i < B_CH; ++i) {
        int c = tid + i * NT;
        int row = c >> 3, kc = c & 7;
        rbk[i] = *reinterpret_cast<const u32x4*>(B + (int64_t)(n0 + row) * g.ldb + k0 + kc * 8);
      }
    } else {
#pragma unroll
      for (int i = 0; i < B_UN; ++i) {
        int u = tid + i * NT;
        int ngrp = u % (BN / 4), kgrp = u / (BN / 4);
        const uint16_t* p = B + (int64_t)(k0 + kgrp * 8) * g.ldb + n0 + ngrp * 4;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) rbn[i][kk] = *reinterpret_cast<const u32x2*>(p + (int64_t)kk * g.ldb);
      }
    }
  };

  auto store_lds = [&](int buf) {
    uint16_t* as = As + buf * BM * kLdsStride;
    uint16_t* bs = Bs + buf * BN * kLdsStride;
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      int c = tid + i * NT;
      int row = c >> 3, kc = c & 7;
      *reinterpret_cast<u32x4*>(as + row * kLdsStride + kc * 8) = ra[i];
    }
    if constexpr (B_KC) {
#pragma unroll
      for (int i = 0; i < B_CH; ++i) {
        int c = tid + i * NT;
        int row = c >> 3, kc = c & 7;
        *reinterpret_cast<u32x4*>(bs + row * kLdsStride + kc * 8) = rbk[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < B_UN; ++i) {
        int u = tid + i * NT;
        int ngrp = u % (BN / 4), kgrp = u / (BN / 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // Column j of the 8 x 4 register block becomes a k-contiguous row of 8 values.
          const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
          u32x4 w;
#pragma unroll
          for (int d = 0; d < 4; ++d)
            w[d] = __builtin_amdgcn_perm(rbn[i][2 * d + 1][j >> 1], rbn[i][2 * d][j >> 1], sel);
          *reinterpret_cast<u32x4*>(bs + (ngrp * 4 + j) * kLdsStride + kgrp * 8) = w;
        }
      }
    }
  };

  f32x16 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  const int nk = g.K / kBK;
  load_global(0);
  store_lds(0);
  __syncthreads();

  const int frag_row = lane & 31;
  const int frag_k = (lane >> 5) * 8;

  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) load_global((kt + 1) * kBK);

    const uint16_t* as = As + buf * BM * kLdsStride + (wm0 + frag_row) * kLdsStride + frag_k;
    const uint16_t* bs = Bs + buf * BN * kLdsStride + (wn0 + frag_row) * kLdsStride + frag_k;
#pragma unroll
    for (int ks = 0; ks < kBK / 16; ++ks) {
      u32x4 fb[TN], fa[TM];
#pragma unroll
      for (int i = 0; i < TN; ++i) fb[i] = *reinterpret_cast<const u32x4*>(bs + i * 32 * kLdsStride + ks * 16);
#pragma unroll
      for (int j = 0; j < TM; ++j) fa[j] = *reinterpret_cast<const u32x4*>(as + j * 32 * kLdsStride + ks * 16);
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = Mfma16<DT>::mma(fb[i], fa[j], acc[i][j]);
    }

    if (kt + 1 < nk) store_lds(buf ^ 1);
    __syncthreads();
  }

  // acc[i][j][4q+e] = C[m0+wm0+32j+lane%32][n0+wn0+32i+8q+4(lane/32)+e]
  const int m_base = m0 + wm0 + (lane & 31);
  const int n_base = n0 + wn0 + 4 * (lane >> 5);
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        epilogue4<DT>(g, m_base + 32 * j, n_base + 32 * i + 8 * q, acc[i][j][4 * q], acc[i][j][4 * q + 1],
                      acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
}


// Any shape / stride / transpose; 64 x 64 x 32 tiles, 256 threads, bounds-checked.
template <int DT>
__global__ void __launch_bounds__(256) gemm16_generic(GemmArgs g) {
  constexpr int BM = 64, BN = 64, BK = 32, STR = BK + 8;
  __shared__ __attribute__((aligned(16))) uint16_t As[BM * STR];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[BN * STR];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm0 = (wave >> 1) * 32, wn0 = (wave & 1) * 32;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const uint16_t* A = reinterpret_cast<const uint16_t*>(g.a);
  const uint16_t* B = reinterpret_cast<const uint16_t*>(g.b);
  const bool ta = (g.flags & LH_GEMM_TRANSPOSE_A) != 0, tb = (g.flags & LH_GEMM_TRANSPOSE_B) != 0;
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  for (int k0 = 0; k0 < g.K; k0 += BK) {
    for (int e = tid; e < BM * BK; e += 256) {
      // Thread order follows the contiguous dimension of the stored operand.
      int r, c;
      if (ta) { r = e % BM; c = e / BM; } else { r = e / BK; c = e % BK; }
      int m = m0 + r, k = k0 + c;
      uint16_t v = 0;
      if (m < g.M && k < g.K) v = ta ? A[(int64_t)k * g.lda + m] : A[(int64_t)m * g.lda + k];
      As[r * STR + c] = v;
    }
    for (int e = tid; e < BN * BK; e += 256) {
      int r, c;
      if (tb) { r = e / BK; c = e % BK; } else { r = e % BN; c = e / BN; }
      int n = n0 + r, k = k0 + c;
      uint16_t v = 0;
      if (n < g.N && k < g.K) v = tb ? B[(int64_t)n * g.ldb + k] : B[(int64_t)k * g.ldb + n];
      Bs[r * STR + c] = v;
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      u32x4 fb = *reinterpret_cast<const u32x4*>(&Bs[(wn0 + (lane & 31)) * STR + ks * 16 + (lane >> 5) * 8]);
      u32x4 fa = *reinterpret_cast<const u32x4*>(&As[(wm0 + (lane & 31)) * STR + ks * 16 + (lane >> 5) * 8]);
      acc = Mfma16<DT>::mma(fb, fa, acc);
    }
    __syncthreads();
  }
  const int m = m0 + wm0 + (lane & 31);
  if (m >= g.M) return;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    int n = n0 + wn0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
    if (n >= g.N) continue;
    epilogue1<DT>(g, m, n, acc[v]);
  }
}

template <int DT, int BM, int BN, int WAVES_M, int WAVES_N, bool B_KC>
static int launch_fast(const GemmArgs& g, hipStream_t s) {
  auto kern = gemm16_fast<DT, BM, BN, WAVES_M, WAVES_N, B_KC>;
  constexpr size_t lds = gemm16_lds_bytes<BM, BN>();
  static bool configured = false;
  if (!configured && !planning()) {
    LH_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds));
    configured = true;
  }
  dim3 grid((g.M / BM) * (g.N / BN));
  LH_LAUNCH(kern, grid, dim3(WAVES_M * WAVES_N * 64), lds, s, g);
  return check_launch("gemm16_fast");
}

// Tile choice for the direct kernels: 0 = 256 x 256, 1 = 256 x 128, 2 = 128 x 256, 3 = 128 x 128, 4 = 128 x 192.
// Time of a launch, in us and apart from what all share: rounds of resident workgroups (edge tiles count in full)
// times a tile's a + b K, where a is what its output costs and b K the main loop.  The 128 x 128 tile has two workgroups
// on a CU.  A last round that does not fill the CUs costs less than a full one: the persistent workgroups are not in step, so the
// extra tiles run while others still finish, and fewer busy CUs hold a higher clock.  Of a round, a fraction r costs
// part + (1 - part) r^2 (the 128 x 128 tile: r).  Least squares over 1870 problems on each of the first four tiles (M 128 ... 8192,
// N 512 ... 50256, K 256 ... 4096), on rings of two stages: what was chosen was within 0.9 % of the best tile on average, 1.24 x at worst (the
// rule before it, which priced a tile by its flops, 2.4 to 5.0 %, 1.67 x).
// Where no CU gets a second workgroup all but the 256 x 256 tile, which fills the LDS as it is, run with deeper rings
// (gemm16_deep), and 128 x 192 for nothing else; `alone`, fitted to 4096 x 2048, 4096 x 1536, 2048 x 2048 and 8192 x 768 over K = 512 ... 4096.
// Both tables together, over 3950 problems of 60 to 1024 tiles of 128 x 128 of which some tile gives no CU two workgroups (M 129 ... 8192, N 64 ... 8192,
// K 64 ... 5000, either B, every kind of output, edges and partial rounds among them) on every tile: within 0.9 % of the best one on average with
// operands in the caches, 1.33 x at worst, 0.5 % and 1.24 x from memory.  Against the table without `alone` and rings of two stages 0.91 and 0.88 of
// the time; 0.6 % of them take 3 % longer or more (3840 x 2048 x 128 into f32: 9.7 -> 10.9 us on 256 x 128).
// bf16, what was chosen without and with it, operands in the caches / in memory: 8192 x 768 x 3072 with a residual 43.6 -> 40.1 /
// 56.8 -> 49.2 us (128 x 192), K = 768 19.7 -> 18.7 / 27.2 -> 24.9, 4096 x 1536 x 2048 29.0 -> 26.5 / 34.0 -> 30.2, 4096 x 2048 x 2048 33.1 -> 32.3 /
// 39.2 -> 35.2 (256 x 128), with f32 results 34.2 -> 33.7 / 46.8 -> 38.5 (128 x 256).
// `whole_k`: K is a multiple of 64; else the 256 x 256 and 128 x 192 tiles are left out.  `time`: the estimate.
struct DirectTile {
  int bm, bn;
  double b, part;
  double a[4];  // 16-bit result; f32 in rows of whole 64-byte pieces; other f32; accumulator input
};
static constexpr DirectTile kDirectTiles[5] = {
    {256, 256, 0.0244, 0.69, {6.5, 9.6, 12.9, 20.5}},
    {256, 128, 0.0141, 0.72, {4.4, 6.4, 7.5, 11.3}},
    {128, 256, 0.0138, 0.77, {4.1, 5.9, 7.4, 10.9}},
    {128, 128, 0.0136, 0.47, {4.1, 6.4, 6.8, 9.6}},
    {128, 192},
};
static constexpr DirectTile kDirectAlone[5] = {
    kDirectTiles[0],
    {256, 128, 0.0131, 0.80, {4.3, 6.2, 7.3, 13.0}},
    {128, 256, 0.0128, 0.80, {5.1, 6.4, 7.9, 10.5}},
    {128, 128, 0.0077, 1.00, {2.9, 4.5, 4.8, 6.7}},
    {128, 192, 0.0103, 0.80, {4.2, 5.7, 9.0, 9.3}},
};
static int64_t direct_tiles(const GemmArgs& g, int v) {
  const DirectTile& t = kDirectTiles[v];
  return (int64_t)((g.M + t.bm - 1) / t.bm) * ((g.N + t.bn - 1) / t.bn);
}
static int direct_variant(const GemmArgs& g, bool whole_k, double* time) {
  const int out = (g.flags & LH_GEMM_ACCUMULATE_C) ? 3 : g.out_dt != LH_F32 ? 0 : rows_of_pieces(g) ? 1 : 2;
  const int cus = num_cus();
  int best = -1;
  double best_us = 0.0;
  for (int v = whole_k ? 0 : 1; v < (whole_k ? 5 : 4); ++v) {
    const int64_t n = direct_tiles(g, v);
    const bool alone = n <= cus;
    if (v == 4 && !alone) continue;
    const DirectTile& t = alone ? kDirectAlone[v] : kDirectTiles[v];
    const int slots = v == 3 && !alone ? 2 * cus : cus;
    const double r = (double)(n % slots) / slots;
    const double rounds = (double)(n / slots) + (r > 0.0 ? t.part + (1.0 - t.part) * (slots == cus ? r * r : r) : 0.0);
    const double us = rounds * (t.a[out] + t.b * g.K);
    if (best < 0 || us < best_us) {
      best = v;
      best_us = us;
    }
  }
  *time = best_us;
  return best;
}

// Columns of a row of the split-K blocks: whole 16-byte chunks.
__host__ __device__ static inline int splitk_row(int N) { return (N + 3) / 4 * 4; }

// Sum of the split-K blocks (f32, [splits][M][splitk_row(N)]) and the problem's own epilogue, 4 columns per thread; any
// alignment of output, bias and accumulator input.
template <int DT>
__global__ void __launch_bounds__(256) gemm16_splitk_reduce(GemmArgs g, const float* partial, int splits) {
  const int row = splitk_row(g.N);
  const int64_t idx = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (idx >= (int64_t)g.M * row) return;
  const int m = (int)(idx / row), n = (int)(idx % row);
  epilogue4_any<DT>(g, m, n, splitk_sum4(partial + idx, (int64_t)g.M * row, splits, blockDim.x == 64));
}

// Cuts along K for the library's own choice: decode shapes, so few 128 x 128 tiles that most CUs would idle, and
// a K long enough to cut.  1: whole.
static int splitk_count(int M, int N, int K) {
  const int cus = num_cus();
  const int64_t tiles = (int64_t)((M + 127) / 128) * ((N + 127) / 128);
  int splits = 1;
  if (tiles * 2 > cus || K < 2048) return 1;
  // Doubling the cut is taken while the k steps it saves each workgroup outweigh the f32 blocks it
  // adds for the second kernel to read: 0.225 us per 32 k saved (half of that once the workgroups
  // outnumber the CUs and share them), 0.62 us per MB of blocks written and read back, 2.5 us for
  // the second kernel itself.  Measured optima this reproduces (M x N x K: cut): 1024 x 1024 x 4096: 4,
  // 128 x 4096 x 4096: 4, 128 x 8192 x 8192: 4, 16 x 8192 x 8192: 8, 32 x 4096 x 4096: 8,
  // 2048 x 768 x 3072: 2, 512 x 4096 x 4096: 2, 512 x 768 x 3072: 4, 512 x 4096 x 2048 and
  // 256 x 8192 x 2048: whole.
  const double block_mb = (double)M * N * sizeof(float) * 1e-6;
  while (splits < 8) {
    const int to = splits * 2;
    if (tiles * to > 2 * cus || K % (to * kBK) != 0 || K / to < 512) break;
    const double saved = (double)(K / splits - K / to) / 32 * 0.225 * (tiles * to > cus ? 0.5 : 1.0);
    const double added = (splits == 1 ? to * block_mb * 0.62 + 2.5 : (to - splits) * block_mb * 0.62);
    if (saved <= added) break;
    splits = to;
  }
  return splits;
}

// Time of an untransposed, aligned problem on the direct kernels, in us, where few tiles make it latency-bound
// (what the small-tile kernels are weighed against; median 0.97 of the measured time on the problems of
// gemm_small.hip's fit, nine in ten between 0.86 and 1.14).  `sp`: the cuts along K that it will run with.
static double direct_us(const GemmArgs& g, int sp) {
  const double x = (double)sp * ((g.M + 127) / 128) * ((g.N + 127) / 128) / num_cus();
  const double per_cu = x <= 1.0 ? 1.0 : 1.0 + 0.55 * (x - 1.0);
  return 3.6 + 0.0072 * g.K / sp * per_cu + (x > 1.0 ? 0.6 * (x - 1.0) : 0.0) +
         (sp > 1 ? 3.2 + 1.2e-6 * sp * g.M * g.N : 0.0);
}

// What K has to be a multiple of for the operands to stay as they are: 8, or the 64 of a whole step where copies that make
// it one pay:
//  * a long K and tiles for less than half the CUs, which stream the operands at a fraction of the rate at which all of them
//    copy them, and where K may be cut (5 x 2032 x 5480 with a transposed A: 31 us on copies, 56 as it is);
//  * the 256 x 256 tile, which has no registers for the end of K; with more than two tiles per CU rows that do not start on
//    128-byte lines cost a tile 1.4 times its time besides (2555 x 5480 x 3000: 103 us on copies and the 256 x 256 tile, 127 on
//    smaller tiles as it is; 1000 x 4096 x 1000, one tile per CU: 23 and 14).
static int direct_k_multiple(const GemmArgs& g) {
  if (g.K % kBK == 0 || (g.flags & (LH_GEMM_TILE_MASK | LH_GEMM_SPLITK_MASK))) return kBK;
  const int64_t tiles = (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128);
  const int cus = num_cus();
  if (tiles * 2 <= cus && g.K >= 2048) return kBK;
  const bool b_in_place = (g.flags & LH_GEMM_TRANSPOSE_B) && g.ldb % 8 == 0 && aligned16(g.b) && g.K % 8 == 0;
  // The problem as the direct kernels would get it: an operand that is copied in any case has rows of its own.
  const OperandCopies copied = operand_copies<2>(g, 8, 8, b_in_place);
  GemmArgs p = g;
  p.K = (g.K + 7) / 8 * 8;
  if (copied.a) p.lda = p.K;
  if (copied.b) {
    p.ldb = (g.N + 7) / 8 * 8;
    p.flags &= ~(uint32_t)LH_GEMM_TRANSPOSE_B;
  }
  if (!direct_offsets_fit(p)) return kBK;
  const double copies = operand_copies_us<2>(g, kBK, 8, false, 0.65) - operand_copies_us<2>(g, 8, 8, b_in_place, 0.65);
  double as_is, whole;
  const bool odd_rows = tiles > 2 * cus && p.lda % 64 != 0;
  p.K = (g.K + kBK - 1) / kBK * kBK;
  direct_variant(p, false, &as_is);
  direct_variant(p, true, &whole);
  if (odd_rows) as_is *= 1.4;
  return whole + copies <= as_is ? kBK : 8;
}

// A B that the loads into LDS cannot take (rows that are no whole aligned 16-byte chunks) is read as it is where one round of
// workgroups of the 128 x 128 tile covers the result: the copy in a launch of its own is a good part of such a product's time.
// Larger ones spread it over more rows of A and have the larger tiles besides; with two workgroups on a CU and a long K the tile
// on a copy catches up: 84 such products, as it is against on a copy, 0.69 of the time for K <= 512, 0.84 up to 1536, 0.87 up to 2560 and
// 1.10 up to 3072 (3146 x 1547 x 2784 49.0 us on a copy, 55.4 as it is; one workgroup, 2000 x 2001 x 4096: 49.6 and 41.4).
static bool odd_rows_stay(const GemmArgs& g) {
  if (planning() || g.b_padded || (g.flags & (LH_GEMM_TILE_MASK | LH_GEMM_SPLITK_MASK | LH_GEMM_TRANSPOSE_A | LH_GEMM_TRANSPOSE_B)))
    return false;
  if (g.N % 8 == 0 && g.ldb % 8 == 0 && aligned16(g.b)) return false;
  const int64_t tiles = (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128);
  return g.N >= 8 && g.K % 8 == 0 && g.lda % 8 == 0 && aligned16(g.a) && (int64_t)g.M * g.N * g.K >= (1 << 22) &&
         (tiles <= num_cus() || (tiles <= 2 * num_cus() && g.K <= 2560)) && direct_offsets_fit(g) && splitk_count(g.M, g.N, (g.K + kBK - 1) / kBK * kBK) == 1;
}

// Decode shapes: so few 128 x 128 tiles that most CUs would idle, and a K long enough to cut.
// Returns 1 when the problem does not qualify.
// `request`: LH_GEMM_SPLITK_* bits of the call; an explicit 2 / 4 / 8 bypasses the criteria.
template <int DT>
static int gemm16_splitk(const GemmArgs& g, uint32_t request, hipStream_t s) {
  int splits = 1;
  if (request == LH_GEMM_SPLITK_NONE) return 1;
  if (request != LH_GEMM_SPLITK_AUTO) {
    splits = request == LH_GEMM_SPLITK_2 ? 2 : request == LH_GEMM_SPLITK_4 ? 4 : 8;
    LH_REQUIRE(g.K % (splits * kBK) == 0 && g.K / splits >= 2 * kBK,
               "gemm: a cut of K = %d into %d needs K / %d to be a multiple of %d and at least %d", g.K, splits, splits,
               kBK, 2 * kBK);
  } else {
    splits = splitk_count(g.M, g.N, g.K);
    if (splits == 1) return 1;
  }
  void* taken = nullptr;
  if (int rc = scratch_take(g.ws, s, kScratchSplitK, (size_t)splits * g.M * splitk_row(g.N) * sizeof(float), "gemm (split K)", &taken))
    return rc;
  float* partial = static_cast<float*>(taken);
  GemmArgs p = g;
  p.K = g.K / splits;
  p.splits = splits;
  p.out = partial;
  p.c = partial;
  p.ldc = splitk_row(g.N);
  p.out_dt = LH_F32;
  p.bias = nullptr;
  p.flags = g.flags & LH_GEMM_TRANSPOSE_B;
  if (int rc = launch_direct_splitk<DT>(p, s)) return rc;
  const int64_t groups = (int64_t)g.M * splitk_row(g.N) / 4;
  const int rb = reduce_block(groups);
  LH_LAUNCH(gemm16_splitk_reduce<DT>, dim3((unsigned)((groups + rb - 1) / rb)), dim3(rb), 0, s, g, partial, splits);
  return check_launch("gemm16_splitk_reduce");
}

template <int DT>
static int gemm16_dispatch(const GemmArgs& g_in, hipStream_t s) {
  GemmArgs g = g_in;
  // (a size query counts the copies of whole steps, the upper bound it always was)
  const int kmul = planning() ? kBK : g.k_multiple ? g.k_multiple : direct_k_multiple(g);
  // A transposed B ([N, K], k contiguous) with aligned rows goes through the direct kernels as it is
  // (its panel is loaded and read like A's); a transposed A is copied into [M, K] first.
  const bool b_in_place = (g.flags & LH_GEMM_TRANSPOSE_B) && g.ldb % 8 == 0 && aligned16(g.b) && g.K % kmul == 0;
  // An output side of whole 16-byte chunks: what requests ask for.  Without it, or with a K that is no multiple of 64, a small
  // problem needs no memory of a caller's workspace, here and in a size query alike (the copies of such a K are made where
  // there is room for them).  The library's own pool it may use where the untransposed operands then fit the direct kernels, or
  // K is long: a transposed A of fewer rows than the small tiles take, 1 x 768 x 3200 bf16, runs 34 us on a copy and 260 on the
  // bounds-checked kernel, which gains from one as well (B unaligned, 1 x 896 x 2560: 221 -> 171; at K = 128 it loses 2 of 14).
  // So it is with a K that ends inside a step, which may be so short that the copy is most of the time: 4 x 512 x 24 7.3 us as
  // it is and 10.6 on a copy, K = 72 10.3 and 10.6, K = 136 15.3 and 10.9; 1 x 16 x 104 12.4 and 10.9.
  const bool vec_c = g.N % 8 == 0 && g.ldc % 8 == 0 && aligned16(g.out) && (!(g.flags & LH_GEMM_HAS_BIAS) || aligned16(g.bias));
  const bool copy_fits = rows_fit_untransposed<2>(g), copy_pays = g.K >= 512 || copy_fits;
  const bool may_copy = (int64_t)g.M * g.N * g.K >= (1 << 22) ||
                        (g.K % kBK == 0 ? vec_c || (!g.ws && copy_pays)
                                        : copy_pays && g.K >= 80 && (!g.ws || (vec_c && untransposed_room<2>(g, b_in_place))));
  if ((g.flags & LH_GEMM_TILE_MASK) == LH_GEMM_TILE_AUTO && (g.flags & LH_GEMM_SPLITK_MASK) <= LH_GEMM_SPLITK_NONE &&
      !planning()) {
    // Few tiles: the small-tile kernels, if they are the faster ones.  Against them stand the direct kernels, plus
    // the transposed or padded copies of operands that the direct kernels cannot take as they are.
    const bool tb = g.flags & LH_GEMM_TRANSPOSE_B;
    const bool fits = g.K % kmul == 0 && (tb || g.N % 8 == 0 || g.b_padded) && g.lda % 8 == 0 && g.ldb % 8 == 0 &&
                      aligned16(g.a) && aligned16(g.b);
    // (a copy has whole k-steps where kmul says so)
    const int cuts = may_copy && !(g.flags & LH_GEMM_SPLITK_MASK) ? splitk_count(g.M, g.N, (g.K + kmul - 1) / kmul * kmul) : 1;
    // B in odd rows takes 1.25 of the direct kernels' time (median 1.28 on 1000 products) and no copy.  855 of them, M 1 ... 8192,
    // N 65 ... 16384, K 64 ... 8192: chosen so 0.3 % slower than the better of the two on average, one of them slower than with the copy
    // counted alone, by 1.23 (priced at 1.0 37 were, 8 x 14521 x 1552 10.5 -> 21.7 us).  An f32 result counts the copy: the small tiles
    // add up eight shares of K, and one chain of sums instead would be 1.2 (K = 128) to 3 times (K = 7000) as far from 64 bits.
    const bool odd_rows = odd_rows_stay(g);
    double other = direct_us(g, cuts) + operand_copies_us<2>(g, kmul, 8, b_in_place, 0.65);
    if (odd_rows && g.out_dt != LH_F32) other = std::min(other, 1.25 * direct_us(g, 1));
    int tile;
    const double us = gemm_small_choose(g, DT, &tile);
    if (tile >= 0 && (us * kSmallMargin < other || (!fits && (int64_t)g.M * g.N * g.K < (1 << 22)))) return gemm_small(g, DT, tile, s);
    if (odd_rows) return launch_odd_rows<DT>(g, s);
  }
  if ((g.flags & LH_GEMM_TILE_MASK) == LH_GEMM_TILE_AUTO && may_copy) {
    if (b_in_place) g.flags &= ~(uint32_t)LH_GEMM_TRANSPOSE_B;
    const int rc = untranspose_operands<2>(g, kmul, 8, s);
    if (b_in_place) g.flags |= LH_GEMM_TRANSPOSE_B;
    if (rc < 0) return rc;
  }
  const bool ta = g.flags & LH_GEMM_TRANSPOSE_A;
  const bool tb = (g.flags & LH_GEMM_TRANSPOSE_B) && !b_in_place;  // a transposed B the direct kernels cannot take
  const bool rows_ok = !ta && g.K % kmul == 0 && g.lda % 8 == 0 && g.ldb % 8 == 0 && aligned16(g.a) && aligned16(g.b);
  const bool operands_ok = rows_ok && g.K % kBK == 0;
  const bool direct = rows_ok && (b_in_place || (!tb && (g.N % 8 == 0 || g.b_padded)));
  const uint32_t tile = g.flags & LH_GEMM_TILE_MASK;
  const uint32_t splitk = g.flags & LH_GEMM_SPLITK_MASK;
  const bool cut_requested = splitk > LH_GEMM_SPLITK_NONE;
  if (tile == LH_GEMM_TILE_AUTO && !cut_requested && !direct && (int64_t)g.M * g.N * g.K >= (1 << 22)) {
    // not a shape for the direct kernels as it stands: run it on padded copies of the operands
    const int rc = gemm_padded<2, false>(g, kmul, 8, s, [&](const GemmArgs& p) { return gemm16_dispatch<DT>(p, s); });
    if (rc <= 0) return rc;
  }
  if (tile != LH_GEMM_TILE_AUTO) {
    static const int bm[4] = {256, 256, 128, 128}, bn[4] = {256, 128, 256, 128};
    const int v = (int)(tile >> 8) - 1;
    LH_REQUIRE(direct && g.K % kBK == 0 && vec_c && g.M % bm[v] == 0 && g.N % bn[v] == 0 && direct_offsets_fit(g),
               "gemm: the requested %d x %d tile needs an untransposed A, M %% %d == 0, N %% %d == 0, "
               "K %% 64 == 0 and 16-byte aligned rows, also of a transposed B (M=%d N=%d K=%d)",
               bm[v], bn[v], bm[v], bn[v], g.M, g.N, g.K);
  }
  if (cut_requested)
    LH_REQUIRE(direct && g.K % kBK == 0 && vec_c && direct_offsets_fit(g),
               "gemm: a split-K request needs an untransposed A, K %% 64 == 0, N %% 8 == 0 and 16-byte aligned rows, "
               "also of a transposed B (M=%d N=%d K=%d)", g.M, g.N, g.K);
  if (direct && direct_offsets_fit(g)) {
    if (tile == LH_GEMM_TILE_AUTO && may_copy) {
      const int rc = gemm16_splitk<DT>(g, splitk, s);
      if (rc <= 0) return rc;
    }
    double us;
    const int v = tile != LH_GEMM_TILE_AUTO ? (int)(tile >> 8) - 1 : direct_variant(g, g.K % kBK == 0, &us);
    if (v == 0) return launch_direct<DT, 4, 2>(g, s);
    const bool deep = direct_tiles(g, v) <= num_cus();
    if (v == 1) return deep ? launch_deep<DT, 4, 1>(g, s) : launch_direct<DT, 4, 1>(g, s);
    if (v == 2) return deep ? launch_deep<DT, 2, 2>(g, s) : launch_direct<DT, 2, 2>(g, s);
    if (v == 3) return deep ? launch_deep<DT, 2, 1>(g, s) : launch_direct<DT, 2, 1>(g, s);
    if (v == 4) return launch_deep<DT, 2, 3>(g, s);
  }
  if (operands_ok && g.ldc % 4 == 0 && aligned16(g.out) && (!(g.flags & LH_GEMM_HAS_BIAS) || aligned16(g.bias))) {
    // (B as it is stored, also where the direct kernels would have read a transposed one in place but a row stride
    // is too large for their 32-bit offsets)
    const bool b_kc = g.flags & LH_GEMM_TRANSPOSE_B;
    const int cus = num_cus();
    const bool big = g.M % 256 == 0 && g.N % 256 == 0 && (int64_t)(g.M / 256) * (g.N / 256) >= cus;
    if (big) {
      return b_kc ? launch_fast<DT, 256, 256, 2, 4, true>(g, s) : launch_fast<DT, 256, 256, 2, 4, false>(g, s);
    }
    if (g.M % 128 == 0 && g.N % 128 == 0) {
      return b_kc ? launch_fast<DT, 128, 128, 2, 2, true>(g, s) : launch_fast<DT, 128, 128, 2, 2, false>(g, s);
    }
  }
  dim3 grid((g.N + 63) / 64, (g.M + 63) / 64);
  LH_LAUNCH(gemm16_generic<DT>, grid, dim3(256), 0, s, g);
  return check_launch("gemm16_generic");
}

double gemm16_us(const GemmArgs& g, int ab_dtype) {
  int tile;
  const double direct = direct_us(g, 1), small = gemm_small_choose(g, ab_dtype, &tile);
  return tile >= 0 && small * kSmallMargin < direct ? small * kSmallMargin : direct;
}

int gemm16(const GemmArgs& g, int ab_dtype, hipStream_t s) {
  if (ab_dtype == LH_BF16) return gemm16_dispatch<LH_BF16>(g, s);
  return gemm16_dispatch<LH_F16>(g, s);
}

}  // namespace lh
