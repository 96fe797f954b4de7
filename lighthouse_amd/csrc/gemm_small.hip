// GEMM for problems with few output tiles, any operand layout and alignment: 16-bit, f32 and fp8 inputs
// with the fused epilogue of the matmul payload (emit_mlp_layer,
// lighthouse/ingress/mlir_gen/gpu_mlp_payload.py:110-156).
//
// What bounds a GEMM of a few dozen to a few hundred rows is not arithmetic but the chain of dependent
// steps one workgroup walks: on the 128 x 128 tile kernel, M = 100, N = 2304, K = 768 is 18 workgroups that
// each take 24 k-steps one after the other behind barriers (14 us).  Here a workgroup owns a small tile
// (16 MT x 16 NT) and its NW waves share out the K dimension: a wave multiplies a contiguous share of the k-steps
// on its own, without a barrier, with P steps of both operands requested ahead in registers; the NW
// partial tiles are added through LDS once, in wave order.  A step is 64 bytes of k per row for every
// element type (32 values of 16 bit, 64 of fp8, 16 of f32): a lane's operand is one 16-byte chunk.
//
//  * A k-contiguous operand (A stored [M, K], B stored [N, K]) is loaded straight into the MFMA's operand
//    layout and never touches LDS.
//  * An operand contiguous along M or N (A stored [K, M], B stored [K, N]) goes through a few KiB of LDS
//    that belong to the wave alone and is read back with the transposing LDS reads.
//
// Global accesses are 16 bytes wide at element alignment (gfx9 global memory takes any alignment), so odd
// leading dimensions and unaligned views need no padded copies; everything past K counts as zero.  Rows that split
// dwords are slow all the same (kSmallSplit below).
#include "gemm_small.h"

namespace lh {

template <int DT, int MT, int NT, int NW, bool AKC, bool BKC>
struct SmallCfg {
  typedef SmallPanel<DT, MT, AKC> PA;
  typedef SmallPanel<DT, NT, BKC> PB;
  static constexpr int kWaveLds = PA::kLdsBytes + PB::kLdsBytes;
  static constexpr int kSumBytes = NW * MT * NT * 1024;
  static constexpr int kLdsBytes = kSumBytes > NW * kWaveLds ? kSumBytes : NW * kWaveLds;
  // Steps requested ahead: what fits next to the accumulators in the registers of NW waves.
  static constexpr int P = MT + NT <= 3 ? 3 : 2;
  static constexpr bool kLoadEpilogue = MT * NT < 16;  // (the largest tile has no registers to hold it)
  static constexpr bool kTight = MT * NT == 16 && !AKC && !BKC && PA::ES == 2;  // (all 256 registers that 8 waves have)
};

// The wave's share of the k-steps.
template <typename Cfg, int DT, int MT, int NT, int NW, bool WHOLE>
__device__ __forceinline__ void small_multiply(const typename Cfg::PA& pa, const typename Cfg::PB& pb, f32x4 (&acc)[MT][NT],
                                               int K, int wave, int lane, uint8_t* lds_a, uint8_t* lds_b) {
  constexpr int P = Cfg::P, KSTEP = Cfg::PA::KSTEP;
  // Its list of steps: the one K ends in first (if it is not whole: the last wave's, whose share of the
  // others is the smallest), then its contiguous share of the whole steps.
  const int full = K / KSTEP;
  const int begin = (full * wave + NW - 1) / NW;
  const bool tail = K % KSTEP != 0 && wave == NW - 1;
  const int mine = (tail ? 1 : 0) + (full * (wave + 1) + NW - 1) / NW - begin;
  const int first = tail ? begin - 1 : begin;  // step i of the list is step first + i of K (the tail apart)
  if (mine == 0) return;
  u32x4 ra[P][MT], rb[P][NT];
  auto consume = [&](u32x4 (&a)[MT], u32x4 (&b)[NT]) {
    u32x4 fa[MT], fb[NT];
    pb.template stage<WHOLE>(b, lds_b, lane);
    if constexpr (Cfg::kTight) pa.template stage<WHOLE>(a, lds_a, lane);
    pb.fragments(b, lds_b, lane, fb);
    if constexpr (!Cfg::kTight) pa.template stage<WHOLE>(a, lds_a, lane);
    pa.fragments(a, lds_a, lane, fa);
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int i = 0; i < NT; ++i) acc[j][i] = small_mma<DT>(fb[i], fa[j], acc[j][i]);
    // (a step on its own: with the next one's reads and shifts pulled into it this kernel spills registers)
    if constexpr (Cfg::kTight && !WHOLE) __builtin_amdgcn_sched_barrier(0);
  };
  if (tail) {
    pa.load_tail(full * KSTEP, K, lane, ra[0]);
    pb.load_tail(full * KSTEP, K, lane, rb[0]);
  } else {
    pa.load(first * KSTEP, ra[0]);
    pb.load(first * KSTEP, rb[0]);
  }
#pragma unroll
  for (int p = 1; p < P; ++p)
    if (p < mine) {
      pa.load((first + p) * KSTEP, ra[p]);
      pb.load((first + p) * KSTEP, rb[p]);
    }
  if (tail) {
    pa.finish_tail(full * KSTEP, K, lane, ra[0]);
    pb.finish_tail(full * KSTEP, K, lane, rb[0]);
  }
  // Steps i .. i + n - 1 of the list, the first P of them requested already: in straight-line code the
  // number of loads in flight is known and a step waits for its own loads only.
  int i = 0;
  auto run = [&](auto count) {
    constexpr int n = decltype(count)::value;
#pragma unroll
    for (int p = 0; p < n; ++p) {
      consume(ra[p % P], rb[p % P]);
      if (p + P < n) {
        pa.load((first + i + P + p) * KSTEP, ra[p % P]);
        pb.load((first + i + P + p) * KSTEP, rb[p % P]);
      }
    }
  };
#pragma unroll 1
  for (; i + 2 * P <= mine; i += P) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      consume(ra[p], rb[p]);
      pa.load((first + i + P + p) * KSTEP, ra[p]);
      pb.load((first + i + P + p) * KSTEP, rb[p]);
    }
  }
  const int left = mine - i;  // 1 .. 2 P - 1
  if (left == 1) run(std::integral_constant<int, 1>{});
  else if (left == 2) run(std::integral_constant<int, 2>{});
  else if (left == 3) run(std::integral_constant<int, 3>{});
  else if (P == 3 && left == 4) run(std::integral_constant<int, P == 3 ? 4 : 1>{});
  else if (P == 3) run(std::integral_constant<int, P == 3 ? 5 : 1>{});
}

// `next`: nothing, or the Touch of the launches after this one.
template <int DT, int MT, int NT, int NW, bool AKC, bool BKC, typename... Next>
__device__ __forceinline__ void small_run(const GemmArgs& g, const Next&... next) {
  typedef SmallCfg<DT, MT, NT, NW, AKC, BKC> Cfg;
  constexpr int EDT = DT == LH_F8E4M3 ? LH_BF16 : DT;  // the type a 16-bit output, bias or accumulator input has
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_small[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The workgroups of one XCD (ids congruent modulo 8) take a contiguous range of the tiles counted down
  // the columns: a B panel is read by one XCD's L2 (two at the ends of a range), neighbouring panels
  // share its cache lines.
  const int tiles_m = (g.M + 16 * MT - 1) / (16 * MT), tiles_n = (g.N + 16 * NT - 1) / (16 * NT);
  const int per_xcd = (tiles_m * tiles_n + 7) / 8;
  if constexpr (sizeof...(Next) > 0) {
    // (their number as an argument, asked for first, cost 0.2 us: the other arguments were loaded behind it)
    if ((int)blockIdx.x >= 8 * per_xcd) return touch_lines(next..., blockIdx.x - 8 * per_xcd);
  }
  const int tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (tile >= tiles_m * tiles_n) return;
  const int m0 = (tile % tiles_m) * 16 * MT, n0 = (tile / tiles_m) * 16 * NT;

  SmallEpilogue<EDT, MT, NT, NW> epilogue;
  const bool loaded = Cfg::kLoadEpilogue && g.N >= 4;
  if (loaded) epilogue.load(g, m0, n0, wave, lane);
  typename Cfg::PA pa;
  typename Cfg::PB pb;
  pa.place(g.a, m0, g.M, g.lda, lane);
  pb.place(g.b, n0, g.N, g.ldb, lane);
  uint8_t* const lds_a = smem_small + wave * Cfg::kWaveLds;
  uint8_t* const lds_b = lds_a + Cfg::PA::kLdsBytes;

  f32x4 acc[MT][NT];
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[j][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // (the panels that end inside the tile take a copy of the loop of their own: no branch inside a step)
  if ((AKC || pa.whole) && (BKC || pb.whole)) small_multiply<Cfg, DT, MT, NT, NW, true>(pa, pb, acc, g.K, wave, lane, lds_a, lds_b);
  else small_multiply<Cfg, DT, MT, NT, NW, false>(pa, pb, acc, g.K, wave, lane, lds_a, lds_b);

  if constexpr (Cfg::kWaveLds > 0) __syncthreads();  // (the areas overlap)
  epilogue.sum_and_store(loaded, g, acc, smem_small, m0, n0, wave, lane);
}

template <int DT, int MT, int NT, int NW, bool AKC, bool BKC>
__global__ void __launch_bounds__(NW * 64) gemm_small_kernel(GemmArgs g) {
  small_run<DT, MT, NT, NW, AKC, BKC>(g);
}
// ... of which the workgroups behind those of the work touch what later launches read.  (A kernel of its own: as an argument of the one above
// what to touch cost every product on small tiles 0.03 to 0.1 us, 1 % of 3.6 us, f32 and fp8 ones that never touch anything too.)
template <int DT, int MT, int NT, int NW>
__global__ void __launch_bounds__(NW * 64) gemm_small_touching(GemmArgs g, Touch next) {
  small_run<DT, MT, NT, NW, true, false>(g, next);
}

template <int DT, int MT, int NT, int NW, bool AKC, bool BKC>
static int launch_small_layout(const GemmArgs& g, hipStream_t s) {
  typedef SmallCfg<DT, MT, NT, NW, AKC, BKC> Cfg;
  const int tiles = ((g.M + 16 * MT - 1) / (16 * MT)) * ((g.N + 16 * NT - 1) / (16 * NT));
  const unsigned blocks = 8 * (((unsigned)tiles + 7) / 8);
  const auto launch = [&](auto kern, unsigned grid, auto... more) -> int {
    static bool configured = false;
    if (Cfg::kLdsBytes > 64 * 1024 && !configured && !planning()) {
      LH_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       Cfg::kLdsBytes));
      configured = true;
    }
    LH_LAUNCH(kern, dim3(grid), dim3(NW * 64), Cfg::kLdsBytes, s, g, more...);
    return check_launch("gemm_small");
  };
  // (what touches is the nanoGPT block, whose operands are untransposed and not fp8)
  if constexpr (NW == 8 && AKC && !BKC && DT != LH_F8E4M3) {
    if (const unsigned touching = g.ws ? touch_blocks(g.ws->next, blocks) : 0)
      return launch(gemm_small_touching<DT, MT, NT, NW>, blocks + touching, g.ws->next);
  }
  return launch(gemm_small_kernel<DT, MT, NT, NW, AKC, BKC>, blocks);
}

template <int DT, int MT, int NT, int NW>
static int launch_small(const GemmArgs& g, hipStream_t s) {
  if constexpr (DT == LH_F8E4M3) {  // (fp8 products take no transposed operands)
    return launch_small_layout<DT, MT, NT, NW, true, false>(g, s);
  } else {
    const bool ta = g.flags & LH_GEMM_TRANSPOSE_A, tb = g.flags & LH_GEMM_TRANSPOSE_B;
    if (ta) return tb ? launch_small_layout<DT, MT, NT, NW, false, true>(g, s) : launch_small_layout<DT, MT, NT, NW, false, false>(g, s);
    return tb ? launch_small_layout<DT, MT, NT, NW, true, true>(g, s) : launch_small_layout<DT, MT, NT, NW, true, false>(g, s);
  }
}

// ---- choice of tile ---------------------------------------------------------------------------
// Time of a launch, in us: kSmallFixed + r (b + c steps), r = workgroups per compute unit (at least 1), steps =
// 64-byte steps of K.  From 8 steps on the last round of workgroups counts for more than its share, from 24 on 0.7 of
// what it lacks of a whole one: 672 x 512 x 3072 bf16, 1.3 workgroups per CU, takes 20 us where 1.3 alone would say 12.
// What a step costs is the operand bytes the CU pulls from its L2 (about 20 bytes per
// clock whatever the depth of the prefetch), so a larger tile costs less per result and more per workgroup:
// the cheapest tile is about the largest that still gives every CU one.  b and c are least squares over 400
// problems per type (M 1 .. 3000, N and K 16 .. 8192, both log-uniform); choosing by them is within 2.5 % of the
// best tile, or of the other kernels where those are faster, on average.  Not for more than 4 workgroups per CU,
// where tiles whose waves share their operands win.
struct SmallTile {
  int mt, nt;
  float b[3], c[3];  // 16-bit, f32, fp8
};
constexpr SmallTile kSmallTiles[] = {
    {1, 1, {1.10f, 1.33f, 1.22f}, {0.0468f, 0.0392f, 0.0665f}},  // 16 waves
    {1, 2, {0.74f, 0.93f, 0.80f}, {0.0586f, 0.0606f, 0.0700f}},  // 8 waves
    {1, 4, {1.02f, 1.23f, 1.03f}, {0.0791f, 0.1047f, 0.0749f}},  // 8 waves
    {2, 2, {0.93f, 1.16f, 1.00f}, {0.0720f, 0.0938f, 0.0829f}},  // 8 waves
    {2, 4, {1.42f, 1.47f, 1.36f}, {0.1024f, 0.1819f, 0.0995f}},  // 4 waves
    {4, 4, {2.40f, 2.90f, 2.40f}, {0.1200f, 0.3020f, 0.1200f}},  // 8 waves, whose sums fill a CU's LDS: whole rounds
};
constexpr float kSmallFixed = 2.0f;
// What a step costs more per 16 rows of a k-contiguous operand whose rows do not start at multiples of 4 bytes, in us: its
// chunks go through the L1 at a fraction of the rate (multiples of 4 bytes cost nothing measurable, and an operand that is
// not k-contiguous little).  178 x 1576 x 7168 bf16 with both operands k-contiguous, one element off: 136 us, 46 on copies
// for the tile kernels, where the estimate said 22.  Fitted on 1000 such problems on every tile.
constexpr float kSmallSplit[3] = {0.045f, 0.0f, 0.058f};

double gemm_small_choose(const GemmArgs& g, int dtype, int* tile) {
  const int es = (int)dtype_size(dtype), epc = 16 / es, type = dtype == LH_F32 ? 1 : es == 1 ? 2 : 0;
  const bool ta = g.flags & LH_GEMM_TRANSPOSE_A, tb = g.flags & LH_GEMM_TRANSPOSE_B;
  *tile = -1;
  // (every chunk load reads one whole chunk of a row; 32-bit step and tile counts)
  if ((ta ? g.M : g.K) < epc || (tb ? g.K : g.N) < epc || g.K >= 1 << 24 || (int64_t)g.M * g.N >= 1ll << 36) return 0.0;
  const int steps = (g.K + 64 / es - 1) / (64 / es);
  auto split_cost = [&](const void* p, int64_t ld, bool k_contiguous) {
    return k_contiguous && ((reinterpret_cast<uintptr_t>(p) | (uintptr_t)(ld * es)) & 3) ? kSmallSplit[type] : 0.0f;
  };
  const float split_a = split_cost(g.a, g.lda, !ta), split_b = split_cost(g.b, g.ldb, tb);
  const double stream = 1e-6 * es * ((double)g.M * g.K + (double)g.K * g.N) / 3.6;  // (each operand from memory once)
  // (this runs in front of every launch: shifts for divisions, no library calls; 0.1 us of host time were measurable)
  const int cus = num_cus(), m16 = (g.M + 15) >> 4, n16 = (g.N + 15) >> 4;
  const double rows_a = g.M / 16.0, rows_b = g.N / 16.0;
  const double rest = steps <= 8 ? 0.0 : steps >= 24 ? 0.7 : 0.7 / 16.0 * (steps - 8);
  double best = 0.0;
  for (int i = 0; i < (int)(sizeof(kSmallTiles) / sizeof(kSmallTiles[0])); ++i) {
    const SmallTile& t = kSmallTiles[i];
    const int64_t tiles = (int64_t)((m16 + t.mt - 1) >> __builtin_ctz(t.mt)) * ((n16 + t.nt - 1) >> __builtin_ctz(t.nt));
    if (tiles > 4 * (int64_t)cus) continue;
    double r = 1.0;
    if (tiles > cus) {
      const double rounds = tiles <= 2 * cus ? 2.0 : tiles <= 3 * cus ? 3.0 : 4.0;
      r = (double)tiles / cus;
      r += (t.mt * t.nt == 16 ? 1.0 : rest) * (rounds - r);
    }
    const double step = t.c[type] + (t.mt < rows_a ? t.mt : rows_a) * split_a + (t.nt < rows_b ? t.nt : rows_b) * split_b;
    const double busy = r * (t.b[type] + step * steps), us = kSmallFixed + (busy > stream ? busy : stream);
    if (*tile < 0 || us < best) {
      best = us;
      *tile = i;
    }
  }
  return best;
}

template <int DT>
static int gemm_small_dispatch(const GemmArgs& g, int tile, hipStream_t s) {
  switch (tile) {
    case 0: return launch_small<DT, 1, 1, 16>(g, s);
    case 1: return launch_small<DT, 1, 2, 8>(g, s);
    case 2: return launch_small<DT, 1, 4, 8>(g, s);
    case 3: return launch_small<DT, 2, 2, 8>(g, s);
    case 4: return launch_small<DT, 2, 4, 4>(g, s);
    default: return launch_small<DT, 4, 4, 8>(g, s);
  }
}

int gemm_small(const GemmArgs& g, int dtype, int tile, hipStream_t s) {
  switch (dtype) {
    case LH_F32: return gemm_small_dispatch<LH_F32>(g, tile, s);
    case LH_BF16: return gemm_small_dispatch<LH_BF16>(g, tile, s);
    case LH_F16: return gemm_small_dispatch<LH_F16>(g, tile, s);
    default: return gemm_small_dispatch<LH_F8E4M3>(g, tile, s);
  }
}

}  // namespace lh
