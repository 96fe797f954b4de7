// LayerNorm and the projections that read it, in one launch, for few rows: out_i = act(LN(x) W_i + bias_i), x in f32, W and the
// LayerNorm's result in the matmul type (the first half of either branch of the nanoGPT block,
// examples/xegpu/nanoGPT_payload.py:299-317; rounding points as in the separate kernels: LN(x) rounded once to the
// matmul type, sums in f32).
//
// With few rows each of the block's launches is a chain of latencies of a few us.  Here every workgroup of the
// small-tile GEMM (gemm_small.hip) normalises the 16 MT rows of its tile itself: its waves request the weights of their
// whole share of K first, normalise a few rows each while those are on their way (a wave holds its rows in registers)
// and leave them in LDS, from where every wave reads its operand.  The rows are normalised again by every workgroup beside
// this one: L2 traffic and a few hundred instructions, against a launch and a trip of the result through memory.  Up to
// three weight matrices side by side (separate q, k and v) are one launch.
//
// The arithmetic is that of the separate kernels but for the order of the f32 sums: a row is added up over 32 lanes (layer_norm_vec:
// 64), and K is shared by eight waves on every tile (gemm_small.hip's 32 x 64 tile: by four).  A block of 100 rows of 768 bf16
// differs by 1.5e-5 for it, 12 of them, where 16-bit roundings fall the other way, by 3.2e-3; the error against 64 bits is the
// same (8 seeds each: block 8.503e-4 apart and 8.500e-4 here, 12 layers and a head 2.903e-3 and 2.901e-3).
#include "gemm_small.h"

namespace lh {

// Sum over 32 lanes, in each of them: the other half's 16 lanes, then rotations within 16 lanes.
__device__ __forceinline__ float norm_half_sum(float v) {
  float a = v, b = v;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  v = a + b;
  auto rotated = [](float x, auto n) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + decltype(n)::value, 0xf, 0xf, true));
  };
  v += rotated(v, std::integral_constant<int, 8>{});
  v += rotated(v, std::integral_constant<int, 4>{});
  v += rotated(v, std::integral_constant<int, 2>{});
  return v + rotated(v, std::integral_constant<int, 1>{});
}

// K = 128 V.  Half a wave holds a row (4 V elements per lane).
template <int DT, int MT, int NT, int NW, int V>
struct NormCfg {
  typedef SmallPanel<DT, NT, false> PB;
  static constexpr int ES = PB::ES, KSTEP = PB::KSTEP, K = 128 * V;
  static constexpr int P = (K / KSTEP + NW - 1) / NW;             // k-steps of a wave, at most; all are requested up front
  static constexpr int kRowBytes = K * ES + 16;                   // of a normalised row in LDS (one chunk of padding)
  static constexpr int kWorkBytes = 16 * MT * kRowBytes + NW * PB::kLdsBytes;
  static constexpr int kSumBytes = NW * MT * NT * 1024;
  static constexpr int kLdsBytes = kWorkBytes > kSumBytes ? kWorkBytes : kSumBytes;
};

template <int DT, int MT, int NT, int NW, int V>
__global__ void __launch_bounds__(NW * 64) gemm_normed_kernel(NormedGemm n) {
  typedef NormCfg<DT, MT, NT, NW, V> Cfg;
  constexpr int K = Cfg::K, KSTEP = Cfg::KSTEP, P = Cfg::P, ES = Cfg::ES;
  constexpr int R = 8 * MT / NW;  // pairs of rows a wave normalises
  static_assert(R >= 1 && R * NW == 8 * MT, "whole pairs of rows per wave");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_norm[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  GemmArgs g = n.g;
  // (tiles to workgroups as in gemm_small_kernel, the groups of columns one behind the other)
  const int tiles_m = (g.M + 16 * MT - 1) / (16 * MT), tiles_n = (g.N + 16 * NT - 1) / (16 * NT);
  const int tiles = tiles_m * tiles_n * n.groups, per_xcd = (tiles + 7) / 8;
  if ((int)blockIdx.x >= 8 * per_xcd) {
    touch_lines(n.next, blockIdx.x - 8 * per_xcd);
    return;
  }
  const int tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (tile >= tiles) return;
  const int panel = tile / tiles_m, group = panel / tiles_n;
  const int m0 = (tile % tiles_m) * 16 * MT, n0 = (panel % tiles_n) * 16 * NT;
  // (the group's columns of the output, and its bias)
  g.out = reinterpret_cast<uint8_t*>(g.out) + (int64_t)group * g.N * ES;
  g.bias = group == 0 ? n.bias[0] : group == 1 ? n.bias[1] : n.bias[2];
  uint8_t* const rows = smem_norm;
  uint8_t* const lds_b = smem_norm + 16 * MT * Cfg::kRowBytes + wave * Cfg::PB::kLdsBytes;

  // The wave's rows of x, gamma and beta, then its steps of the weights and what the epilogue needs: requested in this order,
  // waited for in this order.
  const int l32 = lane & 31, row0 = wave * 2 * R + (lane >> 5);
  f32x4 x[R][V], gamma[V], beta[V];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float* p = reinterpret_cast<const float*>(g.a) + (int64_t)min(m0 + row0 + 2 * r, g.M - 1) * g.lda + 4 * l32;
#pragma unroll
    for (int i = 0; i < V; ++i) x[r][i] = *reinterpret_cast<const f32x4*>(p + 128 * i);
  }
#pragma unroll
  for (int i = 0; i < V; ++i) {
    gamma[i] = *reinterpret_cast<const f32x4*>(n.gamma + 128 * i + 4 * l32);
    beta[i] = *reinterpret_cast<const f32x4*>(n.beta + 128 * i + 4 * l32);
  }
  asm volatile("" ::: "memory");  // (the weights, which come from further away, behind them)
  typename Cfg::PB pb;
  pb.place(group == 0 ? n.b[0] : group == 1 ? n.b[1] : n.b[2], n0, g.N, g.ldb, lane);
  constexpr int full = K / KSTEP;
  const int begin = full * wave / NW, mine = full * (wave + 1) / NW - begin;
  u32x4 rb[P][NT];
#pragma unroll
  for (int p = 0; p < P; ++p) pb.load(min(begin + p, full - 1) * KSTEP, rb[p]);
  asm volatile("" ::: "memory");
  SmallEpilogue<DT, MT, NT, NW> epilogue;
  epilogue.load(g, m0, n0, wave, lane);

  // LayerNorm of the rows, two at a time
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < V; ++i) s += (x[r][i][0] + x[r][i][1]) + (x[r][i][2] + x[r][i][3]);
    const float mean = norm_half_sum(s) * n.inv_n;
    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < V; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[r][i][e] -= mean;
        q += x[r][i][e] * x[r][i][e];
      }
    const float inv_std = rsqrtf(norm_half_sum(q) * n.inv_n + n.eps);
    uint8_t* const row = rows + (row0 + 2 * r) * Cfg::kRowBytes + 4 * ES * l32;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = x[r][i][e] * inv_std * gamma[i][e] + beta[i][e];
      *reinterpret_cast<u32x2*>(row + 128 * ES * i) = u32x2{pack2<DT>(o[0], o[1]), pack2<DT>(o[2], o[3])};
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  f32x4 acc[MT][NT];
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[j][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const uint8_t* const frag_row = rows + (lane & 15) * Cfg::kRowBytes + (lane >> 4) * 16 + begin * 64;
  const bool whole = pb.whole;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    if (p >= mine) break;
    u32x4 fa[MT], fb[NT];
    if (whole) pb.template stage<true>(rb[p], lds_b, lane);
    else pb.template stage<false>(rb[p], lds_b, lane);
#pragma unroll
    for (int j = 0; j < MT; ++j) fa[j] = *reinterpret_cast<const u32x4*>(frag_row + 16 * j * Cfg::kRowBytes + p * 64);
    pb.fragments(rb[p], lds_b, lane, fb);
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int i = 0; i < NT; ++i) acc[j][i] = small_mma<DT>(fb[i], fa[j], acc[j][i]);
  }
  __syncthreads();  // (the areas overlap)
  epilogue.sum_and_store(true, g, acc, smem_norm, m0, n0, wave, lane);
}

template <int DT, int MT, int NT, int NW, int V>
static int launch_normed_rows(const NormedGemm& n, hipStream_t s) {
  typedef NormCfg<DT, MT, NT, NW, V> Cfg;
  auto kern = gemm_normed_kernel<DT, MT, NT, NW, V>;
  static bool configured = false;
  if (Cfg::kLdsBytes > 64 * 1024 && !configured && !planning()) {
    LH_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     Cfg::kLdsBytes));
    configured = true;
  }
  const int tiles = ((n.g.M + 16 * MT - 1) / (16 * MT)) * ((n.g.N + 16 * NT - 1) / (16 * NT)) * n.groups;
  static_assert(NW == 8, "touch_lines counts on 512 threads");
  const unsigned blocks = 8 * (((unsigned)tiles + 7) / 8);
  LH_LAUNCH(kern, dim3(blocks + touch_blocks(n.next, blocks)), dim3(NW * 64), Cfg::kLdsBytes, s, n);
  return check_launch("gemm_normed");
}

template <int DT, int MT, int NT, int NW>
static int launch_normed(const NormedGemm& n, hipStream_t s) {
  switch (n.g.K / 128) {
    case 1: return launch_normed_rows<DT, MT, NT, NW, 1>(n, s);
    case 2: return launch_normed_rows<DT, MT, NT, NW, 2>(n, s);
    case 3: return launch_normed_rows<DT, MT, NT, NW, 3>(n, s);
    case 4: return launch_normed_rows<DT, MT, NT, NW, 4>(n, s);
    case 5: return launch_normed_rows<DT, MT, NT, NW, 5>(n, s);
    case 6: return launch_normed_rows<DT, MT, NT, NW, 6>(n, s);
    case 7: return launch_normed_rows<DT, MT, NT, NW, 7>(n, s);
    default: return launch_normed_rows<DT, MT, NT, NW, 8>(n, s);
  }
}

// ---- choice of tile ---------------------------------------------------------------------------
// Time of the launch, in us: fixed + r (b + c K), r = workgroups per compute unit (at least 1; a last round that is not whole
// counts for 0.6 of what it lacks).  Least squares over 140 problems (M 16 .. 1000, K 256 .. 1024, N 3 K and 4 K; 5 to 7 % rms); 16 x 16 and
// 32 x 32 tiles were never the fastest by more than 0.3 us.  What stands against it: 5.25 us for the LayerNorm's launch and its
// gap, and each product at 1.4 times gemm16_us (which was fitted on operands that stayed in the caches) plus 1.5 for
// every launch after the first.  Choosing so is within 0.4 % of the faster way on average (1.13 x at worst); M = 100, K = 768,
// N = 2304 bf16: 3.1 + 5.6 us and a gap against 7.3 us, M = 400: 3.9 + 9.3 against 14.3, and the LayerNorm stays on its own.
struct NormedTile {
  int mt, nt;
  double fixed, b, c;
};
constexpr NormedTile kNormedTiles[] = {{1, 2, 3.05, -0.11, 0.0040}, {1, 4, 2.99, -0.02, 0.0055}, {2, 4, 2.50, 0.89, 0.0066}};

int gemm_normed_choose(const NormedGemm& n, int dtype) {
  const GemmArgs& g = n.g;
  if (dtype == LH_F32 || g.K % 128 != 0 || g.K > 1024 || g.N < 8 || g.lda % 4 != 0 || !aligned16(g.a) || !aligned16(n.gamma) ||
      !aligned16(n.beta) || (int64_t)g.M * g.N >= 1ll << 36)
    return -1;
  const int cus = num_cus();
  int tile = -1;
  double best = 0.0;
  for (int i = 0; i < 3; ++i) {
    const NormedTile& t = kNormedTiles[i];
    const int64_t tiles = (int64_t)((g.M + 16 * t.mt - 1) / (16 * t.mt)) * ((g.N + 16 * t.nt - 1) / (16 * t.nt)) * n.groups;
    if (tiles > 4 * (int64_t)cus) continue;
    double r = 1.0;
    if (tiles > cus) {
      r = (double)tiles / cus;
      r += 0.6 * ((double)((tiles + cus - 1) / cus) - r);
    }
    const double us = t.fixed + r * (t.b + t.c * g.K);
    if (tile < 0 || us < best) {
      best = us;
      tile = i;
    }
  }
  if (tile < 0) return -1;
  GemmArgs one = g;
  one.b = n.b[0];
  one.a = n.b[0];  // (for its alignment, which the LayerNorm's own output has as well)
  one.lda = g.K;
  const double apart = 5.25 + 1.4 * n.groups * gemm16_us(one, dtype) + 1.5 * (n.groups - 1);
  return best < apart ? tile : -1;
}

int gemm_normed(const NormedGemm& n, int dtype, int tile, hipStream_t s) {
  if (dtype == LH_BF16)
    return tile == 0 ? launch_normed<LH_BF16, 1, 2, 8>(n, s) : tile == 1 ? launch_normed<LH_BF16, 1, 4, 8>(n, s) : launch_normed<LH_BF16, 2, 4, 8>(n, s);
  return tile == 0 ? launch_normed<LH_F16, 1, 2, 8>(n, s) : tile == 1 ? launch_normed<LH_F16, 1, 4, 8>(n, s) : launch_normed<LH_F16, 2, 4, 8>(n, s);
}

}  // namespace lh
