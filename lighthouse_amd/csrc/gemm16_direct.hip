// Direct-to-LDS GEMM kernels for 16-bit inputs.  This source is compiled once per instantiation (the objects
// are what takes long to build): LH_GEMM16_DT the element type, LH_GEMM16_TM and LH_GEMM16_TN the workgroup tile
// (64 TM) x (128 TN); LH_GEMM16_TM 0: the launches cut along K; LH_GEMM16_LARGE 1: the launches of large results (256 x 256); LH_GEMM16_ODD 1:
// the 128 x 128 tile on a B in rows of any length; LH_GEMM16_DEEP 1: the tile (128 x 128, 128 x 192, 128 x 256, 256 x 128) where no CU gets
// two workgroups.
#include <type_traits>

#include "gemm16.h"

namespace lh {

constexpr int kBK = 64;

// ---- direct-to-LDS kernels --------------------------------------------------------------
// Workgroup tile (64 TM) x (128 TN), 8 waves as 2 x 4, (32 TM) x (32 TN) per wave; TM x TN is
// 4 x 2 (256 x 256), 4 x 1 (256 x 128), 2 x 2 (128 x 256) or 2 x 1 (128 x 128).  Both panels go
// global -> LDS with buffer_load_dwordx4 ... lds (no register staging, no LDS store instructions) in
// their GLOBAL orientation.  The k-contiguous A fragment is one 16-byte LDS read; the
// n-contiguous B panel is read with ds_read_b64_tr_b16, which hands each lane 4 k-values of one
// column, i.e. the MFMA operand layout, transposing in the LDS crossbar.
//
// The matrix instruction is v_mfma_f32_16x16x32 (16 rows x 16 columns x 32 k), not 32x32x16: for
// the same products it keeps the matrix cores' clock higher on random operands (a register-only
// loop of either runs at the published peak on zeros, but at 2.02 against 1.74 PFLOP/s on N(0,1)
// data).  A wave's sub-tile is 2 TM fragments of 16 rows by 2 TN fragments of 16 columns per 32 k.
//
// LDS rings: A in 2 stages of 64 k (rows of 128 bytes: every global request is a full 128-byte
// line), B in 4 stages of 32 k.  The main loop advances 32 k per step, each step in two phases:
// the MFMAs of the wave's lower TM row fragments, then of its upper ones, all against the step's
// 2 TN column fragments.  The LDS reads of a phase fetch what the next phase needs (the other
// half of the A fragments; in the second phase also the next step's B fragments, each after the
// last MFMA that uses its predecessor), so reads always overlap MFMAs.  The barrier sits between
// the two phases of a step and the buffers a step has finished reading are refilled right
// behind it (B: 3 stages ahead, A: on odd steps, one 64-k stage ahead).
// That is the form of the launches cut along K; the others run one with a single barrier per 64 k, the rings as two
// halves: direct_step_pair_1b.  Where no CU gets a second workgroup, rings of three or four such halves: gemm16_deep.
//
// A wave-wide load into LDS writes 64 x 16 contiguous LDS bytes, so rows cannot be padded;
// bank conflicts are avoided by XOR-swizzling which 16-byte chunk of a row each lane fetches
// (A: chunk ^ ((row / 2) % 8); B: chunk ^ 4 (k % 4) ^ 2 ((k / 8) % 2)).
// TN 3 stands for 192 columns (gemm16_deep alone): three fragments of 16 columns for each of the four waves side by side.
constexpr int direct_frags(int TN) { return TN == 3 ? 3 : 2 * TN; }
template <int TM, int TN>
struct DirectCfg {
  static constexpr int NF = direct_frags(TN);             // 16-column fragments of a wave
  static constexpr int BM = 64 * TM, BN = 64 * NF;
  static constexpr int WTM = 32 * TM, WTN = 16 * NF;      // per-wave sub-tile
  static constexpr int kABytes = BM * 64 * 2;             // one A stage (64 k)
  static constexpr int kBRow = BN * 2;                    // bytes of one k row of a B stage
  static constexpr int kBBytes = 32 * kBRow;              // one B stage (32 k)
  static constexpr int kBtBytes = BN * 64 * 2;            // one stage (64 k) of a transposed B: rows n, like A
  // What the 16-byte chunks of k row `k` of an n-contiguous B are swapped with.  Rows of a multiple of 256 bytes start at the same
  // bank; of the rows of 384 bytes every other one starts half way through the banks.
  __device__ static constexpr int b_swizzle(int k) {
    return TN == 3 ? (4 * ((k >> 1) & 1)) ^ (2 * ((k >> 3) & 1)) : (4 * (k & 3)) ^ (2 * ((k >> 3) & 1));
  }
  static constexpr int kBBase = 2 * kABytes;
  static constexpr int kRingBytes = kBBase + 4 * kBBytes;
  static constexpr int kStageBytes = 8 * 32 * WTN * 2;    // output staging: 32 rows of each wave's sub-tile
  static constexpr int kStagedStores = TM * NF;           // 16-byte stores per lane of a staged epilogue
  static constexpr int kLdsBytes = kRingBytes + kStageBytes;
  static constexpr int kBChunks = kBRow / 16;             // 16-byte chunks per B row
  static constexpr int kBRowsPerLoad = 1024 / kBRow;      // k rows one wave-wide load covers
  // Loads a lane has in flight per stage, hence the s_waitcnt immediates of the main loop.
  static constexpr int kWaitEven = TM + 2 * TN;
  static constexpr int kWaitOdd = 2 * TN;
};

typedef __attribute__((address_space(3))) void lds_void_t;
typedef short s16x4 __attribute__((ext_vector_type(4)));

// 16 bytes per lane from a buffer resource (base + per-lane byte offset + scalar byte offset)
// straight into LDS, 1 KiB per wave starting at lds_wave_base.  The buffer form of the LDS-DMA
// load, not the global (flat-encoded) one: with a flat-encoded LDS access in flight the compiler
// must assume that LDS operations complete out of order and turns every s_waitcnt on an LDS read
// into lgkmcnt(0); with the buffer form it counts, so a fragment read issued a few MFMAs ago is
// not waited for behind the ones issued last.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, int lane_bytes, int scalar_bytes,
                                      uint8_t* lds_wave_base) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t*)lds_wave_base, 16, lane_bytes, scalar_bytes, 0, 0);
}
// A resource over [base, base + 2 GiB): raw (unstructured) addressing, offsets in bytes; a load at kOutside or beyond
// touches no memory and leaves zeros in LDS.  The kernels cut along K (the
// object without a tile) say that the base is uniform: the compiler keeps the panel addresses of their edge tiles, which come
// out of the divisions that select a piece of K, in vector registers and wrote a loop over the lanes' resources around every
// load (M = 1, N = 5376, K = 4736 bf16: 24.0 us without such loops, 28.4 with them).
constexpr uint32_t kOutside = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t panel_resource(const void* base) {
#if LH_GEMM16_TM == 0
  const uint64_t address = reinterpret_cast<uint64_t>(base);
  base = reinterpret_cast<const void*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(address >> 32)) << 32 |
                                       (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)address));
#endif
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, kOutside, 0x00020000);
}
template <int TM, int TN>
struct DirectCtx {
  const uint16_t* a_base;     // the tile's A row panel and B column panel (uniform; the buffer
  const uint16_t* b_base;     // resources are made from them at each load: four scalar moves)
  int a_src[TM];              // lane's byte offset in the A panel for load i at k = 0
  int b_src[TN];
  int b_step;                 // bytes between B stages (32 k rows)
  // Fragment reads.  A: the lane's first row (wm0 + lane % 16) of a stage, its 16-byte chunk for the
  // first / second 32 k of the stage's 64 (fragment jj, 16 rows further on, adds 2048 jj: the
  // swizzle term (row / 2) % 8 does not change with 16 rows).
  int a_rd[2];
  int wave, b_off, b_chunk, b_swz;
  int k_end;                  // (TAIL) K: loads past it bring zeros
  // B stored transposed ([N, K], k contiguous): its panel is laid out, loaded and read like A's
  int bt_src[direct_frags(TN)];         // lane's byte offset in the B^T panel for load i at k = 0
  int bt_rd[2];               // like a_rd, for row wn0 + lane % 16 of a B^T stage
};

// Fragments in registers: the A fragments of the lower (a[0]) and upper (a[1]) half of the wave's
// rows, TM of 16 rows each, and the step's 2 TN B fragments of 16 columns.
template <int TM, int TN>
struct DirectFrags {
  u32x4 a[2][TM];
  u32x4 b[direct_frags(TN)];
};

// The lane's 16-byte chunk of a 128-byte row of a k-contiguous stage lies past the end of K (of which `left` remain at the
// start of the stage): the chunk is (lane % 8) ^ ((row / 2) % 8) of row 8 (8 i + wave) + lane / 8, the same for every i.
__device__ __forceinline__ bool direct_past_k(int wave, int left) {
  const int lane = lane_now();
  return 8 * ((lane & 7) ^ ((4 * wave + (lane >> 4)) & 7)) >= left;
}
// A stage `sa` (k = 64 sa .. +64): TM loads per lane.  TAIL: K may end inside it, at a multiple of 8.
template <int TM, int TN, bool TAIL>
__device__ __forceinline__ void direct_load_a(const DirectCtx<TM, TN>& c, int sa, uint8_t* __restrict__ abuf) {
  const __amdgpu_buffer_rsrc_t rsrc = panel_resource(c.a_base);
  if (TAIL && 64 * sa + 64 > c.k_end) {
    const bool past = direct_past_k(c.wave, c.k_end - 64 * sa);
#pragma unroll
    for (int i = 0; i < TM; ++i) dma16(rsrc, past ? (int)kOutside : c.a_src[i], sa * 128, abuf + (8 * i + c.wave) * 1024);
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) dma16(rsrc, c.a_src[i], sa * 128, abuf + (8 * i + c.wave) * 1024);
}
// B stage `sb` (k = 32 sb .. +32; 192 columns: 64 sb .. +64, TAIL not): TN loads per lane.  BT (B stored [N, K]): stage sb is k = 64 sb .. +64
// of the panel's rows, 2 TN loads per lane.
template <int TM, int TN, bool BT, bool TAIL>
__device__ __forceinline__ void direct_load_b(const DirectCtx<TM, TN>& c, int sb, uint8_t* __restrict__ bbuf) {
  const __amdgpu_buffer_rsrc_t rsrc = panel_resource(c.b_base);
  if constexpr (BT) {
    if (TAIL && 64 * sb + 64 > c.k_end) {
      const bool past = direct_past_k(c.wave, c.k_end - 64 * sb);
#pragma unroll
      for (int i = 0; i < direct_frags(TN); ++i) dma16(rsrc, past ? (int)kOutside : c.bt_src[i], sb * 128, bbuf + (8 * i + c.wave) * 1024);
      return;
    }
#pragma unroll
    for (int i = 0; i < direct_frags(TN); ++i) dma16(rsrc, c.bt_src[i], sb * 128, bbuf + (8 * i + c.wave) * 1024);
  } else {
    static_assert(!TAIL || TN != 3, "whole stages");
    if (TAIL && 32 * sb + 32 > c.k_end) {
      using Cfg = DirectCfg<TM, TN>;
      const int lane = lane_now();
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        const int k = 32 * sb + (8 * i + c.wave) * Cfg::kBRowsPerLoad + lane / Cfg::kBChunks;
        dma16(rsrc, k >= c.k_end ? (int)kOutside : c.b_src[i], sb * c.b_step, bbuf + (8 * i + c.wave) * 1024);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < TN; ++i) dma16(rsrc, c.b_src[i], (TN == 3 ? 2 * sb : sb) * c.b_step, bbuf + (8 * i + c.wave) * 1024);
  }
}

// A fragments of one half of the wave's rows (HALF 0: 16-row fragments 0 .. TM-1, 1: TM .. 2 TM-1)
// for the 32 k `kc` (0 / 1) of the 64-k stage `as`.
template <int TM, int TN, int HALF>
__device__ __forceinline__ void direct_read_a(const DirectCtx<TM, TN>& c, const uint8_t* __restrict__ as, int kc,
                                              u32x4 (&a)[TM]) {
#pragma unroll
  for (int j = 0; j < TM; ++j) a[j] = *reinterpret_cast<const u32x4*>(as + c.a_rd[kc] + 2048 * (HALF * TM + j));
}
// B fragment i (16 columns) of a 32-k step: from the 32-k stage `bs` of an n-contiguous B through two
// transposing reads, or (BT) from the 32 k `kc` of the 64-k stage `bs` of a transposed B like an A fragment.
template <int TM, int TN, bool BT>
__device__ __forceinline__ u32x4 direct_read_b(const DirectCtx<TM, TN>& c, const uint8_t* __restrict__ bs, int kc,
                                               int i) {
  if constexpr (BT) {
    return *reinterpret_cast<const u32x4*>(bs + c.bt_rd[kc] + 2048 * i);
  } else {
    constexpr int row = DirectCfg<TM, TN>::kBRow;
    const int p = (c.b_chunk + 2 * i) ^ c.b_swz;
    const uint8_t* p0 = bs + c.b_off + p * 16;
    s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p0);
    s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p0 + 4 * row));
    u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
    return u32x4{l2[0], l2[1], h2[0], h2[1]};
  }
}

// Scheduling hint for one phase: spread its NR LDS reads evenly between its NM MFMAs.
template <int I, int NM, int NR>
__device__ __forceinline__ void direct_interleave_step() {
  __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                // MFMA
  __builtin_amdgcn_sched_group_barrier(0x100, (I + 1) * NR / NM - I * NR / NM, 0);  // DS reads
  if constexpr (I + 1 < NM) direct_interleave_step<I + 1, NM, NR>();
}

// First phase of a step: the MFMAs of the lower row fragments (f.a[0]) against the step's B
// fragments, under the reads of the same step's upper row fragments (32 k `kc` of stage `as`).
template <int DT, int TM, int TN>
__device__ __forceinline__ void direct_phase_lo(const DirectCtx<TM, TN>& c, f32x4 (&acc)[direct_frags(TN)][2 * TM],
                                                DirectFrags<TM, TN>& f, const uint8_t* __restrict__ as, int kc) {
  direct_read_a<TM, TN, 1>(c, as, kc, f.a[1]);
#pragma unroll
  for (int i = 0; i < direct_frags(TN); ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = Mfma16<DT>::mma16(f.b[i], f.a[0][j], acc[i][j]);
  direct_interleave_step<0, direct_frags(TN) * TM, TM>();
}
// Second phase: the MFMAs of the upper row fragments (f.a[1]) under the reads of the NEXT step's
// lower row fragments (32 k `kc_n` of A stage `as_n`) and B fragments (stage `bs_n`; BT: its 32 k
// `kc_n`), each B fragment requested behind the last MFMA that uses the one it replaces.
// LOAD false: the tile's last step, nothing left to read.
template <int DT, int TM, int TN, bool BT, bool LOAD = true>
__device__ __forceinline__ void direct_phase_hi(const DirectCtx<TM, TN>& c, f32x4 (&acc)[direct_frags(TN)][2 * TM],
                                                DirectFrags<TM, TN>& f, const uint8_t* __restrict__ as_n,
                                                const uint8_t* __restrict__ bs_n, int kc_n) {
  if constexpr (LOAD) direct_read_a<TM, TN, 0>(c, as_n, kc_n, f.a[0]);
  u32x4 bn[direct_frags(TN)];
#pragma unroll
  for (int i = 0; i < direct_frags(TN); ++i) {
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][TM + j] = Mfma16<DT>::mma16(f.b[i], f.a[1][j], acc[i][TM + j]);
    if constexpr (LOAD) bn[i] = direct_read_b<TM, TN, BT>(c, bs_n, kc_n, i);
  }
  if constexpr (LOAD) {
#pragma unroll
    for (int i = 0; i < direct_frags(TN); ++i) f.b[i] = bn[i];
    direct_interleave_step<0, direct_frags(TN) * TM, TM + (BT ? 1 : 2) * direct_frags(TN)>();
  }
}
// Wait until at most N of this wave's loads are still in flight and all its LDS reads have
// returned, then barrier.  One asm block: a __syncthreads() would add a release fence, i.e. a
// wait for ALL outstanding loads, and drain the rings.
template <int N>
__device__ __forceinline__ void direct_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}


// Steps kt (even) and kt + 1 of the main loop; both have a successor step.  On entry f holds the
// lower row fragments and the B fragments of step kt.  a_cur = A stage kt / 2, a_nxt = the next A
// stage, b1 / b2 = B stages kt + 1, kt + 2.  The refill pointers alias a_cur and B stages kt and
// kt + 1: every read of a buffer precedes the barrier after which it is refilled.  They are
// separate restrict parameters so that the compiler does not make LDS reads wait for the
// asynchronous writes.
//
// In-flight loads, oldest first, when a barrier is reached (steady state):
//   even step: [A(kt/2) B(kt+1)] [B(kt+2)] [A(kt/2+1) B(kt+3)]  -> B(kt+1) needed: TM + 2 TN may remain
//   odd step : [B(kt+1)] [A((kt+1)/2) B(kt+2)] [B(kt+3)]        -> A needed: 2 TN may remain
// Near the end loads are no longer issued and the waits become full waits.
template <int DT, int TM, int TN, bool TAIL>
__device__ __forceinline__ void direct_step_pair(const DirectCtx<TM, TN>& c, f32x4 (&acc)[direct_frags(TN)][2 * TM],
                                                 DirectFrags<TM, TN>& f, const uint8_t* __restrict__ a_cur,
                                                 const uint8_t* __restrict__ a_nxt, const uint8_t* __restrict__ b1,
                                                 const uint8_t* __restrict__ b2, uint8_t* __restrict__ a_refill,
                                                 uint8_t* __restrict__ b_refill0, uint8_t* __restrict__ b_refill1,
                                                 int kt, int nk) {
  using Cfg = DirectCfg<TM, TN>;
  const bool steady = kt + 6 < nk;  // all loads of both steps are real
  // ---- even step kt
  direct_phase_lo<DT>(c, acc, f, a_cur, 0);
  if (steady) direct_wait_barrier<Cfg::kWaitEven>();
  else direct_wait_barrier<0>();
  if (kt + 4 < nk) direct_load_b<TM, TN, false, TAIL>(c, kt + 4, b_refill0);
  direct_phase_hi<DT, TM, TN, false>(c, acc, f, a_cur, b1, 1);
  // ---- odd step kt + 1
  direct_phase_lo<DT>(c, acc, f, a_cur, 1);
  if (steady) direct_wait_barrier<Cfg::kWaitOdd>();
  else direct_wait_barrier<0>();
  if (kt + 4 < nk) direct_load_a<TM, TN, TAIL>(c, kt / 2 + 2, a_refill);
  if (kt + 5 < nk) direct_load_b<TM, TN, false, TAIL>(c, kt + 5, b_refill1);
  direct_phase_hi<DT, TM, TN, false>(c, acc, f, a_nxt, b2, 0);
}

// Source pointers of tile `id` (its position in the XCD-grouped order) and the tile's origin.
// EDGE: M and N need not be multiples of the tile (K of 64, or with TAIL of 8; an n-contiguous B has rows of a multiple of
// 8 columns, padded if N is none): loads of rows / column chunks past the end are redirected to the last valid
// row / chunk (their products land in accumulators that are never stored).  The epilogue skips what lies
// outside the matrix and takes any alignment of output, bias and accumulator input.
template <int TM, int TN, bool EDGE, bool BT = false>
__device__ __forceinline__ void direct_place(const GemmArgs& g, int id, DirectCtx<TM, TN>& c, int& m0, int& n0) {
  using Cfg = DirectCfg<TM, TN>;
  constexpr int BM = Cfg::BM, BN = Cfg::BN;
  const int lane = lane_now();
  const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
  // Tiles are walked in groups of GROUP_M tile rows: 1024 rows of A.  For the 128-row tiles that
  // is 8 up to K = 1536 (1-3 % faster than 4 there; 0.3-1.4 % slower from K = 3072 on).
  const int GROUP_M = (BM == 128 && g.K <= 1536) ? 8 : 4;
  const int group_size = GROUP_M * tiles_n;
  const int first_m = (id / group_size) * GROUP_M;
  const int gm = min(tiles_m - first_m, GROUP_M);
  m0 = (first_m + (id % group_size) % gm) * BM;
  n0 = ((id % group_size) / gm) * BN;
  const uint16_t* A = reinterpret_cast<const uint16_t*>(g.a);
  const uint16_t* B = reinterpret_cast<const uint16_t*>(g.b);
  const int lda = (int)g.lda, ldb = (int)g.ldb;
  c.a_base = A + (int64_t)m0 * g.lda;
  c.b_base = BT ? B + (int64_t)n0 * g.ldb : B + n0;
  c.b_step = 64 * ldb;
  // A: load i of wave w fills rows (8 i + w) 8 .. +8 (1024 bytes); lane -> row += lane / 8, LDS
  // chunk p = lane % 8 holds global chunk p ^ ((row / 2) % 8).
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int ar = (8 * i + c.wave) * 8 + (lane >> 3);
    const int ac = (lane & 7) ^ ((ar >> 1) & 7);
    const int arow = EDGE ? min(ar, g.M - 1 - m0) : ar;  // row within the panel
    c.a_src[i] = (arow * lda + ac * 8) * 2;
  }
  // B: load i of wave w fills k rows (8 i + w) R .. +R with R = 1024 / row bytes; lane ->
  // row += lane / chunks-per-row, LDS chunk p holds global chunk p ^ 4 (k % 4) ^ 2 ((k / 8) % 2): the
  // four k rows a 16-lane group reads at once land in different banks, and so do the rows (8 apart)
  // of the group next to it.
  if constexpr (BT) {
    // B^T: exactly A's scheme on the panel's BN rows (row n of B^T = column n of B)
#pragma unroll
    for (int i = 0; i < direct_frags(TN); ++i) {
      const int br = (8 * i + c.wave) * 8 + (lane >> 3);
      const int bc = (lane & 7) ^ ((br >> 1) & 7);
      const int brow = EDGE ? min(br, g.N - 1 - n0) : br;
      c.bt_src[i] = (brow * ldb + bc * 8) * 2;
    }
  } else {
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      // (192 columns: i = 0 .. 2 are the two stages of 64 k rows, 24 chunks each, one behind the other)
      const int chunk = (8 * i + c.wave) * 64 + lane, bk = chunk / Cfg::kBChunks;
      const int bc = chunk % Cfg::kBChunks ^ Cfg::b_swizzle(bk);
      const int bcol = EDGE ? min(bc * 8, (g.N + 7) / 8 * 8 - 8 - n0) : bc * 8;  // column within the panel
      c.b_src[i] = (bk * ldb + bcol) * 2;
    }
  }
}

// The same two steps with ONE barrier, in the middle of the odd step: the rings work as two halves
// of 64 k.  At the barrier every read of this pair's stages has returned and the next pair's
// stages (issued at the previous barrier, 64 k ago) are awaited in full; the pair after that is
// then requested into this pair's buffers.  BT: b1 is the pair's one 64-k stage of B^T, b2 the next.
template <int DT, int TM, int TN, bool TAIL, bool BT = false>
__device__ __forceinline__ void direct_step_pair_1b(const DirectCtx<TM, TN>& c, f32x4 (&acc)[direct_frags(TN)][2 * TM],
                                                    DirectFrags<TM, TN>& f, const uint8_t* __restrict__ a_cur,
                                                    const uint8_t* __restrict__ a_nxt, const uint8_t* __restrict__ b1,
                                                    const uint8_t* __restrict__ b2, uint8_t* __restrict__ a_refill,
                                                    uint8_t* __restrict__ b_refill0, uint8_t* __restrict__ b_refill1,
                                                    int kt, int nk, bool stores_behind) {
  using Cfg = DirectCfg<TM, TN>;
  direct_phase_lo<DT>(c, acc, f, a_cur, 0);
  direct_phase_hi<DT, TM, TN, BT>(c, acc, f, a_cur, b1, 1);
  direct_phase_lo<DT>(c, acc, f, a_cur, 1);
  // At a tile's first barrier the only operations in flight are the previous tile's stores (the
  // tile's first loads, older than they, were awaited when the main loop began): they may stay.
  // Matters for the 128 x 128 tile, whose first 64 k pass in 0.5 us (M = 8192, N = 2304, K = 768:
  // 35.15 -> 34.9 us); the large tiles' stores have long completed by then.
  if (TM * TN == 2 && stores_behind && kt == 0) direct_wait_barrier<Cfg::kStagedStores>();
  else direct_wait_barrier<0>();
  if (kt + 4 < nk) {
    direct_load_a<TM, TN, TAIL>(c, kt / 2 + 2, a_refill);
    if constexpr (BT) {
      direct_load_b<TM, TN, true, TAIL>(c, kt / 2 + 2, b_refill0);
    } else {
      direct_load_b<TM, TN, false, TAIL>(c, kt + 4, b_refill0);
      direct_load_b<TM, TN, false, TAIL>(c, kt + 5, b_refill1);
    }
  }
  direct_phase_hi<DT, TM, TN, BT>(c, acc, f, a_nxt, b2, 0);
}

// First loads of a tile: A stages 0, 1 and B stages 0 .. 3 (nk >= 2); BT: both 64-k stages of B^T.
template <int TM, int TN, bool TAIL, bool BT = false>
__device__ __forceinline__ void direct_prologue(const DirectCtx<TM, TN>& c, int nk, uint8_t* __restrict__ ring) {
  using Cfg = DirectCfg<TM, TN>;
  direct_load_a<TM, TN, TAIL>(c, 0, ring);
  if (nk > 2) direct_load_a<TM, TN, TAIL>(c, 1, ring + Cfg::kABytes);
  if constexpr (BT) {
    direct_load_b<TM, TN, true, TAIL>(c, 0, ring + Cfg::kBBase);
    if (nk > 2) direct_load_b<TM, TN, true, TAIL>(c, 1, ring + Cfg::kBBase + Cfg::kBtBytes);
  } else {
#pragma unroll
    for (int st = 0; st < 4; ++st)
      if (st < nk) direct_load_b<TM, TN, false, TAIL>(c, st, ring + Cfg::kBBase + st * Cfg::kBBytes);
  }
}

// Touches B, 4 bytes of every 128 (into the idle staging area, where nobody reads them), so that a B that is not in the caches
// comes out of memory at once.  Left to the main loop it comes 64 rows at a time, which every workgroup of the chip waits for
// together.  The workgroups share out the lines; more than 128 for each cost more at the start than the loop waits for later.
// bf16, M = 8192, N = 2304, K = 768: 45.6 us with B in memory before, 36.0 now (33.7 and 34.4 with B in the caches); N = 3072
// 56.6 and 48.2; with 256 lines for each workgroup (2048^3) 28.1 and 29.1.
// From K = 512 on.  Over 1700 products of 257 to 2048 tiles of 128 x 128, on it / without it, operands in the caches, B in memory, all in
// memory: K <= 448 1.010, 1.004, 1.000; 512 and 576 1.008, 1.000, 0.992; 640 ... 896 1.008, 0.992, 0.988; above 1.002, 0.970, 0.991 (B stored [N, K] gains
// a little earlier, at 512 0.98 with B in memory, and [K, N] later).
// (The launcher decides, and the code lies behind the kernel's: in its way it cost launches that touch nothing 0.1 to 0.3 us.
// The 256 x 256 tile has none of it: there a B of so few lines is a short K or a narrow result, and 4096^3 took 0.7 us longer.)
constexpr int kTouchFrom = 512;
template <bool BT>
__device__ __forceinline__ void direct_touch_b(const GemmArgs& g, int wave, uint8_t* __restrict__ stage) {
  const int per_row = ((BT ? g.K : g.N) + 63) / 64, lines = (BT ? g.N : g.K) * per_row, grid = (int)gridDim.x;
  if (64 * wave * grid >= lines) return;
  const int line = (64 * wave + lane_now()) * grid + (int)blockIdx.x;
  const int at = (line / per_row * (int)g.ldb + line % per_row * 64) * 2;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(panel_resource(g.b), (lds_void_t*)(stage + 256 * wave), 4,
                                           line < lines ? at : (int)kOutside, 0, 0, 0);
}

// The lane's 16-bit bias values for a staged epilogue, columns n_base + 16 i .. +4, as packed
// pairs; all loads are issued back to back.  (An f32 bias is read by the epilogue itself.)
template <int TN, bool EDGE>
__device__ __forceinline__ void direct_load_bias(const GemmArgs& g, int n_base, u32x2 (&bias)[direct_frags(TN)]) {
#pragma unroll
  for (int i = 0; i < direct_frags(TN); ++i) bias[i] = u32x2{0u, 0u};
  if (!(g.flags & LH_GEMM_HAS_BIAS) || g.bias_dt == LH_F32) return;
#pragma unroll
  for (int i = 0; i < direct_frags(TN); ++i) {
    const int n = n_base + 16 * i;
    const uint16_t* b = reinterpret_cast<const uint16_t*>(g.bias);
    if constexpr (EDGE) {
      if (n + 4 <= g.N) {
        bias[i] = *reinterpret_cast<const u32x2_any*>(b + n);
      } else {
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (n + e < g.N) bias[i][e >> 1] |= (uint32_t)b[n + e] << (16 * (e & 1));
      }
    } else {
      bias[i] = *reinterpret_cast<const u32x2*>(b + n);
    }
  }
}

// Main loop of one tile, whose first loads have been issued.
// `stores_behind`: the previous tile's staged epilogue issued exactly Cfg::kStagedStores stores
// per lane AFTER this tile's first loads; vector memory operations complete in issue order, so
// those stores may stay in flight.
// `staged`: the epilogue will want `bias` (for columns from n_base); it is loaded ahead of the
// last two steps, whose full wait covers it.
template <int DT, int TM, int TN, bool EDGE, bool TAIL, bool BT, bool SPLITK>
__device__ __forceinline__ void direct_mainloop(const GemmArgs& g, const DirectCtx<TM, TN>& c,
                                                f32x4 (&acc)[direct_frags(TN)][2 * TM], uint8_t* smem_d, int nk,
                                                bool stores_behind, bool staged, int n_base, u32x2 (&bias)[direct_frags(TN)]) {
  using Cfg = DirectCfg<TM, TN>;
  // One barrier per 64 k (loads one 64-k half of the rings ahead) or, where K is cut, two (B three 32-k stages
  // ahead): there B is streamed from memory and the deeper look-ahead wins (M = 16, N = K = 8192: 26.7 against 27.4 us).
  // One is 1-3 % faster for every tile with a 256 side (4096^3 109.8 -> 108.3 us) and 2-7 % for two 128 x 128 workgroups on a
  // CU (M = 8192, N = 768, K = 3072: 46.0 -> 42.9 us).
  // A transposed B lives in the rings as two 64-k stages like A and always takes the one-barrier form.
  constexpr bool one_barrier = BT || !SPLITK;
  uint8_t* const abuf = smem_d;
  uint8_t* const bbuf = smem_d + Cfg::kBBase;
  if (stores_behind) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(Cfg::kStagedStores) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  DirectFrags<TM, TN> f;
  direct_read_a<TM, TN, 0>(c, abuf, 0, f.a[0]);
#pragma unroll
  for (int i = 0; i < direct_frags(TN); ++i) f.b[i] = direct_read_b<TM, TN, BT>(c, bbuf, 0, i);
  int kt = 0;
  auto pair = [&] {
    uint8_t* a_cur = abuf + ((kt >> 1) & 1) * Cfg::kABytes;
    uint8_t* a_nxt = abuf + (((kt >> 1) + 1) & 1) * Cfg::kABytes;
    if constexpr (BT) {
      uint8_t* b_cur = bbuf + ((kt >> 1) & 1) * Cfg::kBtBytes;
      uint8_t* b_nxt = bbuf + (((kt >> 1) + 1) & 1) * Cfg::kBtBytes;
      direct_step_pair_1b<DT, TM, TN, TAIL, true>(c, acc, f, a_cur, a_nxt, b_cur, b_nxt, a_cur, b_cur, b_cur, kt, nk,
                                            stores_behind);
    } else {
      uint8_t* b0 = bbuf + (kt & 3) * Cfg::kBBytes;
      uint8_t* b1 = bbuf + ((kt + 1) & 3) * Cfg::kBBytes;
      uint8_t* b2 = bbuf + ((kt + 2) & 3) * Cfg::kBBytes;
      if constexpr (one_barrier) direct_step_pair_1b<DT, TM, TN, TAIL>(c, acc, f, a_cur, a_nxt, b1, b2, a_cur, b0, b1, kt, nk, stores_behind);
      else direct_step_pair<DT, TM, TN, TAIL>(c, acc, f, a_cur, a_nxt, b1, b2, a_cur, b0, b1, kt, nk);
    }
  };
  for (; kt + 2 < nk; kt += 2) pair();
  {
    // Last two steps: nothing left to load; stage nk - 1 of B must have landed.
    const uint8_t* a_cur = abuf + ((kt >> 1) & 1) * Cfg::kABytes;
    const uint8_t* b1 = BT ? bbuf + ((kt >> 1) & 1) * Cfg::kBtBytes : bbuf + ((kt + 1) & 3) * Cfg::kBBytes;
    if (staged) direct_load_bias<TN, EDGE>(g, n_base, bias);
    direct_phase_lo<DT>(c, acc, f, a_cur, 0);
    if constexpr (!one_barrier) direct_wait_barrier<0>();  // (one barrier per pair: awaited at the pair before)
    direct_phase_hi<DT, TM, TN, BT>(c, acc, f, a_cur, b1, 1);
    direct_phase_lo<DT>(c, acc, f, a_cur, 1);
    direct_phase_hi<DT, TM, TN, BT, false>(c, acc, f, a_cur, b1, 0);
  }
}

// f32 results in rows that do not start at multiples of 64 bytes (a language-model head over 50257 words), without an
// accumulator input.  A store that covers part of a 64-byte piece of memory costs far more than its share (the pieces
// are read and merged on the way out), and a row segment per wave leaves two such pieces in every 128 bytes.  Here the
// four waves side by side put 16 rows of their columns next to each other in `stage`, a wave then writes whole rows of
// the tile: the pieces that lie inside the row in 16-byte stores past the caches, the up to 15 elements in front of
// the first and behind the last such piece one by one through the L2, where the neighbouring tile's may still join them.
// M = 8192, N = 50257, K = 768 bf16, 256 x 256 tile: 1338 us with a segment per wave, 680 with whole rows.
template <int DT, int TM, int TN>
__device__ __forceinline__ void direct_finish_rows(const GemmArgs& g, int wave, uint8_t* __restrict__ stage,
                                                   const f32x4 (&acc)[direct_frags(TN)][2 * TM], int m0, int n0, int wm0, int wn0) {
  using Cfg = DirectCfg<TM, TN>;
  constexpr int BN = Cfg::BN, RB = BN * 4;            // bytes of a staged row, 32 of them
  static_assert(32 * RB == Cfg::kStageBytes, "16 rows of each half of the tile's rows");
  constexpr int RPS = 2 / TN, NS = 4 / RPS;           // rows per 64-lane store of 16 bytes; stores per wave
  const int lane = lane_now();
  const int l16 = lane & 15, g4 = lane >> 4;
  const int len = min(BN, g.N - n0);
  // Staged row r in turn j: row (r / 16) WTM + 16 j + r % 16 of the tile.  16 rows are a multiple of 64 bytes, so where
  // the pieces of a row start does not depend on j and all addresses below move by `turn` from one j to the next.
  const int64_t turn = 16 * g.ldc;
  auto tile_row = [](int r) { return (r >> 4) * Cfg::WTM + (r & 15); };
  // 16-byte chunk k of staged row r, swapped with one of 8 by the row against bank conflicts
  auto at = [](int r, int k) { return r * RB + ((k ^ (r & 7)) << 4); };
  struct Row {
    float* p;    // the row's first element in the tile
    int head;    // elements in front of the first piece
    int pieces;  // whole pieces
  };
  auto row_of = [&](int r) -> Row {
    float* const p = reinterpret_cast<float*>(g.out) + (int64_t)(m0 + tile_row(r)) * g.ldc + n0;
    const int head = (int)(-(reinterpret_cast<uintptr_t>(p) >> 2) & 15);
    return Row{p, head, max(len - head, 0) >> 4};
  };
  // Whole pieces: the lane stores elements head + 4 c .. +4 of its row, the end of one chunk and the start of the next.
  float* wide[NS];
  int wide_row[NS], wide_lds[NS];
  bool wide_ok[NS], by1[NS], by2[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) {
    const int r = 4 * wave + RPS * t + (RPS == 2 ? lane >> 5 : 0), c = RPS == 2 ? lane & 31 : lane;
    const Row row = row_of(r);
    wide[t] = row.p + row.head + 4 * c;
    wide_row[t] = m0 + tile_row(r);
    wide_ok[t] = c < 4 * row.pieces;
    wide_lds[t] = at(r, min((row.head >> 2) + c, RB / 16 - 1));
    by1[t] = row.head & 1;
    by2[t] = row.head & 2;
  }
  // The elements in front and behind: lanes 0 .. 15 and 16 .. 31 of a row's 32.
  float* edge[2];
  int edge_row[2], edge_lds[2];
  bool edge_ok[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int r = 4 * wave + 2 * t + (lane >> 5), c = lane & 15;
    const Row row = row_of(r);
    const bool tail = lane & 16;
    const int d = tail ? row.head + 16 * row.pieces + c : c;
    edge[t] = row.p + d;
    edge_row[t] = m0 + tile_row(r);
    edge_ok[t] = d < (tail ? len : min(row.head, len));
    edge_lds[t] = at(r, min(d, BN - 1) >> 2) + 4 * (d & 3);
  }
  epi_dispatch_linear(g, [&](auto variant) {
    using E = decltype(variant);
    f32x4 b4[direct_frags(TN)];
    int put[direct_frags(TN)];
#pragma unroll
    for (int i = 0; i < direct_frags(TN); ++i) {
      b4[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if (epi_has_bias<E>(g)) b4[i] = bias4<DT, true>(g, n0 + wn0 + 16 * i + 4 * g4);
      put[i] = at((wm0 ? 16 : 0) + l16, (wn0 >> 2) + 4 * i + g4);
    }
#pragma unroll
    for (int j = 0; j < 2 * TM; ++j) {
#pragma unroll
      for (int i = 0; i < direct_frags(TN); ++i) {
        float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        epi_apply4<E>(g, b4[i], v);
        *reinterpret_cast<f32x4*>(stage + put[i]) = f32x4{v[0], v[1], v[2], v[3]};
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      u32x4 own[NS];
      uint32_t one[2];
#pragma unroll
      for (int t = 0; t < NS; ++t) own[t] = *reinterpret_cast<const u32x4*>(stage + wide_lds[t]);
#pragma unroll
      for (int t = 0; t < 2; ++t) one[t] = *reinterpret_cast<const uint32_t*>(stage + edge_lds[t]);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        // (every lane takes part: the next chunk comes from the next lane; the last lane of a row needs none)
        uint32_t w[7], u[6];
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = own[t][e];
#pragma unroll
        for (int e = 0; e < 3; ++e) w[4 + e] = __builtin_amdgcn_update_dpp(0, own[t][e], 0x130, 0xf, 0xf, false);
#pragma unroll
        for (int e = 0; e < 6; ++e) {
          const uint32_t a = w[e], b = w[e + 1];
          u[e] = by1[t] ? b : a;
        }
        u32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t a = u[e], b = u[e + 2];
          v[e] = by2[t] ? b : a;
        }
        if (wide_ok[t] && wide_row[t] + 16 * j < g.M)
          __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(wide[t] + j * turn));
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
        if (edge_ok[t] && edge_row[t] + 16 * j < g.M) reinterpret_cast<uint32_t*>(edge[t] + j * turn)[0] = one[t];
    }
  });
}

// End of a tile: once every wave has left the rings, the first loads of the workgroup's NEXT tile
// are issued into them (their latency and the cold start of the pipeline hide behind this tile's
// stores), then the accumulators are written out.  16-bit outputs are staged through `stage`, an
// LDS area of its own (32 rows of the wave's sub-tile at a time, 16-byte chunk ^ ((row / 2) % chunks)
// against bank conflicts), and leave as full row segments of 16 bytes per lane.  `ring` and
// `stage` are separate restrict parameters so that the staging traffic does not wait for the
// asynchronous ring writes.
// BLOCKS (a launch cut along K): the accumulators go out as they are, f32, to rows of whole aligned 16-byte chunks.
// None of the epilogue variants is in that code: with the element-aligned accesses of an edge tile they took the
// 128 x 128 tile to 136 registers, where two workgroups no longer fit a CU (M = 16, N = K = 8192 bf16: 34 -> 40 us).
template <int DT, int TM, int TN, bool EDGE, bool TAIL, bool HAS_NEXT, bool BT, bool BLOCKS, bool STREAM>
__device__ __forceinline__ void direct_finish(const GemmArgs& g, const DirectCtx<TM, TN>& next, int nk,
                                              uint8_t* __restrict__ ring, uint8_t* __restrict__ stage,
                                              const f32x4 (&acc)[direct_frags(TN)][2 * TM], const u32x2 (&bias)[direct_frags(TN)], int m0,
                                              int n0, int wm0, int wn0) {
  using Cfg = DirectCfg<TM, TN>;
  constexpr int WTN = Cfg::WTN;
  // The lane-dependent addresses below do not change from tile to tile; lane_now() has them
  // recomputed here instead of kept in registers (and spilled) across the main loop.
  // Accumulator acc[i][j][e] of a lane: row wm0 + 16 j + lane % 16, column wn0 + 16 i + 4 (lane / 16) + e.
  const int lane = lane_now();
  const int l16 = lane & 15, g4 = lane >> 4;
  const int n_base = n0 + wn0 + 4 * g4;
  if (!BLOCKS && g.out_dt != LH_F32 && !(g.flags & LH_GEMM_ACCUMULATE_C)) {
    // The bias values (loaded by the main loop, whose last wait covered them) are pinned down here:
    // a wait for them placed after the ring loads below would wait for those loads as well.
#pragma unroll
    for (int i = 0; i < direct_frags(TN); ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) asm volatile("" ::"v"(bias[i][e]));
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave is done with the rings
    if constexpr (HAS_NEXT) direct_prologue<TM, TN, TAIL, BT>(next, nk, ring);
    constexpr int RB = WTN * 2;                // bytes of a staged row
    constexpr int chunks = RB / 16;            // 16-byte chunks per staged row
    auto at = [&](int row, int ch) { return row * RB + ((TN == 3 ? ch : ch ^ ((row >> 1) & (chunks - 1))) << 4); };
    // With a next tile loading into the rings, 32 rows at a time go through the wave's slice of
    // `stage`; the last tile of a workgroup stages its whole sub-tile in the idle rings at once.
    constexpr int JB = HAS_NEXT ? 1 : TM;
    uint8_t* cw = HAS_NEXT ? stage + next.wave * (32 * RB) : ring + next.wave * (TM * 32 * RB);
    uint16_t* outp = reinterpret_cast<uint16_t*>(g.out);
    // One variant of the bias / activation code per tile, chosen here, not per element group.
    epi_dispatch(g, [&](auto variant) {
      using E = decltype(variant);
      // The bias of fragment i's 4 columns, converted where it is used (a converted copy of all of
      // them would be 8 TN more live registers in an epilogue that has none to spare).
      auto bias_of = [&](int i) -> f32x4 {
        if constexpr (!E::kAny && !E::kBias) return f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        const int n = n_base + 16 * i;
        return (g.bias_dt == LH_F32)
                   ? bias4<DT, EDGE>(g, n)
                   : f32x4{unpack_lo<DT>(bias[i][0]), unpack_hi<DT>(bias[i][0]), unpack_lo<DT>(bias[i][1]),
                           unpack_hi<DT>(bias[i][1])};
      };
#pragma unroll
      for (int j0 = 0; j0 < TM; j0 += JB) {
#pragma unroll
        for (int jj = 0; jj < 2 * JB; ++jj)
#pragma unroll
          for (int i = 0; i < direct_frags(TN); ++i) {
            const int j = 2 * j0 + jj;           // 16-row fragment; staged row 16 jj + l16
            const u32x2 w = epi_pack4<DT, E>(g, bias_of(i), acc[i][j]);
            const int row = 16 * jj + l16;
            *reinterpret_cast<u32x2*>(cw + at(row, 2 * i + (g4 >> 1)) + 8 * (g4 & 1)) = w;
          }
        // Cfg::kStagedStores stores per lane in all; the main loop's first wait counts on it.
#pragma unroll
        for (int t = 0; t < JB * 32 * chunks / 64; ++t) {
          const int row = TN == 3 ? (64 * t + lane) / chunks : 64 / chunks * t + lane / chunks;
          const int ch = TN == 3 ? (64 * t + lane) % chunks : lane % chunks;
          u32x4 w = *reinterpret_cast<const u32x4*>(cw + at(row, ch));
          const int m = m0 + wm0 + 32 * j0 + row, n = n0 + wn0 + ch * 8;
          if constexpr (EDGE) {
            if (m < g.M && n < g.N) store8_any<STREAM>(outp + (int64_t)m * g.ldc + n, w, g.N - n);
          } else {
            u32x4* const to = reinterpret_cast<u32x4*>(outp + (int64_t)m * g.ldc + n);
            if constexpr (STREAM) __builtin_nontemporal_store(w, to);
            else *to = w;
          }
        }
      }
    });
    return;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if constexpr (HAS_NEXT) direct_prologue<TM, TN, TAIL, BT>(next, nk, ring);
  if constexpr (EDGE && !BLOCKS && TN != 3) {
    if (g.out_dt == LH_F32 && !(g.flags & LH_GEMM_ACCUMULATE_C) && !rows_of_pieces(g)) {
      direct_finish_rows<DT, TM, TN>(g, next.wave, stage, acc, m0, n0, wm0, wn0);
      return;
    }
  }
  {
    // f32 output (with or without an accumulator input), or a 16-bit output with an accumulator
    // input: the scaled f32 accumulators of a block of 32 rows x 16 NI columns go through the wave's
    // slice of `stage` so that the accumulator input is read and the result written as whole row
    // segments (4 elements per lane, 64 or 128 bytes per row) instead of pieces of 64 different
    // rows.  Order of operations as in epilogue4 (one rounding, after the sum).
    constexpr int NI = TN == 3 ? 1 : TN;       // 16-column fragments per staged block
    constexpr int NBLK = Cfg::NF / NI;         // blocks of a wave side by side
    constexpr int RB = NI * 64;                // bytes of a staged row
    constexpr int chunks = RB / 16;
    constexpr int rows_per_pass = 64 / chunks;
    uint8_t* cw = stage + next.wave * (32 * RB);
    const int ch = lane % chunks, row0 = lane / chunks;
    // The output type, the accumulator input and the bias / activation variant are fixed per tile:
    // out32 / has_c as compile-time booleans, the variant from epi_dispatch_linear (an activation
    // takes the variant that tests the flags).
    auto body = [&](auto variant, auto out32_c, auto has_c_c) {
      using E = decltype(variant);
      constexpr bool out32 = decltype(out32_c)::value, has_c = decltype(has_c_c)::value;
      // The 128 x 128 and 128 x 192 tiles request their whole accumulator input up front (8 and 12 row
      // segments per lane, all in flight at once) instead of block by block between the stores of the
      // blocks before, which the loads cannot pass (input and output may be the same buffer): one exposed
      // memory latency per tile instead of eight or twelve.  The larger tiles have no registers for that.
      constexpr bool kPreloadC = TM == 2 && TN != 2 && has_c;
      constexpr int NPASS = 32 / rows_per_pass;
      auto load_c = [&](int64_t off, int n) -> f32x4 {
        if constexpr (EDGE) {
          return load4_any<out32 ? LH_F32 : DT>(g.c, off, g.N - n);
        } else if constexpr (out32) {
          return *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(g.c) + off);
        } else {
          const u32x2 cc = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(g.c) + off);
          return f32x4{unpack_lo<DT>(cc[0]), unpack_hi<DT>(cc[0]), unpack_lo<DT>(cc[1]), unpack_hi<DT>(cc[1])};
        }
      };
      f32x4 cin[kPreloadC ? NBLK * TM * NPASS : 1];
      if constexpr (kPreloadC) {
#pragma unroll
        for (int ib = 0; ib < NBLK; ++ib)
#pragma unroll
          for (int j32 = 0; j32 < TM; ++j32)
#pragma unroll
            for (int t = 0; t < NPASS; ++t) {
              const int n = n0 + wn0 + 16 * NI * ib + 4 * ch;
              const int m = m0 + wm0 + 32 * j32 + rows_per_pass * t + row0;
              f32x4 c4 = {0.0f, 0.0f, 0.0f, 0.0f};
              if (!EDGE || (n < g.N && m < g.M)) c4 = load_c((int64_t)m * g.ldc + n, n);
              cin[(ib * TM + j32) * NPASS + t] = c4;
            }
      }
#pragma unroll
      for (int ib = 0; ib < NBLK; ++ib) {
        const int n = n0 + wn0 + 16 * NI * ib + 4 * ch;  // the lane's 4 output columns
        const bool n_ok = !EDGE || n < g.N;
        f32x4 b4 = {0.0f, 0.0f, 0.0f, 0.0f};
        if (epi_has_bias<E>(g)) b4 = bias4<DT, EDGE>(g, n);
#pragma unroll
        for (int j32 = 0; j32 < TM; ++j32) {
#pragma unroll
          for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int ii = 0; ii < NI; ++ii) {
              const f32x4& a4 = acc[NI * ib + ii][2 * j32 + jj];
              f32x4 w = a4;
              if constexpr (E::kAlpha) w = f32x4{a4[0] * g.alpha, a4[1] * g.alpha, a4[2] * g.alpha, a4[3] * g.alpha};
              const int row = 16 * jj + l16;
              *reinterpret_cast<f32x4*>(cw + row * RB + (((4 * ii + g4) ^ ((row >> 1) & (chunks - 1))) << 4)) = w;
            }
#pragma unroll
          for (int t = 0; t < 32 / rows_per_pass; ++t) {
            const int row = rows_per_pass * t + row0;
            f32x4 v = *reinterpret_cast<const f32x4*>(cw + row * RB + ((ch ^ ((row >> 1) & (chunks - 1))) << 4));
            const int m = m0 + wm0 + 32 * j32 + row;
            if (EDGE && !(n_ok && m < g.M)) continue;
            const int64_t off = (int64_t)m * g.ldc + n;
            if constexpr (has_c) {
              f32x4 c4;
              if constexpr (kPreloadC) c4 = cin[(ib * TM + j32) * NPASS + t];
              else c4 = load_c(off, n);
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] += c4[e];
            }
            if constexpr (E::kAny) {
              if (g.flags & LH_GEMM_HAS_BIAS) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += b4[e];
              }
              if (g.flags & LH_GEMM_HAS_GELU) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
              }
              if (g.flags & LH_GEMM_HAS_RELU) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = relu_nan(v[e]);
              }
            } else if constexpr (E::kBias) {
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] += b4[e];
            }
            if constexpr (EDGE && !BLOCKS) {
              store4_any<out32 ? LH_F32 : DT, STREAM>(g.out, off, v, g.N - n);
            } else if constexpr (out32) {
              f32x4* const to = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(g.out) + off);
              if constexpr (STREAM) __builtin_nontemporal_store(v, to);
              else *to = v;
            } else {
              *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(g.out) + off) =
                  u32x2{pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
            }
          }
        }
      }
    };
    if constexpr (BLOCKS) {
      body(EpiFixed<false, false, 0>{}, std::true_type{}, std::false_type{});
    } else {
      const bool out32 = g.out_dt == LH_F32;
      const bool has_c = (g.flags & LH_GEMM_ACCUMULATE_C) != 0;
      epi_dispatch_linear(g, [&](auto variant) {
        if (out32 && has_c) body(variant, std::true_type{}, std::true_type{});
        else if (out32) body(variant, std::true_type{}, std::false_type{});
        else body(variant, std::false_type{}, std::true_type{});  // a 16-bit output comes here only with an accumulator input
      });
    }
  }
}

// Where a lane's fragments are in the stages; the wave's sub-tile starts at (wm0, wn0).
template <int TM, int TN>
__device__ __forceinline__ void direct_lane_reads(DirectCtx<TM, TN>& c, int wave, int lane, int wm0, int wn0) {
  using Cfg = DirectCfg<TM, TN>;
  const int l16 = lane & 15, g4 = lane >> 4;
  c.wave = wave;
  // A fragment jj (second MFMA operand): row wm0 + 16 jj + l16, logical 16-byte chunk 4 kc + g4 of
  // the row's 8 (physical chunk: ^ ((row / 2) % 8); 4 kc only flips bit 2).
  {
    const int r = wm0 + l16;
    c.a_rd[0] = r * 128 + ((g4 ^ ((r >> 1) & 7)) << 4);
    c.a_rd[1] = c.a_rd[0] ^ 64;
  }
  // B fragment i (first MFMA operand) through the transposing read: the 16 lanes of group g4
  // address k rows 8 g4 + l16 / 4 (+4 for the second read), columns wn0 + 16 i + 4 (l16 % 4) .. +4,
  // and each receives the 4 k-values of column wn0 + 16 i + l16.
  {
    const int krow = 8 * g4 + (l16 >> 2);
    const int col = wn0 + 4 * (l16 & 3);
    c.b_chunk = col >> 3;
    c.b_swz = Cfg::b_swizzle(krow);
    c.b_off = krow * Cfg::kBRow + 8 * ((col >> 2) & 1);
  }
  // (transposed B: row wn0 + 16 i + l16 of the stage, like the A fragment)
  {
    const int r = wn0 + l16;
    c.bt_rd[0] = r * 128 + ((g4 ^ ((r >> 1) & 7)) << 4);
    c.bt_rd[1] = c.bt_rd[0] ^ 64;
  }
}

// Persistent workgroups: one (two for the 128 x 128 tile, whose LDS is 80 KiB) per CU, each
// walking the tile list with the grid as stride.  Tile ids congruent modulo 8 stay on one XCD,
// which is what xcd_remap assumes.  Launching one workgroup per tile instead costs a
// workgroup launch plus a cold prologue per tile, about a third of a K = 768 tile's time.
// SPLITK: the tile list is g.splits copies of the problem's tiles, copy sp working on its own K
// columns of A / rows of B and its own block of the (f32) output; a second kernel adds the blocks.
// For problems with few tiles and a long K (decode shapes), where the tile count cannot fill the CUs.
// BT: B is stored transposed ([N, K] with row stride ldb, the layout of a torch Linear weight); its
// panel goes through the rings like A's and no transposed copy is made.
// STREAM (large results, which are cut into 256 x 256 tiles): whole vectors are stored past the caches.  A kernel of its own:
// choosing between the two stores inside one cost smaller results 1 to 3 us of instruction fetches.
// TAIL: K is a multiple of 8 but not of 64, the last step's loads bring zeros from K on (not for the 256 x 256 tile, which
// has no registers for it).  A kernel of its own too: asking at every load cost a lone workgroup 5 % (3 x 512 x 8000).
template <int DT, int TM, int TN, bool EDGE, bool TAIL, bool SPLITK, bool BT, bool STREAM>
__device__ __forceinline__ void direct_run(const GemmArgs& g) {
  using Cfg = DirectCfg<TM, TN>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_d[];
  const int tiles1 = ((g.M + Cfg::BM - 1) / Cfg::BM) * ((g.N + Cfg::BN - 1) / Cfg::BN);
  const int ntiles = SPLITK ? tiles1 * g.splits : tiles1;
  GemmArgs g_cur = g, g_nxt = g;  // (SPLITK) the problem copy that the current / next tile belongs to
  auto select = [&](int t, GemmArgs& ga) -> int {  // -> the tile's id within its copy
    if constexpr (SPLITK) {
      const int sp = t / tiles1;
      ga.a = reinterpret_cast<const uint16_t*>(g.a) + (int64_t)sp * g.K;
      ga.b = reinterpret_cast<const uint16_t*>(g.b) + (BT ? (int64_t)sp * g.K : (int64_t)sp * g.K * g.ldb);
      ga.out = reinterpret_cast<float*>(g.out) + (int64_t)sp * g.M * g.ldc;
      ga.c = ga.out;
      return t - sp * tiles1;
    }
    return t;
  };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int WN = 4;
  const int wm0 = (wave / WN) * Cfg::WTM, wn0 = (wave % WN) * Cfg::WTN;
  const int g4 = lane >> 4;

  // Large results, one workgroup per CU: workgroups in step store their tiles in step, and the main loops in between leave
  // the memory idle.  So some start half a tile late: those that have a tile fewer than the others where that is up to half
  // of them (they have the time), half of them where all have as many and those are enough.  M = 8192, N = 50432, K = 768
  // bf16: 559 -> 540 us, with f32 results 633 -> 605.
  if constexpr (STREAM) {
    const int grid = (int)gridDim.x;
    if (ntiles > grid) {
      const int rest = ntiles % grid;
      if ((rest || ntiles >= 8 * grid) && (int)blockIdx.x >= max(rest, grid / 2))
        for (int i = min(g.K, 8192) / 40 + 2; i > 0; --i) __builtin_amdgcn_s_sleep(16);  // 16 x 64 clocks
    }
  }

  DirectCtx<TM, TN> c;
  direct_lane_reads(c, wave, lane, wm0, wn0);

  // (even: K is a multiple of 64, or the steps from K on multiply zeros)
  const int nk = TAIL ? (g.K + 63) / 64 * 2 : g.K / 32;
  c.k_end = g.K;
  int t = blockIdx.x;       // < ntiles: the grid is never larger than the tile list
  int m0, n0;
  {
    const int id = select(t, g_cur);
    direct_place<TM, TN, EDGE, BT>(SPLITK ? g_cur : g, xcd_remap(id, tiles1), c, m0, n0);
  }
  direct_prologue<TM, TN, TAIL, BT>(c, nk, smem_d);
  if constexpr (!SPLITK && TM * TN < 8)
    if (__builtin_expect(g.touch_b, 0)) direct_touch_b<BT>(g, wave, smem_d + Cfg::kRingBytes);
  // Without EDGE every lane issues all stores of a staged epilogue.
  const bool staged = !SPLITK && g.out_dt != LH_F32 && !(g.flags & LH_GEMM_ACCUMULATE_C);
  const bool counted_stores = !EDGE && staged;
  bool first = true;
  for (;;) {
    f32x4 acc[direct_frags(TN)][2 * TM];
#pragma unroll
    for (int i = 0; i < direct_frags(TN); ++i)
#pragma unroll
      for (int j = 0; j < 2 * TM; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.0f;
    u32x2 bias[direct_frags(TN)];
    const GemmArgs& ga = SPLITK ? g_cur : g;
    direct_mainloop<DT, TM, TN, EDGE, TAIL, BT, SPLITK>(ga, c, acc, smem_d, nk, counted_stores && !first, staged, n0 + wn0 + 4 * g4, bias);
    first = false;
    const int tn = t + (int)gridDim.x;
    const bool more = tn < ntiles;
    DirectCtx<TM, TN> cn = c;
    int m1 = 0, n1 = 0;
    uint8_t* const stage = smem_d + Cfg::kRingBytes;
    if (more) {
      const int idn = select(tn, g_nxt);
      direct_place<TM, TN, EDGE, BT>(SPLITK ? g_nxt : g, xcd_remap(idn, tiles1), cn, m1, n1);
      direct_finish<DT, TM, TN, EDGE, TAIL, true, BT, SPLITK, STREAM>(ga, cn, nk, smem_d, stage, acc, bias, m0, n0, wm0, wn0);
    } else {
      direct_finish<DT, TM, TN, EDGE, TAIL, false, BT, SPLITK, STREAM>(ga, cn, nk, smem_d, stage, acc, bias, m0, n0, wm0, wn0);
    }
    if (!more) break;
    if constexpr (SPLITK) g_cur = g_nxt;
    if constexpr (TN == 2) {
      // The next tile's load offsets are computed again rather than carried through the epilogue in
      // registers: the 256-wide tiles spilled them (16 bytes per lane), and a kernel that touches
      // scratch memory at all pays for it at every dispatch (4096^3 100.5 -> 99.4 us without).
      const int idn = select(tn, g_cur);
      direct_place<TM, TN, EDGE, BT>(SPLITK ? g_cur : g, xcd_remap(idn, tiles1), c, m0, n0);
    } else {
      c = cn;
      m0 = m1;
      n0 = n1;
    }
    t = tn;
  }
}

template <int DT, int TM, int TN, bool EDGE, bool SPLITK = false, bool BT = false, bool STREAM = false>
__global__ void __launch_bounds__(512) gemm16_direct(GemmArgs g) {
  direct_run<DT, TM, TN, EDGE, false, SPLITK, BT, STREAM>(g);
}
template <int DT, int TM, int TN, bool BT>
__global__ void __launch_bounds__(512) gemm16_direct_tail(GemmArgs g) {
  direct_run<DT, TM, TN, true, true, false, BT, false>(g);
}

template <int DT, int TM, int TN, bool EDGE, bool BT = false, bool STREAM = false, bool TAIL = false>
static int launch_direct_edge(const GemmArgs& g, hipStream_t s) {
  using Cfg = DirectCfg<TM, TN>;
  auto kern = gemm16_direct<DT, TM, TN, EDGE, false, BT, STREAM>;
  if constexpr (TAIL) kern = gemm16_direct_tail<DT, TM, TN, BT>;
  constexpr size_t lds = Cfg::kLdsBytes;
  static bool configured = false;
  if (!configured && !planning()) {
    LH_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds));
    configured = true;
  }
  const int ntiles = ((g.M + Cfg::BM - 1) / Cfg::BM) * ((g.N + Cfg::BN - 1) / Cfg::BN);
  const int resident = num_cus() * (2 * lds <= 160 * 1024 ? 2 : 1);
  GemmArgs ga = g;
  const int grid = ntiles < resident ? ntiles : resident;
  const int64_t rows = BT ? g.N : g.K;
  ga.touch_b = g.K >= kTouchFrom && rows * (((BT ? g.K : g.N) + 63) / 64) <= 128 * grid && rows * g.ldb < (1ll << 30);
  LH_LAUNCH(kern, dim3(grid), dim3(512), lds, s, ga);
  return check_launch("gemm16_direct");
}

template <int DT, int TM, int TN>
int launch_direct(const GemmArgs& g, hipStream_t s) {
  using Cfg = DirectCfg<TM, TN>;
  const bool whole = whole_tiles(g, Cfg::BM, Cfg::BN);
  if constexpr (TM * TN < 8)
    if (g.K % 64 != 0)
      return (g.flags & LH_GEMM_TRANSPOSE_B) ? launch_direct_edge<DT, TM, TN, true, true, false, true>(g, s)
                                             : launch_direct_edge<DT, TM, TN, true, false, false, true>(g, s);
  if constexpr (TM * TN == 8)
    if (large_result(g)) return launch_direct_large<DT>(g, whole, s);
  if (g.flags & LH_GEMM_TRANSPOSE_B)
    return whole ? launch_direct_edge<DT, TM, TN, false, true>(g, s) : launch_direct_edge<DT, TM, TN, true, true>(g, s);
  return whole ? launch_direct_edge<DT, TM, TN, false>(g, s) : launch_direct_edge<DT, TM, TN, true>(g, s);
}

#if LH_GEMM16_LARGE
template <int DT>
int launch_direct_large(const GemmArgs& g, bool whole, hipStream_t s) {
  if (g.flags & LH_GEMM_TRANSPOSE_B)
    return whole ? launch_direct_edge<DT, 4, 2, false, true, true>(g, s) : launch_direct_edge<DT, 4, 2, true, true, true>(g, s);
  return whole ? launch_direct_edge<DT, 4, 2, false, false, true>(g, s) : launch_direct_edge<DT, 4, 2, true, false, true>(g, s);
}
#endif

#if LH_GEMM16_DEEP || LH_GEMM16_TM == 0
// ---- one workgroup per CU ---------------------------------------------------------------------
// Where no CU gets a second workgroup nobody covers the latency of its operands, but all of the CU's LDS is its own.  Both rings
// hold four stages of 64 k (128 x 128 and 128 x 192 tiles; 128 x 256 and 256 x 128: three), so that a stage is requested three (two) pairs of
// steps before it is read, through one barrier per pair; what one of them takes, 0.45 us at 128 x 128, is less than a line's way out
// of memory.  One tile per workgroup: the output is staged in the idle rings.
// The price: 128 KiB of a CU's LDS at 128 x 128 (two stages: 80), 144 to 160 at the others, so that products on two streams no longer share
// CUs.  Two of one size, each on a stream of its own, us per pair with two stages and with four: 2048^3 32.5 -> 35.8, 8192 x 768 x 768
// 19.9 -> 23.0, 1000 x 4096 x 1000 19.8 -> 22.7 (tiles for more than half of the CUs); 1536 x 1536 x 1024 15.0 -> 13.8, 2048 x 1024 x 1024
// 14.2 -> 11.6 (for less).
// bf16, with two stages (and two barriers) and with four, operands in the caches / in memory: 2048^3 23.5 -> 20.5 / 28.3 -> 22.4 us,
// on a transposed B 22.8 -> 18.8 / 30.9 -> 21.7; 512 x 8192 x 2048 21.9 -> 19.3 / 28.2 -> 22.3; 2048 x 768 x 768 with a residual 11.3 -> 9.7 /
// 16.6 -> 13.6.
template <int TM, int TN>
struct DeepCfg {
  using Cfg = DirectCfg<TM, TN>;
  static constexpr int kABytes = Cfg::kABytes, kBBytes = 2 * Cfg::kBBytes;        // of a stage of 64 k
  static constexpr int kStages = 160 * 1024 / (kABytes + kBBytes) < 4 ? 160 * 1024 / (kABytes + kBBytes) : 4;
  static constexpr int kBBase = kStages * kABytes;
  static constexpr int kLdsBytes = kStages * (kABytes + kBBytes);                 // (the output is staged in the rings)
  static constexpr int kLoads = TM + Cfg::NF;                                     // of a lane per stage
};
template <int TM, int TN, bool BT, bool TAIL>
__device__ __forceinline__ void deep_load(const DirectCtx<TM, TN>& c, int p, uint8_t* __restrict__ abuf, uint8_t* __restrict__ bbuf) {
  direct_load_a<TM, TN, TAIL>(c, p, abuf);
  if constexpr (BT || TN == 3) {
    direct_load_b<TM, TN, BT, TAIL>(c, p, bbuf);
  } else {
    direct_load_b<TM, TN, false, TAIL>(c, 2 * p, bbuf);
    direct_load_b<TM, TN, false, TAIL>(c, 2 * p + 1, bbuf + DirectCfg<TM, TN>::kBBytes);
  }
}
// Pair p of steps (direct_step_pair_1b), of which a successor is read next: NEWER stages behind that have been requested and may
// be on their way.  LOAD: stage p + kStages goes where p was.
template <int DT, int TM, int TN, bool TAIL, bool BT, int NEWER, bool LOAD>
__device__ __forceinline__ void deep_step_pair(const DirectCtx<TM, TN>& c, f32x4 (&acc)[direct_frags(TN)][2 * TM], DirectFrags<TM, TN>& f,
                                               const uint8_t* __restrict__ a_cur, const uint8_t* __restrict__ a_nxt,
                                               const uint8_t* __restrict__ b_cur, const uint8_t* __restrict__ b_nxt,
                                               uint8_t* __restrict__ a_refill, uint8_t* __restrict__ b_refill, int p) {
  using Deep = DeepCfg<TM, TN>;
  const uint8_t* const b1 = BT ? b_cur : b_cur + DirectCfg<TM, TN>::kBBytes;
  direct_phase_lo<DT>(c, acc, f, a_cur, 0);
  direct_phase_hi<DT, TM, TN, BT>(c, acc, f, a_cur, b1, 1);
  direct_phase_lo<DT>(c, acc, f, a_cur, 1);
  direct_wait_barrier<NEWER * Deep::kLoads>();
  if constexpr (LOAD) deep_load<TM, TN, BT, TAIL>(c, p + Deep::kStages, a_refill, b_refill);
  direct_phase_hi<DT, TM, TN, BT>(c, acc, f, a_nxt, b_nxt, 0);
}

// SPLITK: the grid is g.splits copies of the tiles, each on its own piece of K and f32 block of the output (direct_run).
template <int DT, int TM, int TN, bool EDGE, bool TAIL, bool BT, bool SPLITK = false>
__global__ void __launch_bounds__(512) gemm16_deep(GemmArgs g) {
  using Cfg = DirectCfg<TM, TN>;
  using Deep = DeepCfg<TM, TN>;
  constexpr int S = Deep::kStages;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_d[];
  const int tiles = ((g.M + Cfg::BM - 1) / Cfg::BM) * ((g.N + Cfg::BN - 1) / Cfg::BN);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm0 = (wave / 4) * Cfg::WTM, wn0 = (wave % 4) * Cfg::WTN;
  DirectCtx<TM, TN> c;
  direct_lane_reads(c, wave, lane, wm0, wn0);
  c.k_end = g.K;
  int m0, n0;
  int id = blockIdx.x;
  if constexpr (SPLITK) {
    const int sp = __builtin_amdgcn_readfirstlane(id / tiles);
    id -= sp * tiles;
    g.a = reinterpret_cast<const uint16_t*>(g.a) + (int64_t)sp * g.K;
    g.b = reinterpret_cast<const uint16_t*>(g.b) + (int64_t)sp * g.K * (BT ? 1 : g.ldb);
    g.out = reinterpret_cast<float*>(g.out) + (int64_t)sp * g.M * g.ldc;
  }
  direct_place<TM, TN, EDGE, BT>(g, xcd_remap(id, tiles), c, m0, n0);
  const int pairs = TAIL ? (g.K + 63) / 64 : g.K / 64;
  auto a_stage = [&](int slot) { return smem_d + slot * Deep::kABytes; };
  auto b_stage = [&](int slot) { return smem_d + Deep::kBBase + slot * Deep::kBBytes; };
#pragma unroll
  for (int p = 0; p < S; ++p)
    if (p < pairs) deep_load<TM, TN, BT, TAIL>(c, p, a_stage(p), b_stage(p));

  f32x4 acc[Cfg::NF][2 * TM];
#pragma unroll
  for (int i = 0; i < Cfg::NF; ++i)
#pragma unroll
    for (int j = 0; j < 2 * TM; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // (the first stage; those behind it may be on their way)
  if (pairs >= S) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 1) * Deep::kLoads) : "memory");
  else if (S > 3 && pairs == 3) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * Deep::kLoads) : "memory");
  else if (pairs == 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(Deep::kLoads) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  DirectFrags<TM, TN> f;
  direct_read_a<TM, TN, 0>(c, a_stage(0), 0, f.a[0]);
#pragma unroll
  for (int i = 0; i < Cfg::NF; ++i) f.b[i] = direct_read_b<TM, TN, BT>(c, b_stage(0), 0, i);
  int p = 0, slot = 0;
  auto pair = [&](auto newer, auto load) {
    const int next = slot + 1 == S ? 0 : slot + 1;
    deep_step_pair<DT, TM, TN, TAIL, BT, decltype(newer)::value, decltype(load)::value>(
        c, acc, f, a_stage(slot), a_stage(next), b_stage(slot), b_stage(next), a_stage(slot), b_stage(slot), p);
    ++p;
    slot = next;
  };
  while (p + S < pairs) pair(std::integral_constant<int, S - 2>{}, std::true_type{});
  if (p + S - 1 < pairs) pair(std::integral_constant<int, S - 2>{}, std::false_type{});
  if (S > 3 && p + S - 2 < pairs) pair(std::integral_constant<int, S - 3>{}, std::false_type{});
  if (p + 1 < pairs) pair(std::integral_constant<int, 0>{}, std::false_type{});
  const bool staged = !SPLITK && g.out_dt != LH_F32 && !(g.flags & LH_GEMM_ACCUMULATE_C);
  u32x2 bias[Cfg::NF];
  if (staged) direct_load_bias<TN, EDGE>(g, n0 + wn0 + 4 * (lane >> 4), bias);
  direct_phase_lo<DT>(c, acc, f, a_stage(slot), 0);
  direct_phase_hi<DT, TM, TN, BT>(c, acc, f, a_stage(slot), b_stage(slot) + (BT ? 0 : Cfg::kBBytes), 1);
  direct_phase_lo<DT>(c, acc, f, a_stage(slot), 1);
  direct_phase_hi<DT, TM, TN, BT, false>(c, acc, f, a_stage(slot), b_stage(slot), 0);
  direct_finish<DT, TM, TN, EDGE, TAIL, false, BT, SPLITK, false>(g, c, 2 * pairs, smem_d, smem_d, acc, bias, m0, n0, wm0, wn0);
}

#if LH_GEMM16_DEEP
template <int DT, int TM, int TN>
int launch_deep(const GemmArgs& g, hipStream_t s) {
  using Cfg = DirectCfg<TM, TN>;
  using Deep = DeepCfg<TM, TN>;
  static_assert(Deep::kStages == 3 || Deep::kStages == 4, "the kernel's last pairs");
  constexpr bool tail = TN != 3;  // (192 columns take whole stages only)
  static constexpr decltype(&gemm16_deep<DT, TM, TN, true, false, false>) kernels[2][3] = {
      {gemm16_deep<DT, TM, TN, false, false, false>, gemm16_deep<DT, TM, TN, true, false, false>, gemm16_deep<DT, TM, TN, true, tail, false>},
      {gemm16_deep<DT, TM, TN, false, false, true>, gemm16_deep<DT, TM, TN, true, false, true>, gemm16_deep<DT, TM, TN, true, tail, true>}};
  static bool configured = false;
  if (!configured && !planning()) {
    for (auto& layout : kernels)
      for (auto k : layout)
        LH_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, Deep::kLdsBytes));
    configured = true;
  }
  const bool whole = whole_tiles(g, Cfg::BM, Cfg::BN);
  auto kern = kernels[(g.flags & LH_GEMM_TRANSPOSE_B) ? 1 : 0][g.K % 64 != 0 ? 2 : whole ? 0 : 1];
  LH_LAUNCH(kern, dim3((unsigned)(((g.M + Cfg::BM - 1) / Cfg::BM) * ((g.N + Cfg::BN - 1) / Cfg::BN))), dim3(512), Deep::kLdsBytes, s, g);
  return check_launch("gemm16_deep");
}
template int launch_deep<LH_GEMM16_DT, LH_GEMM16_TM, LH_GEMM16_TN>(const GemmArgs&, hipStream_t);
#endif
#endif

#if LH_GEMM16_ODD
// ---- B in rows of any length ------------------------------------------------------------------
// The 128 x 128 tile on an n-contiguous B whose rows are no whole aligned 16-byte chunks (N or the row stride odd, a pointer
// off 16 bytes), which the loads into LDS cannot take.  B comes through registers instead, 16 bytes a load at element
// alignment, and is stored into the swizzled rows that direct_read_b expects; everything else is the kernel above with one
// barrier per 64 k.  Pair p of steps stores what pair p - 1 requested, the 64 rows of pair p + 1, into the half of the ring that
// pair p - 1 has left, and requests the rows of pair p + 2 at once: they have a whole pair to arrive (requested behind the barrier,
// a quarter later, 600 x 4001 x 1600 took 29.7 us instead of 22.3).  What bounds it is the latency of the operands; against it
// stands a copy of B in a launch of its own.  bf16, on a copy and as it is: 1000 x 4097 x 1000 25.9 and 21.1 us, B in memory
// 28.3 and 23.8; 100 x 50257 x 768, f32 result, B in memory 51.6 and 29.5.
struct OddRows {
  const uint8_t* base;  // the tile's first column of B (uniform)
  int src;              // the lane's byte offset at k = 0 of the first of its two rows of 64, the other is 32 rows on
  int row;              // its row in them
  int col;              // its first column of the tile, past the end of B where `over` says how far
  int over;             // elements of the chunk that lie past the end of their row (0 .. 7)
};
// Rows 64 p .. of B.  LAST: those that K ends in.  Rows from K on are the last one; its chunk that crosses its end, which may be
// that of B's memory, is read from its last 8 elements.
template <bool LAST>
__device__ __forceinline__ void odd_request(const GemmArgs& g, const OddRows& o, int p, u32x4 (&r)[2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (LAST) {
      const int k = min(64 * p + 32 * i + o.row, g.K - 1);
      const int col = k == g.K - 1 ? o.col - o.over : o.col;
      r[i] = *reinterpret_cast<const u32x4_any*>(o.base + ((int64_t)k * g.ldb + col) * 2);
    } else {
      r[i] = *reinterpret_cast<const u32x4_any*>(o.base + (int64_t)(64 * p + 32 * i) * g.ldb * 2 + (uint32_t)o.src);
    }
  }
}
// ... into the pair's two stages at `to`.
template <bool LAST>
__device__ __forceinline__ void odd_store(const GemmArgs& g, const OddRows& o, int p, u32x4 (&r)[2], int wave, uint8_t* __restrict__ to) {
  using Cfg = DirectCfg<2, 1>;
  const int lane = lane_now();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (LAST) {
      const int k = 64 * p + 32 * i + o.row;
      if (k >= g.K) {
        r[i] = u32x4{0u, 0u, 0u, 0u};
      } else if (k == g.K - 1 && o.over) {
        // the chunk moved down by `over` elements
        uint64_t lo = (uint64_t)r[i][1] << 32 | r[i][0], hi = (uint64_t)r[i][3] << 32 | r[i][2];
        if (o.over >= 4) {
          lo = hi;
          hi = 0;
        }
        const int bits = 16 * (o.over & 3);
        if (bits) lo = lo >> bits | hi << (64 - bits);
        hi >>= bits;
        r[i] = u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
      }
    }
    *reinterpret_cast<u32x4*>(to + i * Cfg::kBBytes + wave * 1024 + lane * 16) = r[i];
  }
}
// A pair of steps (direct_step_pair_1b).  REQUEST: pair p + 2 exists, LAST_REQUEST: and K ends in it; LAST_STORE: K ends in p + 1.
template <int DT, bool TAIL, bool REQUEST, bool LAST_REQUEST, bool LAST_STORE>
__device__ __forceinline__ void odd_step_pair(const GemmArgs& g, const DirectCtx<2, 1>& c, const OddRows& o, u32x4 (&rows)[2],
                                              f32x4 (&acc)[2][4], DirectFrags<2, 1>& f, const uint8_t* __restrict__ a_cur,
                                              const uint8_t* __restrict__ a_nxt, const uint8_t* __restrict__ b1,
                                              const uint8_t* __restrict__ b2, uint8_t* __restrict__ a_refill,
                                              uint8_t* __restrict__ b_next, int p) {
  direct_phase_lo<DT>(c, acc, f, a_cur, 0);
  direct_phase_hi<DT, 2, 1, false>(c, acc, f, a_cur, b1, 1);
  odd_store<LAST_STORE>(g, o, p + 1, rows, c.wave, b_next);
  if constexpr (REQUEST) odd_request<LAST_REQUEST>(g, o, p + 2, rows);
  direct_phase_lo<DT>(c, acc, f, a_cur, 1);
  direct_wait_barrier<REQUEST ? 2 : 0>();  // (the two loads of B are the latest)
  if constexpr (REQUEST) direct_load_a<2, 1, TAIL>(c, p + 2, a_refill);
  direct_phase_hi<DT, 2, 1, false>(c, acc, f, a_nxt, b2, 0);
}

template <int DT, bool TAIL>
__global__ void __launch_bounds__(512, 4) gemm16_odd_rows(GemmArgs g) {
  using Cfg = DirectCfg<2, 1>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_d[];
  const int tiles = ((g.M + 127) / 128) * ((g.N + 127) / 128);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm0 = (wave / 4) * Cfg::WTM, wn0 = (wave % 4) * Cfg::WTN;
  DirectCtx<2, 1> c;
  direct_lane_reads(c, wave, lane, wm0, wn0);
  c.k_end = g.K;
  int m0, n0;
  direct_place<2, 1, true>(g, xcd_remap(blockIdx.x, tiles), c, m0, n0);
  OddRows o;
  {
    const int chunk = lane % Cfg::kBChunks;
    o.row = wave * Cfg::kBRowsPerLoad + lane / Cfg::kBChunks;
    // (as direct_place has it; chunks past the end of the row are its last one)
    const int bc = chunk ^ (4 * (o.row & 3)) ^ (2 * ((o.row >> 3) & 1));
    o.col = min(bc * 8, (g.N - 1) / 8 * 8 - n0);
    o.over = max(n0 + o.col + 8 - g.N, 0);
    o.base = reinterpret_cast<const uint8_t*>(reinterpret_cast<const uint16_t*>(g.b) + n0);
    o.src = (o.row * (int)g.ldb + o.col) * 2;
  }
  const int pairs = (g.K + 63) / 64, nk = 2 * pairs;
  uint8_t* const abuf = smem_d;
  uint8_t* const bbuf = smem_d + Cfg::kBBase;
  auto a_stage = [&](int p) { return abuf + (p & 1) * Cfg::kABytes; };
  auto b_pair = [&](int p) { return bbuf + (p & 1) * 2 * Cfg::kBBytes; };

  u32x4 rows[2];
  if (pairs == 1) odd_request<true>(g, o, 0, rows);
  else odd_request<false>(g, o, 0, rows);
  direct_load_a<2, 1, TAIL>(c, 0, abuf);
  if (pairs == 1) odd_store<true>(g, o, 0, rows, wave, bbuf);
  else odd_store<false>(g, o, 0, rows, wave, bbuf);
  if (pairs > 1) {
    if (pairs == 2) odd_request<true>(g, o, 1, rows);
    else odd_request<false>(g, o, 1, rows);
    direct_load_a<2, 1, TAIL>(c, 1, abuf + Cfg::kABytes);
  }

  f32x4 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  DirectFrags<2, 1> f;
  direct_read_a<2, 1, 0>(c, abuf, 0, f.a[0]);
#pragma unroll
  for (int i = 0; i < 2; ++i) f.b[i] = direct_read_b<2, 1, false>(c, bbuf, 0, i);
  int p = 0;
  auto pair = [&](auto request, auto last_request, auto last_store) {
    odd_step_pair<DT, TAIL, decltype(request)::value, decltype(last_request)::value, decltype(last_store)::value>(
        g, c, o, rows, acc, f, a_stage(p), a_stage(p + 1), b_pair(p) + Cfg::kBBytes, b_pair(p + 1), a_stage(p), b_pair(p + 1), p);
    ++p;
  };
  while (p + 3 < pairs) pair(std::true_type{}, std::false_type{}, std::false_type{});
  if (p + 2 < pairs) pair(std::true_type{}, std::true_type{}, std::false_type{});
  if (p + 1 < pairs) pair(std::false_type{}, std::false_type{}, std::true_type{});
  const bool staged = g.out_dt != LH_F32 && !(g.flags & LH_GEMM_ACCUMULATE_C);
  u32x2 bias[2];
  if (staged) direct_load_bias<1, true>(g, n0 + wn0 + 4 * (lane >> 4), bias);
  direct_phase_lo<DT>(c, acc, f, a_stage(p), 0);
  direct_phase_hi<DT, 2, 1, false>(c, acc, f, a_stage(p), b_pair(p) + Cfg::kBBytes, 1);
  direct_phase_lo<DT>(c, acc, f, a_stage(p), 1);
  direct_phase_hi<DT, 2, 1, false, false>(c, acc, f, a_stage(p), b_pair(p), 0);
  direct_finish<DT, 2, 1, true, TAIL, false, false, false, false>(g, c, nk, smem_d, smem_d + Cfg::kRingBytes, acc, bias, m0, n0, wm0, wn0);
}

template <int DT>
int launch_odd_rows(const GemmArgs& g, hipStream_t s) {
  using Cfg = DirectCfg<2, 1>;
  auto kern = g.K % 64 != 0 ? gemm16_odd_rows<DT, true> : gemm16_odd_rows<DT, false>;
  static bool configured = false;
  if (!configured && !planning()) {
    for (auto k : {gemm16_odd_rows<DT, true>, gemm16_odd_rows<DT, false>})
      LH_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::kLdsBytes));
    configured = true;
  }
  const int64_t tiles = (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128);
  LH_LAUNCH(kern, dim3((unsigned)tiles), dim3(512), Cfg::kLdsBytes, s, g);
  return check_launch("gemm16_odd_rows");
}
template int launch_odd_rows<LH_GEMM16_DT>(const GemmArgs&, hipStream_t);
#endif

// One instantiation of the kernel with its K cut (EDGE: tiles past the end of the matrix).
template <int DT, bool EDGE, bool BT>
static int launch_splitk_edge(const GemmArgs& g, hipStream_t s) {
  using Cfg = DirectCfg<2, 1>;
  auto kern = gemm16_direct<DT, 2, 1, EDGE, true, BT>;
  static bool configured = false;
#if LH_GEMM16_TM == 0
  // No CU gets a second workgroup: deeper rings.  bf16, operands in the caches / in memory: 1024 x 1024 x 8192 29.3 -> 27.5 / 35.3 -> 29.0 us,
  // 128 x 4096 x 4096 18.5 -> 15.9 / 21.3 -> 18.6, 2048 x 768 x 3072 with a residual 24.3 -> 22.0 / 30.3 -> 25.3.
  using Deep = DeepCfg<2, 1>;
  auto deep = gemm16_deep<DT, 2, 1, EDGE, false, BT, true>;
  if (!configured && !planning())
    LH_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(deep), hipFuncAttributeMaxDynamicSharedMemorySize, Deep::kLdsBytes));
#endif
  if (!configured && !planning()) {
    LH_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)Cfg::kLdsBytes));
    configured = true;
  }
  const int64_t total = (int64_t)((g.M + Cfg::BM - 1) / Cfg::BM) * ((g.N + Cfg::BN - 1) / Cfg::BN) * g.splits;
  const int64_t resident = 2 * (int64_t)num_cus();
#if LH_GEMM16_TM == 0
  if (2 * total <= resident) {
    LH_LAUNCH(deep, dim3((unsigned)total), dim3(512), Deep::kLdsBytes, s, g);
    return check_launch("gemm16_deep (split K)");
  }
#endif
  LH_LAUNCH(kern, dim3((unsigned)(total < resident ? total : resident)), dim3(512), Cfg::kLdsBytes, s, g);
  return check_launch("gemm16_direct (split K)");
}

template <int DT>
int launch_direct_splitk(const GemmArgs& g, hipStream_t s) {
  using Cfg = DirectCfg<2, 1>;
  const bool edge = g.M % Cfg::BM != 0 || g.N % Cfg::BN != 0;
  if (g.flags & LH_GEMM_TRANSPOSE_B)
    return edge ? launch_splitk_edge<DT, true, true>(g, s) : launch_splitk_edge<DT, false, true>(g, s);
  return edge ? launch_splitk_edge<DT, true, false>(g, s) : launch_splitk_edge<DT, false, false>(g, s);
}

#if LH_GEMM16_ODD || LH_GEMM16_DEEP
#elif LH_GEMM16_TM == 0
template int launch_direct_splitk<LH_GEMM16_DT>(const GemmArgs&, hipStream_t);
#elif LH_GEMM16_LARGE
template int launch_direct_large<LH_GEMM16_DT>(const GemmArgs&, bool, hipStream_t);
#else
template int launch_direct<LH_GEMM16_DT, LH_GEMM16_TM, LH_GEMM16_TN>(const GemmArgs&, hipStream_t);
#endif

}  // namespace lh
