// Fused attention forward for problems with few query rows: 16-bit tensors, head dimension 64 (algorithm and
// rounding points as in attention.hip: ReplaceWithFusedAttentionOp, lighthouse/dialects/transform/transform_ext/ops/
// replace_with_fused_attention.py:332-455).
//
// What bounds such a problem on the 128-row kernel is the chain of key tiles that a few dozen workgroups walk behind
// barriers while the other CUs idle.  Here a workgroup owns 16 or 32 query rows and its 8 waves share out the keys:
// a wave takes a contiguous share of the 32-key steps on its own, without a barrier, the next step's K and V
// requested ahead in registers.  K is k-contiguous and goes straight into the MFMA's operand layout; V goes through
// 4.5 KiB of LDS that belong to the wave and is read back with the transposing LDS read.  S^T = K Q^T leaves a lane
// with keys 4 g .. 4 g + 3 of both 16-key halves of one query, which, in that key order, is the second operand of
// O^T = V^T P^T.  The waves' partial outputs are brought to the common maximum and added through LDS, in wave order.
//
// The scores are scaled in f32, Q stays as stored: one rounding less than the large kernels take.
#include "attention.h"

namespace lh {

typedef short attn_small_s16x4 __attribute__((ext_vector_type(4)));

constexpr int kSmallWaves = 8;
constexpr int kSmallKeys = 32;                                   // keys per step
constexpr int kSmallVRow = 128 + 16;                             // bytes of a V row in LDS (one chunk of padding)
constexpr int kSmallVBytes = kSmallKeys * kSmallVRow;            // per wave
constexpr int kSmallLdsBytes = kSmallWaves * kSmallVBytes;       // (the sums of one query tile, 4 KiB per wave, fit)

template <int DT>
__device__ __forceinline__ f32x4 attn_small_mma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (DT == LH_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <int DT, int QF>
__global__ void __launch_bounds__(kSmallWaves * 64) attention16_small_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[kSmallLdsBytes];
  __shared__ float2 stats[kSmallWaves][QF][16];  // (maximum, row sum) of a wave's share
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The workgroups of one XCD (ids congruent modulo 8) take a contiguous range of (head, query tile): a head's K
  // and V are read by one XCD's L2.  Causal: a head's longest query tile first.
  const int nqb = (a.T + 16 * QF - 1) / (16 * QF), total = nqb * a.Z * a.H;
  const int per_xcd = (total + 7) / 8;
  const int id = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (blockIdx.x / 8 >= per_xcd || id >= total) return;
  const int bh = id / nqb, z = bh / a.H, h = bh % a.H;
  const int q0 = (a.causal ? nqb - 1 - id % nqb : id % nqb) * 16 * QF;
  const uint16_t* Q = reinterpret_cast<const uint16_t*>(a.q) + (int64_t)z * a.sq.z + (int64_t)h * a.sq.h;
  const uint16_t* K = reinterpret_cast<const uint16_t*>(a.k) + (int64_t)z * a.sk.z + (int64_t)h * a.sk.h;
  const uint16_t* V = reinterpret_cast<const uint16_t*>(a.v) + (int64_t)z * a.sv.z + (int64_t)h * a.sv.h;
  uint16_t* O = reinterpret_cast<uint16_t*>(a.out) + (int64_t)z * a.so.z + (int64_t)h * a.so.h;

  u32x4 qf[QF][2];
#pragma unroll
  for (int f = 0; f < QF; ++f)
#pragma unroll
    for (int c = 0; c < 2; ++c)
      qf[f][c] = *reinterpret_cast<const u32x4*>(Q + (int64_t)min(q0 + 16 * f + l16, a.T - 1) * a.sq.t + 32 * c + 8 * g4);

  f32x4 acc[QF][4];
  float m_run[QF], l_run[QF];
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    m_run[f] = -INFINITY;
    l_run[f] = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[f][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }

  const int kv_end = a.causal ? min(a.T, q0 + 16 * QF) : a.T;
  const int steps = (kv_end + kSmallKeys - 1) / kSmallKeys;
  const int begin = (int)((int64_t)steps * wave / kSmallWaves), end = (int)((int64_t)steps * (wave + 1) / kSmallWaves);
  u32x4 kr[2][2], vr[4];
  auto request = [&](int step) {  // rows past the end are the last row's
    const int j0 = step * kSmallKeys;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        kr[i][c] = *reinterpret_cast<const u32x4*>(K + (int64_t)min(j0 + 16 * i + l16, a.T - 1) * a.sk.t + 32 * c + 8 * g4);
#pragma unroll
    for (int p = 0; p < 4; ++p)
      vr[p] = *reinterpret_cast<const u32x4*>(V + (int64_t)min(j0 + 8 * p + (lane >> 3), a.T - 1) * a.sv.t + 8 * (lane & 7));
  };
  uint8_t* const v_lds = lds + wave * kSmallVBytes;
  if (begin < end) request(begin);
#pragma unroll 1
  for (int step = begin; step < end; ++step) {
    const int j0 = step * kSmallKeys;
    f32x4 s[QF][2];
#pragma unroll
    for (int f = 0; f < QF; ++f)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        s[f][i] = attn_small_mma<DT>(kr[i][0], qf[f][0], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
        s[f][i] = attn_small_mma<DT>(kr[i][1], qf[f][1], s[f][i]);
      }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      // (a row past the end counts as zero: its P is zero, but its values may be no numbers)
      if (j0 + 8 * p + (lane >> 3) >= a.T) vr[p] = u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(v_lds + (8 * p + (lane >> 3)) * kSmallVRow + 16 * (lane & 7)) = vr[p];
    }
    if (step + 1 < end) request(step + 1);
    u32x4 pf[QF];
#pragma unroll
    for (int f = 0; f < QF; ++f) {
      // s[f][i][r] = S[q0 + 16 f + l16][j0 + 16 i + 4 g4 + r], unscaled
      if (j0 + kSmallKeys > a.T || (a.causal && j0 + kSmallKeys - 1 > q0 + 16 * f)) {
        const int last = a.causal ? min(q0 + 16 * f + l16, a.T - 1) : a.T - 1;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (j0 + 16 * i + 4 * g4 + r > last) s[f][i][r] = -INFINITY;
      }
      float mx = fmaxf(s[f][0][0], s[f][1][0]);
#pragma unroll
      for (int r = 1; r < 4; ++r) mx = fmaxf(fmaxf(mx, s[f][0][r]), s[f][1][r]);
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float m_new = fmaxf(m_run[f], mx);
      const float m_safe = m_new == -INFINITY ? 0.0f : m_new;  // (nothing visible yet)
      const float alpha = __builtin_amdgcn_exp2f((m_run[f] - m_safe) * a.scale_log2e);
      m_run[f] = m_new;
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[f][i][r] = __builtin_amdgcn_exp2f((s[f][i][r] - m_safe) * a.scale_log2e);
          sum += s[f][i][r];
        }
      l_run[f] = l_run[f] * alpha + sum;
      pf[f] = u32x4{pack2<DT>(s[f][0][0], s[f][0][1]), pack2<DT>(s[f][0][2], s[f][0][3]),
                    pack2<DT>(s[f][1][0], s[f][1][1]), pack2<DT>(s[f][1][2], s[f][1][3])};
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[f][j] *= alpha;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // group g4: keys 4 g4 + l16 / 4 of either half, columns 16 j + 4 (l16 % 4) .. +4
      uint8_t* p0 = v_lds + (4 * g4 + (l16 >> 2)) * kSmallVRow + 32 * j + 8 * (l16 & 3);
      const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                     (__attribute__((address_space(3))) attn_small_s16x4*)p0));
      const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                     (__attribute__((address_space(3))) attn_small_s16x4*)(p0 + 16 * kSmallVRow)));
      const u32x4 vf = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
      for (int f = 0; f < QF; ++f) acc[f][j] = attn_small_mma<DT>(vf, pf[f], acc[f][j]);
    }
  }

  // acc[f][j][r] = O[q0 + 16 f + l16][16 j + 4 g4 + r], of this wave's keys and relative to its maximum.
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    l_run[f] += __shfl_xor(l_run[f], 16);
    l_run[f] += __shfl_xor(l_run[f], 32);
    if (g4 == 0) stats[wave][f][l16] = make_float2(m_run[f], l_run[f]);
  }
  f32x4* const sums = reinterpret_cast<f32x4*>(lds);
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    __syncthreads();  // (the statistics are there; V, or the tile before, has been read)
    float m_all = -INFINITY, l_all = 0.0f;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) m_all = fmaxf(m_all, stats[w][f][l16].x);
    const float m_safe = m_all == -INFINITY ? 0.0f : m_all;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) {
      const float2 st = stats[w][f][l16];
      l_all += st.y * __builtin_amdgcn_exp2f((st.x - m_safe) * a.scale_log2e);
    }
    const float own = __builtin_amdgcn_exp2f((m_run[f] - m_safe) * a.scale_log2e);
#pragma unroll
    for (int j = 0; j < 4; ++j) sums[(wave * 4 + j) * 64 + lane] = acc[f][j] * own;
    __syncthreads();
    if (tid < 256) {  // fragment wave (< 4) of the tile, in this lane's position
      f32x4 v = sums[tid];
#pragma unroll
      for (int w = 1; w < kSmallWaves; ++w) v += sums[w * 256 + tid];
      const int q = q0 + 16 * f + l16;
      const float inv = 1.0f / l_all;
      if (q < a.T)
        *reinterpret_cast<u32x2*>(O + (int64_t)q * a.so.t + 16 * wave + 4 * g4) =
            u32x2{pack2<DT>(v[0] * inv, v[1] * inv), pack2<DT>(v[2] * inv, v[3] * inv)};
    }
  }
}

template <int DT, int QF>
static int launch_attention_small(const AttnArgs& a, hipStream_t s) {
  const int64_t total = (int64_t)((a.T + 16 * QF - 1) / (16 * QF)) * a.Z * a.H;
  LH_LAUNCH((attention16_small_kernel<DT, QF>), dim3((unsigned)(8 * ((total + 7) / 8))), dim3(kSmallWaves * 64), 0, s, a);
  return check_launch("attention16_small");
}

// Where the line lies (us in a graph, the other kernels / 16 rows / 32 rows per workgroup; non-causal, causal where said):
//  * Every 16-row workgroup has a CU to itself: 16 rows.  [1,4,256] 6.6 / 4.8 / 6.4, [1,12,100] 5.2 / 4.1 / 5.5, [1,2,2000]
//    28.9 / 13.2 / 14.9, [1,1,3000] 40.7 / 17.5 / 19.3.
//  * Every 32-row workgroup does: what a CU then pays for is K and V pulled from its L2 once per workgroup, which two
//    query tiles share.  [2,3,1000] 16.6 / 13.5 / 10.4, [1,12,512] 9.4 / 9.0 / 8.0, [1,2,3900] 51.5 / 40.2 / 25.0.  Below 400 keys
//    the shorter prologue of 16 rows is worth more ([8,4,200] 7.0 / 6.0 / 6.3); below 192 the other kernels have three
//    key tiles at most and win ([8,8,128] 5.1 / 5.4 / 5.8), and up to 64 even with few workgroups ([8,16,17] 3.9 / 4.1 / 5.2).
//  * Two per CU: causal only, where the lighter query tiles fill in, and long sequences only: [1,8,1500] causal 21.6 / 17.9 /
//    15.0, [2,4,2000] 27.6 / 24.6 / 19.6 (non-causal 28.9 / 39.6 / 27.7, [2,8,1000] 16.6 / 23.9 / 19.1, causal 15.7 / 18.4 / 15.2).
int attention_small_tiles(const AttnArgs& a) {
  const int64_t heads = (int64_t)a.Z * a.H, wgs16 = (a.T + 15) / 16 * heads, wgs32 = (a.T + 31) / 32 * heads;
  if (a.T <= 64) return 0;
  if (wgs16 <= a.cus) return 1;
  if (wgs32 <= a.cus && a.T >= 192) return a.T < 400 ? 1 : 2;
  return a.causal && a.T >= 1500 && wgs32 <= 2 * (int64_t)a.cus ? 2 : 0;
}

int attention_small(const AttnArgs& a, int dtype, int tiles, hipStream_t s) {
  if (dtype == LH_BF16) return tiles == 2 ? launch_attention_small<LH_BF16, 2>(a, s) : launch_attention_small<LH_BF16, 1>(a, s);
  return tiles == 2 ? launch_attention_small<LH_F16, 2>(a, s) : launch_attention_small<LH_F16, 1>(a, s);
}

}  // namespace lh
