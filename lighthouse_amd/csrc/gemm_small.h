// Operand panels of the small-tile GEMM kernels (gemm_small.hip, gemm_small_norm.hip): loads, the trip through LDS and the
// matrix instruction of one step.
#pragma once

#include <type_traits>

#include "gemm_common.h"

namespace lh {

typedef short small_s16x4 __attribute__((ext_vector_type(4)));
typedef int small_i32x2 __attribute__((ext_vector_type(2)));

// c += a b for one step: the lane's 16-byte chunks of a row of each operand (lane / 16 selects the chunk of
// the step's four).  First operand = B fragment: a lane's result is 4 consecutive columns of one row.
template <int DT>
__device__ __forceinline__ f32x4 small_mma(u32x4 b, u32x4 a, f32x4 c) {
  if constexpr (DT == LH_BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
  } else if constexpr (DT == LH_F16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, b), __builtin_bit_cast(f16x8, a), c, 0, 0, 0);
  } else if constexpr (DT == LH_F8E4M3) {
    typedef long l2 __attribute__((ext_vector_type(2)));
    const l2 bl = __builtin_bit_cast(l2, b), al = __builtin_bit_cast(l2, a);
    c = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(bl[0], al[0], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(bl[1], al[1], c, 0, 0, 0);
  } else {
    const f32x4 bf = __builtin_bit_cast(f32x4, b), af = __builtin_bit_cast(f32x4, a);
#pragma unroll
    for (int t = 0; t < 4; ++t) c = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[t], af[t], c, 0, 0, 0);
    return c;
  }
}

template <int DT>
constexpr int small_elem_bytes() { return DT == LH_F32 ? 4 : DT == LH_F8E4M3 ? 1 : 2; }

// The chunk moved down by `n` elements (0 .. EPC, or more: nothing is left), zeros on top.
template <int ES>
__device__ __forceinline__ u32x4 small_shift_chunk(u32x4 c, int n) {
  const int bytes = ES * n;
  uint32_t d0 = c[0], d1 = c[1], d2 = c[2], d3 = c[3];
  const bool by8 = bytes & 8, by4 = bytes & 4, all = bytes >= 16;
  d0 = by8 ? d2 : d0;
  d1 = by8 ? d3 : d1;
  d2 = by8 ? 0u : d2;
  d3 = by8 ? 0u : d3;
  d0 = by4 ? d1 : d0;
  d1 = by4 ? d2 : d1;
  d2 = by4 ? d3 : d2;
  d3 = by4 ? 0u : d3;
  const int b = bytes & 3;
  d0 = __builtin_amdgcn_alignbyte(d1, d0, b);
  d1 = __builtin_amdgcn_alignbyte(d2, d1, b);
  d2 = __builtin_amdgcn_alignbyte(d3, d2, b);
  d3 = __builtin_amdgcn_alignbyte(0u, d3, b);
  return u32x4{all ? 0u : d0, all ? 0u : d1, all ? 0u : d2, all ? 0u : d3};
}

// One operand panel of F fragments of 16 rows (A) or columns (B), k-contiguous (KC) or not.  Every load of
// a step is one 16-byte access whatever the sizes: a chunk that would cross the end of its row is read
// from the row's last EPC elements instead and moved down in registers (the contiguous dimension has at
// least EPC elements), so the number of loads in flight is known at compile time and the waits stay exact.
template <int DT, int F, bool KC>
struct SmallPanel {
  static constexpr int ES = small_elem_bytes<DT>(), EPC = 16 / ES, KSTEP = 64 / ES;
  static constexpr int CPR = F * ES;             // !KC: 16-byte chunks per k row
  static constexpr int RPL = 64 / CPR;           // !KC: k rows per load
  static constexpr int RS = CPR * 16 + 16;       // !KC: bytes of a k row in LDS (one chunk of padding)
  static constexpr int kLdsBytes = KC ? 0 : KSTEP * RS;
  const uint8_t* base[KC ? F : 1];  // KC: the lane's chunk of its row in each fragment; !KC: of its first k row
  int64_t ld_bytes;
  int over = 0;              // !KC: elements by which the lane's chunk was moved back to stay inside the row
  bool whole = true;         // !KC: (wave-uniform) no chunk of the panel was moved

  // `p`: the operand as stored; `first`: the panel's first row / column; `count`: rows / columns of the
  // matrix; `ld`: stored row stride.
  __device__ __forceinline__ void place(const void* p, int first, int count, int64_t ld, int lane) {
    ld_bytes = ld * ES;
    const uint8_t* b = reinterpret_cast<const uint8_t*>(p);
    if constexpr (KC) {
#pragma unroll
      for (int f = 0; f < F; ++f)
        base[f] = b + (int64_t)min(first + 16 * f + (lane & 15), count - 1) * ld_bytes + (lane >> 4) * 16;
    } else {
      const int c = first + (lane % CPR) * EPC, cc = min(c, count - EPC);
      over = c - cc;
      whole = first + 16 * F <= count;
      base[0] = b + (int64_t)(lane / CPR) * ld_bytes + (int64_t)cc * ES;
    }
  }
  // Request the step at k0, all of it below K.
  __device__ __forceinline__ void load(int k0, u32x4 (&r)[F]) const {
    typedef typename Chunk<ES>::type C;
    if constexpr (KC) {
#pragma unroll
      for (int f = 0; f < F; ++f) r[f] = *reinterpret_cast<const C*>(base[f] + (int64_t)k0 * ES);
    } else {
      const uint8_t* p = base[0] + (int64_t)k0 * ld_bytes;
#pragma unroll
      for (int f = 0; f < F; ++f) r[f] = *reinterpret_cast<const C*>(p + (int64_t)(f * RPL) * ld_bytes);
    }
  }
  // Request the step at k0 that K ends in; `finish_tail` turns what lies past K into zeros.
  __device__ __forceinline__ void load_tail(int k0, int K, int lane, u32x4 (&r)[F]) const {
    typedef typename Chunk<ES>::type C;
    if constexpr (KC) {
      const int k = k0 + (lane >> 4) * EPC, back = max(k - (K - EPC), 0);
#pragma unroll
      for (int f = 0; f < F; ++f) r[f] = *reinterpret_cast<const C*>(base[f] + (int64_t)(k0 - back) * ES);
    } else {
#pragma unroll
      for (int f = 0; f < F; ++f) {
        const int row = lane / CPR, k = min(k0 + f * RPL + row, K - 1) - row;
        r[f] = *reinterpret_cast<const C*>(base[0] + (int64_t)k * ld_bytes);
      }
    }
  }
  __device__ __forceinline__ void finish_tail(int k0, int K, int lane, u32x4 (&r)[F]) const {
    if constexpr (KC) {
      const int k = k0 + (lane >> 4) * EPC, back = max(k - (K - EPC), 0);
#pragma unroll
      for (int f = 0; f < F; ++f) r[f] = small_shift_chunk<ES>(r[f], back);
    } else {
#pragma unroll
      for (int f = 0; f < F; ++f)
        if (k0 + f * RPL + lane / CPR >= K) r[f] = u32x4{0u, 0u, 0u, 0u};
    }
  }
  // The step's chunks go into the wave's LDS area (!KC) ...
  template <bool WHOLE>
  __device__ __forceinline__ void stage(u32x4 (&r)[F], uint8_t* lds, int lane) const {
    if constexpr (!KC) {
      if constexpr (!WHOLE) {
#pragma unroll
        for (int f = 0; f < F; ++f) r[f] = small_shift_chunk<ES>(r[f], over);
      }
#pragma unroll
      for (int f = 0; f < F; ++f)
        *reinterpret_cast<u32x4*>(lds + (f * RPL + lane / CPR) * RS + (lane % CPR) * 16) = r[f];
    }
  }
  // ... where its fragments come from; KC: the registers themselves.
  __device__ __forceinline__ void fragments(const u32x4 (&r)[F], uint8_t* lds, int lane, u32x4 (&frag)[F]) const {
    if constexpr (KC) {
#pragma unroll
      for (int f = 0; f < F; ++f) frag[f] = r[f];
    } else {
      const int l16 = lane & 15, g4 = lane >> 4;
#pragma unroll
      for (int f = 0; f < F; ++f) {
        if constexpr (ES == 2) {
          // 16 lanes of group g4: k rows 8 g4 + l16 / 4 (+4), columns 16 f + 4 (l16 % 4) .. +4
          uint8_t* p0 = lds + (8 * g4 + (l16 >> 2)) * RS + 32 * f + 8 * (l16 & 3);
          const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                         (__attribute__((address_space(3))) small_s16x4*)p0));
          const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                         (__attribute__((address_space(3))) small_s16x4*)(p0 + 4 * RS)));
          frag[f] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        } else if constexpr (ES == 1) {
          // k rows 16 g4 + l16 / 2 (+8), bytes 16 f + 8 (l16 % 2) .. +8
          uint8_t* p0 = lds + (16 * g4 + (l16 >> 1)) * RS + 16 * f + 8 * (l16 & 1);
          const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                                                         (__attribute__((address_space(3))) small_i32x2*)p0));
          const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                                                         (__attribute__((address_space(3))) small_i32x2*)(p0 + 8 * RS)));
          frag[f] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t)
            frag[f][t] = *reinterpret_cast<const uint32_t*>(lds + (4 * g4 + t) * RS + (16 * f + l16) * 4);
        }
      }
    }
  }
};

// Four consecutive elements of a row as they are in memory, f32 when asked for.  Held unconverted and loaded without a
// branch, so that nothing waits for the load in between.
template <int EDT>
struct SmallRaw4 {
  u32x4 w;
  // Columns n .. n + 3 of the row of N >= 4 at p[at]; four that would cross the end of the row are its last four.
  __device__ __forceinline__ void load(const void* p, bool f32, int64_t at, int n, int N) {
    const int64_t i = at + min(n, N - 4);
    if constexpr (EDT == LH_F32) {
      w = *reinterpret_cast<const Chunk<4>::type*>(reinterpret_cast<const uint32_t*>(p) + i);
    } else {
      const uint16_t* q = reinterpret_cast<const uint16_t*>(p) + (f32 ? 2 * i : i);
      const u32x2 lo = *reinterpret_cast<const u32x2_any*>(q), hi = *reinterpret_cast<const u32x2_any*>(q + (f32 ? 4 : 0));
      w = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  }
  // ... as f32, those past the end undefined; `whole` (uniform): no lane's cross it.
  __device__ __forceinline__ f32x4 get(bool f32, int n, int N, bool whole) const {
    f32x4 v = __builtin_bit_cast(f32x4, w);
    if constexpr (EDT != LH_F32)
      if (!f32) v = f32x4{unpack_lo<EDT>(w[0]), unpack_hi<EDT>(w[0]), unpack_lo<EDT>(w[1]), unpack_hi<EDT>(w[1])};
    if (!whole) {
      const int over = n - min(n, N - 4);
      v = over == 1 ? f32x4{v[1], v[2], v[3], 0.0f} : over == 2 ? f32x4{v[2], v[3], 0.0f, 0.0f} : over == 3 ? f32x4{v[3], 0.0f, 0.0f, 0.0f} : v;
    }
    return v;
  }
};

// The elements of the tile at (m0, n0) that a thread finishes: their bias and accumulator input.  Requested in front of the
// main loop: at its end each would be a trip to memory of its own (M = 100, N = 768, K = 768 bf16 with an f32 residual: 0.9 us
// from the sums to the stores' end).
template <int EDT, int MT, int NT, int NW>
struct SmallEpilogue {
  static constexpr int IT = (MT * NT + NW - 1) / NW;
  SmallRaw4<EDT> bias[IT], c[IT];
  // Fragment f = it NW + wave of the tile: the lane's row and columns.
  static __device__ __forceinline__ void at(int m0, int n0, int f, int lane, int& m, int& n) {
    m = m0 + 16 * (f / NT) + (lane & 15);
    n = n0 + 16 * (f % NT) + 4 * (lane >> 4);
  }
  __device__ __forceinline__ void load(const GemmArgs& g, int m0, int n0, int wave, int lane) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int f = it * NW + wave;
      if (MT * NT % NW != 0 && f >= MT * NT) break;
      int m, n;
      at(m0, n0, f, lane, m, n);
      if (g.flags & LH_GEMM_HAS_BIAS) bias[it].load(g.bias, g.bias_dt == LH_F32, 0, n, g.N);
      if (g.flags & LH_GEMM_ACCUMULATE_C) c[it].load(g.c, g.out_dt == LH_F32, (int64_t)min(m, g.M - 1) * g.ldc, n, g.N);
    }
  }
  // The waves' partial tiles are added through LDS, in wave order, and finished; `loaded` (uniform): with what `load` has brought.
  __device__ __forceinline__ void sum_and_store(bool loaded, const GemmArgs& g, const f32x4 (&acc)[MT][NT], uint8_t* lds, int m0, int n0,
                                                int wave, int lane) const {
    // Fragment f = j NT + i of wave w is 1 KiB at (w MT NT + f) 1024, 16 bytes per lane.
    f32x4* const sums = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int i = 0; i < NT; ++i) sums[(wave * MT * NT + j * NT + i) * 64 + lane] = acc[j][i];
    __syncthreads();
    const bool whole = n0 + 16 * NT <= g.N;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int f = it * NW + wave;
      if (MT * NT % NW != 0 && f >= MT * NT) break;
      f32x4 v = sums[f * 64 + lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) v += sums[(w * MT * NT + f) * 64 + lane];
      int m, n;
      at(m0, n0, f, lane, m, n);
      if (m >= g.M || n >= g.N) continue;
      if (loaded) epilogue4_loaded<EDT>(g, m, n, v, bias[it].get(g.bias_dt == LH_F32, n, g.N, whole), c[it].get(g.out_dt == LH_F32, n, g.N, whole));
      else epilogue4_any<EDT>(g, m, n, v);
    }
  }
};

}  // namespace lh
