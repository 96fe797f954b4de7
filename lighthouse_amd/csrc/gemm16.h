// Shared by the 16-bit GEMM sources: the matrix instructions and the launches of the direct-to-LDS kernels.
#pragma once

#include "gemm_common.h"

namespace lh {

template <int DT>
struct Mfma16;
template <>
struct Mfma16<LH_BF16> {
  __device__ static __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  }
  __device__ static __forceinline__ f32x4 mma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  }
};
template <>
struct Mfma16<LH_F16> {
  __device__ static __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  }
  __device__ static __forceinline__ f32x4 mma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  }
};

// The direct kernels address a tile's operand panels with 32-bit byte offsets from the panel's
// first element: 256 rows of A, of B the rows of whole steps of 64 (those from K on are never read, but addressed).
static inline bool direct_offsets_fit(const GemmArgs& g) {
  if (g.flags & LH_GEMM_TRANSPOSE_B) return g.lda < (1ll << 22) && g.ldb < (1ll << 22);  // 256 rows of B^T
  return g.lda < (1ll << 22) && (g.K + 63ll) / 64 * 64 * g.ldb < (1ll << 30);
}

// Every row of the result starts at a multiple of 64 bytes: stores of whole row segments cover whole 64-byte pieces of memory.
__host__ __device__ static inline bool rows_of_pieces(const GemmArgs& g) {
  return ((reinterpret_cast<uintptr_t>(g.out) | (uintptr_t)(g.ldc * (g.out_dt == LH_F32 ? 4 : 2))) & 63) == 0;
}

// Tiles of bm x bn cover the result exactly, and all of its sides are aligned.
static inline bool whole_tiles(const GemmArgs& g, int bm, int bn) {
  return g.M % bm == 0 && g.N % bn == 0 && g.ldc % 8 == 0 && aligned16(g.out) && (!(g.flags & LH_GEMM_HAS_BIAS) || aligned16(g.bias)) &&
         (!(g.flags & LH_GEMM_ACCUMULATE_C) || aligned16(g.c));
}

// Launch of the direct-to-LDS kernel with a workgroup tile of (64 TM) x (128 TN) (gemm16_direct.hip; each
// combination is an object of its own).
template <int DT, int TM, int TN>
int launch_direct(const GemmArgs& g, hipStream_t s);
// ... of its 256 x 256 tile whose results leave past the caches; `whole`: there are no edge tiles and all sides are aligned.
template <int DT>
int launch_direct_large(const GemmArgs& g, bool whole, hipStream_t s);
// ... with deeper rings, for no more tiles than CUs: 128 x 128, 128 x 192 (TN 3; K a multiple of 64), 128 x 256 and 256 x 128.
template <int DT, int TM, int TN>
int launch_deep(const GemmArgs& g, hipStream_t s);
// The 128 x 128 tile on an n-contiguous B in rows of any length and alignment.
template <int DT>
int launch_odd_rows(const GemmArgs& g, hipStream_t s);
// The 128 x 128 tile on `g.splits` pieces of K, each with an f32 block of the output of its own.
template <int DT>
int launch_direct_splitk(const GemmArgs& g, hipStream_t s);

}  // namespace lh
