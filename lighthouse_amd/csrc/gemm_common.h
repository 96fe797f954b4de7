// Argument block and register epilogue shared by the GEMM kernels.
#pragma once

#include "common.h"

namespace lh {

struct GemmArgs {
  void* out;
  const void* c;  // accumulator input for ACCUMULATE_C (out_dt typed; may alias out)
  const void* a;
  const void* b;
  const void* bias;
  int M, N, K;
  int64_t lda, ldb, ldc;
  uint32_t flags;
  int out_dt;
  int bias_dt;  // element type of bias
  float alpha;  // accumulator scale applied first (1 for the unquantised payloads)
  // Split-K launches of the 16-bit direct kernel: `splits` problems of K columns each, problem sp reads
  // A from column sp K, B from row sp K and writes its own M x ldc block of `out`.
  int splits = 1;
  // Source of the call's temporary device memory; nullptr: the library's pool of the stream.
  Scratch* ws = nullptr;
  // 16-bit direct kernel: the workgroups touch B at the start (set by the launcher).
  int touch_b = 0;
  // B is a copy whose rows hold whole 16-byte chunks past column N (zeros): N need not be a multiple of them.
  bool b_padded = false;
  // The operands are copies made for kernels that want K in multiples of this (0: they are the caller's).  Decided once per
  // call: what is decided for the copies themselves may be another multiple, and a second copy would be written over the first.
  uint8_t k_multiple = 0;
};

// Epilogue for 4 consecutive columns of one row.
template <int DT>
__device__ __forceinline__ void epilogue4(const GemmArgs& g, int m, int n, float v0, float v1, float v2, float v3) {
  float v[4] = {v0 * g.alpha, v1 * g.alpha, v2 * g.alpha, v3 * g.alpha};
  const int64_t off = (int64_t)m * g.ldc + n;
  if (g.flags & LH_GEMM_ACCUMULATE_C) {
    if (g.out_dt == LH_F32) {
      f32x4 c = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(g.c) + off);
      v[0] += c[0]; v[1] += c[1]; v[2] += c[2]; v[3] += c[3];
    } else {
      u32x2 c = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(g.c) + off);
      v[0] += unpack_lo<DT>(c[0]); v[1] += unpack_hi<DT>(c[0]);
      v[2] += unpack_lo<DT>(c[1]); v[3] += unpack_hi<DT>(c[1]);
    }
  }
  if (g.flags & LH_GEMM_HAS_BIAS) {
    if (g.bias_dt == LH_F32) {
      f32x4 bb = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(g.bias) + n);
      v[0] += bb[0]; v[1] += bb[1]; v[2] += bb[2]; v[3] += bb[3];
    } else {
      u32x2 bb = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(g.bias) + n);
      v[0] += unpack_lo<DT>(bb[0]); v[1] += unpack_hi<DT>(bb[0]);
      v[2] += unpack_lo<DT>(bb[1]); v[3] += unpack_hi<DT>(bb[1]);
    }
  }
  if (g.flags & LH_GEMM_HAS_GELU) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
  }
  const bool relu = (g.flags & LH_GEMM_HAS_RELU) != 0;
  if (g.out_dt == LH_F32) {
    if (relu) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = relu_nan(v[e]);
    }
    f32x4 o = {v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(g.out) + off) = o;
  } else {
    if (relu) {
      // ReLU is applied after the conversion (gpu_mlp_payload.py:147-151); max(x,0) and
      // rounding commute for every input (0 is representable and rounding is monotone).
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = relu_nan(v[e]);
    }
    u32x2 o = {pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
    *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(g.out) + off) = o;
  }
}

// Vectors of 4 output-side elements at element alignment (gfx9 global memory takes any alignment): the
// outputs, biases and accumulator inputs of problems whose N or row stride is odd.
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(2)));

typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));

// 4 elements at p[at], of which the first `left` exist (zeros for the others), as f32.
template <int DT>
__device__ __forceinline__ f32x4 load4_any(const void* p, int64_t at, int left) {
  f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (left >= 4) {
    if constexpr (DT == LH_F32) return *reinterpret_cast<const f32x4_any*>(reinterpret_cast<const float*>(p) + at);
    const u32x2 w = *reinterpret_cast<const u32x2_any*>(reinterpret_cast<const uint16_t*>(p) + at);
    return f32x4{unpack_lo<DT>(w[0]), unpack_hi<DT>(w[0]), unpack_lo<DT>(w[1]), unpack_hi<DT>(w[1])};
  }
#pragma unroll
  for (int e = 0; e < 3; ++e)
    if (e < left) v[e] = load_as_f32<DT>(p, at + e);
  return v;
}
// ... and stored (STREAM: whole vectors past the caches).
template <int DT, bool STREAM = false>
__device__ __forceinline__ void store4_any(void* p, int64_t at, const f32x4& v, int left) {
  if (left >= 4) {
    if constexpr (DT == LH_F32) {
      f32x4_any* const d = reinterpret_cast<f32x4_any*>(reinterpret_cast<float*>(p) + at);
      if constexpr (STREAM) __builtin_nontemporal_store(f32x4_any(v), d);
      else *d = v;
    } else {
      u32x2_any* const d = reinterpret_cast<u32x2_any*>(reinterpret_cast<uint16_t*>(p) + at);
      const u32x2 w = {pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
      if constexpr (STREAM) __builtin_nontemporal_store(u32x2_any(w), d);
      else *d = w;
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < 3; ++e)
    if (e < left) store_from_f32<DT>(p, at + e, v[e]);
}
// 8 packed 16-bit values, of which the first `left` are stored (STREAM: all eight past the caches).
template <bool STREAM>
__device__ __forceinline__ void store8_any(uint16_t* p, const u32x4& w, int left) {
  if (left >= 8) {
    if constexpr (STREAM) __builtin_nontemporal_store(u32x4_any(w), reinterpret_cast<u32x4_any*>(p));
    else *reinterpret_cast<u32x4_any*>(p) = w;
    return;
  }
#pragma unroll
  for (int e = 0; e < 7; ++e)
    if (e < left) p[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
}

// Bias of 4 consecutive columns as f32 (zeros without a bias).  ANY: any alignment, zeros from column N on.
template <int DT, bool ANY = false>
__device__ __forceinline__ f32x4 bias4(const GemmArgs& g, int n) {
  f32x4 r = {0.0f, 0.0f, 0.0f, 0.0f};
  if (g.flags & LH_GEMM_HAS_BIAS) {
    if constexpr (ANY) return g.bias_dt == LH_F32 ? load4_any<LH_F32>(g.bias, n, g.N - n) : load4_any<DT>(g.bias, n, g.N - n);
    if (g.bias_dt == LH_F32) {
      r = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(g.bias) + n);
    } else {
      u32x2 bb = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(g.bias) + n);
      r = f32x4{unpack_lo<DT>(bb[0]), unpack_hi<DT>(bb[0]), unpack_lo<DT>(bb[1]), unpack_hi<DT>(bb[1])};
    }
  }
  return r;
}

// ---- epilogue variants fixed at compile time ----------------------------------------------
// epilogue4 tests the flags of the call for every group of 4 elements.  In a tile
// kernel whose epilogue is unrolled over the tile that is a handful of scalar branches around a
// few vector instructions, a hundred times over, in code that runs once per tile and is cold in
// the instruction cache each time: the 256 x 256 bf16 tile spent 5.2 us converting and staging
// 128 KiB of output that way, 2.5 us without the tests.  The tile kernels therefore choose ONE
// variant per tile (epi_dispatch: a chain of wave-uniform branches at the top of the epilogue)
// and run straight-line code specialised for it; EpiAny keeps the run-time tests for the
// combinations that have no variant of their own.  Same operations in the same order either way
// (a scale of exactly 1 is skipped: x * 1 == x bit for bit).
template <bool ALPHA, bool BIAS, int ACT>  // ACT: 0 none, 1 ReLU, 2 tanh-GELU
struct EpiFixed {
  static constexpr bool kAny = false, kAlpha = ALPHA, kBias = BIAS;
  static constexpr int kAct = ACT;
};
struct EpiAny {
  static constexpr bool kAny = true, kAlpha = true, kBias = true;
  static constexpr int kAct = -1;
};
template <typename E>
__device__ __forceinline__ bool epi_has_bias(const GemmArgs& g) {
  if constexpr (E::kAny) return (g.flags & LH_GEMM_HAS_BIAS) != 0;
  else return E::kBias;
}
// Scale, bias and activation on 4 values, in epilogue4's order.
template <typename E>
__device__ __forceinline__ void epi_apply4(const GemmArgs& g, const f32x4& bias, float (&v)[4]) {
  if constexpr (E::kAny) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] *= g.alpha;
    if (g.flags & LH_GEMM_HAS_BIAS) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += bias[e];
    }
    if (g.flags & LH_GEMM_HAS_GELU) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
    }
    if (g.flags & LH_GEMM_HAS_RELU) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = relu_nan(v[e]);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (E::kAlpha) v[e] *= g.alpha;
      if constexpr (E::kBias) v[e] += bias[e];
      if constexpr (E::kAct == 2) v[e] = gelu_tanh(v[e]);
      if constexpr (E::kAct == 1) v[e] = relu_nan(v[e]);
    }
  }
}
// 4 accumulator values -> two packed dwords of a 16-bit output (no accumulator input).
template <int DT, typename E>
__device__ __forceinline__ u32x2 epi_pack4(const GemmArgs& g, const f32x4& bias, const f32x4& a) {
  float v[4] = {a[0], a[1], a[2], a[3]};
  epi_apply4<E>(g, bias, v);
  return u32x2{pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
}
// Calls f with the variant of the call: unscaled accumulators without a bias, with a bias, with a
// bias followed by ReLU or GELU, scaled accumulators without a bias (the fp8 payload); anything
// else takes EpiAny.
template <typename F>
__device__ __forceinline__ void epi_dispatch(const GemmArgs& g, F&& f) {
  const uint32_t k = g.flags & (LH_GEMM_HAS_BIAS | LH_GEMM_HAS_GELU | LH_GEMM_HAS_RELU);
  if (g.alpha == 1.0f) {
    if (k == 0) return f(EpiFixed<false, false, 0>{});
    if (k == LH_GEMM_HAS_BIAS) return f(EpiFixed<false, true, 0>{});
    if (k == (LH_GEMM_HAS_BIAS | LH_GEMM_HAS_RELU)) return f(EpiFixed<false, true, 1>{});
    if (k == (LH_GEMM_HAS_BIAS | LH_GEMM_HAS_GELU)) return f(EpiFixed<false, true, 2>{});
  } else if (k == 0) {
    return f(EpiFixed<true, false, 0>{});
  }
  f(EpiAny{});
}
// The same without the activation variants, for epilogues that also specialise on the output
// type and the accumulator input (residual adds, f32 outputs, split-K blocks).
template <typename F>
__device__ __forceinline__ void epi_dispatch_linear(const GemmArgs& g, F&& f) {
  const uint32_t k = g.flags & (LH_GEMM_HAS_BIAS | LH_GEMM_HAS_GELU | LH_GEMM_HAS_RELU);
  if (g.alpha == 1.0f) {
    if (k == 0) return f(EpiFixed<false, false, 0>{});
    if (k == LH_GEMM_HAS_BIAS) return f(EpiFixed<false, true, 0>{});
  }
  f(EpiAny{});
}
// epilogue4 with the variant, the output type and the presence of an accumulator input fixed.
template <int DT, typename E, bool OUT32, bool HAS_C>
__device__ __forceinline__ void epi_store4(const GemmArgs& g, int m, int n, const f32x4& bias, const f32x4& a) {
  float v[4] = {a[0], a[1], a[2], a[3]};
  const int64_t off = (int64_t)m * g.ldc + n;
  if constexpr (HAS_C) {
    // (the accumulator input is added to the scaled accumulator before the bias, as in epilogue4)
    if constexpr (E::kAlpha) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= g.alpha;
    }
    if constexpr (OUT32) {
      const f32x4 c = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(g.c) + off);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += c[e];
    } else {
      const u32x2 c = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(g.c) + off);
      v[0] += unpack_lo<DT>(c[0]); v[1] += unpack_hi<DT>(c[0]);
      v[2] += unpack_lo<DT>(c[1]); v[3] += unpack_hi<DT>(c[1]);
    }
    if constexpr (E::kAny) {
      if (g.flags & LH_GEMM_HAS_BIAS) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += bias[e];
      }
      if (g.flags & LH_GEMM_HAS_GELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
      }
      if (g.flags & LH_GEMM_HAS_RELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = relu_nan(v[e]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (E::kBias) v[e] += bias[e];
        if constexpr (E::kAct == 2) v[e] = gelu_tanh(v[e]);
        if constexpr (E::kAct == 1) v[e] = relu_nan(v[e]);
      }
    }
  } else {
    epi_apply4<E>(g, bias, v);
  }
  if constexpr (OUT32)
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(g.out) + off) = f32x4{v[0], v[1], v[2], v[3]};
  else
    *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(g.out) + off) = u32x2{pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
}

// Memory of the copies that untranspose_operands makes; `a_bytes`: those of the copy of A, in front.
template <int ELEM_BYTES>
inline size_t untransposed_bytes(const GemmArgs& g, size_t* a_bytes) {
  const bool ta = g.flags & LH_GEMM_TRANSPOSE_A, tb = g.flags & LH_GEMM_TRANSPOSE_B;
  *a_bytes = ta ? ((size_t)g.M * g.K * ELEM_BYTES + 255) / 256 * 256 : 0;
  return *a_bytes + (tb ? (size_t)g.K * g.N * ELEM_BYTES : 0);
}
// The call's workspace has room for the copies (not in a size query, which has none); `b_in_place`: a transposed B stays.
template <int ELEM_BYTES>
inline bool untransposed_room(GemmArgs g, bool b_in_place) {
  if (b_in_place) g.flags &= ~(uint32_t)LH_GEMM_TRANSPOSE_B;
  size_t a_bytes;
  return g.ws->base && (g.ws->used + 255) / 256 * 256 + untransposed_bytes<ELEM_BYTES>(g, &a_bytes) <= g.ws->bytes;
}

// Transposed operands (A stored [K,M], B stored [N,K]) of a problem the direct kernels would
// otherwise take are first transposed into temporary memory (one extra pass over that
// operand, about a tenth of a 4096^3 problem's time) instead of running the slower kernels that
// read them in place.  Returns 0 and rewrites `g` on success, 1 when the problem does not qualify.
template <int ELEM_BYTES>
inline int untranspose_operands(GemmArgs& g, int k_multiple, int n_multiple, hipStream_t s) {
  const bool ta = g.flags & LH_GEMM_TRANSPOSE_A, tb = g.flags & LH_GEMM_TRANSPOSE_B;
  if (!(ta || tb) || g.K % k_multiple != 0 || g.N % n_multiple != 0) return 1;
  size_t a_bytes;
  const size_t bytes = untransposed_bytes<ELEM_BYTES>(g, &a_bytes);
  void* taken = nullptr;
  if (int rc = scratch_take(g.ws, s, kScratchTranspose, bytes, "gemm (transposed operands)", &taken)) return rc;
  char* buf = static_cast<char*>(taken);
  if (ta) {  // stored [K, M] -> [M, K]
    if (int rc = transpose_matrix(buf, g.a, g.K, g.M, g.lda, g.K, ELEM_BYTES, s)) return rc;
    g.a = buf;
    g.lda = g.K;
  }
  if (tb) {  // stored [N, K] -> [K, N]
    if (int rc = transpose_matrix(buf + a_bytes, g.b, g.N, g.K, g.ldb, g.N, ELEM_BYTES, s)) return rc;
    g.b = buf + a_bytes;
    g.ldb = g.N;
  }
  g.flags &= ~(uint32_t)(LH_GEMM_TRANSPOSE_A | LH_GEMM_TRANSPOSE_B);
  return 0;
}

// Every operand that is not transposed (and so copied into rows that are) has rows of aligned 16-byte chunks.
template <int ELEM_BYTES>
inline bool rows_fit_untransposed(const GemmArgs& g) {
  auto fit = [](const void* p, int64_t ld) { return ld % (16 / ELEM_BYTES) == 0 && aligned16(p); };
  return ((g.flags & LH_GEMM_TRANSPOSE_A) || fit(g.a, g.lda)) && ((g.flags & LH_GEMM_TRANSPOSE_B) || fit(g.b, g.ldb));
}

// The copies that the direct kernels need in front of them: what untranspose_operands and gemm_padded will make.
struct OperandCopies {
  bool a, b, odd_k, odd_n;
};
template <int ELEM_BYTES>
inline OperandCopies operand_copies(const GemmArgs& g, int k_multiple, int n_multiple, bool b_in_place) {
  const bool ta = g.flags & LH_GEMM_TRANSPOSE_A, tb = g.flags & LH_GEMM_TRANSPOSE_B;
  const bool odd_k = g.K % k_multiple != 0, odd_n = g.N % n_multiple != 0 && !g.b_padded;
  auto odd_rows = [](const void* p, int64_t ld) { return ld % (16 / ELEM_BYTES) != 0 || !aligned16(p); };
  const bool a = ta || odd_k || odd_rows(g.a, g.lda);
  const bool a_padded = a && (!ta || odd_k || odd_n);  // (by gemm_padded, which then copies a B that could stay, too)
  const bool b = tb ? !b_in_place || a_padded : odd_k || odd_n || odd_rows(g.b, g.ldb);
  return OperandCopies{a, b, odd_k, odd_n};
}

// Their time, in us (0: none): 3.5 us a launch and `us_per_mb` per MB of operand copied or zeroed.
template <int ELEM_BYTES>
inline double operand_copies_us(const GemmArgs& g, int k_multiple, int n_multiple, bool b_in_place, double us_per_mb) {
  const bool ta = g.flags & LH_GEMM_TRANSPOSE_A, tb = g.flags & LH_GEMM_TRANSPOSE_B;
  const OperandCopies c = operand_copies<ELEM_BYTES>(g, k_multiple, n_multiple, b_in_place);
  const double mb_a = c.a ? 1e-6 * ELEM_BYTES * g.M * g.K : 0.0, mb_b = c.b ? 1e-6 * ELEM_BYTES * g.K * g.N : 0.0;
  const bool fill_a = c.a && ta && c.odd_k, fill_b = c.b && tb && (c.odd_k || c.odd_n);  // zeros below a transposed copy
  const int launches = (c.a && ta) + (c.b && tb) + fill_a + fill_b + ((c.a && !ta) || (c.b && !tb));
  return 3.5 * launches + us_per_mb * (mb_a * (1 + fill_a) + mb_b * (1 + fill_b));
}

// A problem whose K the direct kernels cannot take (no multiple of the k-step), or whose operand rows are not
// 16-byte aligned, runs on them all the same: A and B are copied into temporary matrices padded with zeros,
// both in one launch.  The kernels write any N, row stride and alignment themselves, except those of fp8
// (PAD_C), which write a padded result that is copied back.  `run` launches the padded problem.  Returns 1
// when nothing needs padding, a negative status on failure.  (bf16 4096 x 4100 x 4096: 2012 us on the
// bounds-checked kernel, 224 with every operand padded; M = 8192, N = 50257, K = 768 with f32 output: the copy of
// the 1.6 GB result back alone took 1751 us.)
template <int ELEM_BYTES, bool PAD_C, typename Run>
inline int gemm_padded(const GemmArgs& g, int k_multiple, int n_multiple, hipStream_t s, Run run) {
  if (g.k_multiple) return 1;  // (copies already; the memory of the next would be theirs)
  const bool ta = g.flags & LH_GEMM_TRANSPOSE_A, tb = g.flags & LH_GEMM_TRANSPOSE_B;
  const int out_bytes = g.out_dt == LH_F32 ? 4 : 2;
  const int Kp = (g.K + k_multiple - 1) / k_multiple * k_multiple;
  const int Np = (g.N + n_multiple - 1) / n_multiple * n_multiple;
  const bool acc = g.flags & LH_GEMM_ACCUMULATE_C;
  // (a transposed operand is copied in any case: the copy is where it gets untransposed)
  const bool pad_a = ta || Kp != g.K || g.lda % (16 / ELEM_BYTES) != 0 || !aligned16(g.a);
  const bool pad_b = tb || Kp != g.K || Np != g.N || g.ldb % (16 / ELEM_BYTES) != 0 || !aligned16(g.b);
  const bool odd_c = Np != g.N || g.ldc % n_multiple != 0 || !aligned16(g.out) || (acc && !aligned16(g.c));
  if (!(pad_a || pad_b || (PAD_C && odd_c))) return 1;
  auto round256 = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t a_bytes = pad_a ? round256((size_t)g.M * Kp * ELEM_BYTES) : 0;
  const size_t b_bytes = pad_b ? round256((size_t)Kp * Np * ELEM_BYTES) : 0;
  size_t bytes = a_bytes + b_bytes;
  if (PAD_C && odd_c) bytes += round256((size_t)g.M * Np * out_bytes);
  GemmArgs p = g;
  p.K = Kp;
  p.k_multiple = (uint8_t)k_multiple;
  if (bytes > 0) {
    void* taken = nullptr;
    if (int rc = scratch_take(g.ws, s, kScratchPad, bytes, "gemm (padded operands)", &taken)) return rc;
    char* buf = static_cast<char*>(taken);
    PadCopy copies[2];
    int ncopies = 0;
    if (pad_a) {
      if (ta) {  // stored [K, M]: zeros first (the padding), then the transposed matrix on top
        if (Kp != g.K)
          if (int rc = pad_copy_matrix(buf, Kp, g.M, Kp, g.a, g.lda, 0, 0, ELEM_BYTES, s)) return rc;
        if (int rc = transpose_matrix(buf, g.a, g.K, g.M, g.lda, Kp, ELEM_BYTES, s)) return rc;
      } else {
        copies[ncopies++] = PadCopy{buf, g.a, Kp, g.lda, g.M, Kp, g.M, g.K};
      }
      p.a = buf;
      p.lda = Kp;
    }
    if (pad_b) {
      char* bp = buf + a_bytes;
      if (tb) {  // stored [N, K]
        if (Kp != g.K || Np != g.N)
          if (int rc = pad_copy_matrix(bp, Np, Kp, Np, g.b, g.ldb, 0, 0, ELEM_BYTES, s)) return rc;
        if (int rc = transpose_matrix(bp, g.b, g.N, g.K, g.ldb, Np, ELEM_BYTES, s)) return rc;
      } else {
        copies[ncopies++] = PadCopy{bp, g.b, Np, g.ldb, Kp, Np, g.K, g.N};
      }
      p.b = bp;
      p.ldb = Np;
      p.b_padded = true;
    }
    if (ncopies)
      if (int rc = pad_copy_matrices(copies, ncopies, ELEM_BYTES, s)) return rc;
    p.flags &= ~(uint32_t)(LH_GEMM_TRANSPOSE_A | LH_GEMM_TRANSPOSE_B);
    static_assert(!PAD_C || ELEM_BYTES == 1, "fp8 products have neither a bias nor an accumulator input");
    if (PAD_C) {
      p.N = Np;
      if (odd_c) {
        p.out = buf + a_bytes + b_bytes;
        p.c = p.out;
        p.ldc = Np;
      }
    }
  }
  if (int rc = run(p)) return rc;
  if (PAD_C && odd_c) return pad_copy_matrix(g.out, g.ldc, g.M, g.N, p.out, Np, g.M, g.N, out_bytes, s);
  return LH_OK;
}

// Sum over the f32 blocks of a split-K launch for 4 consecutive columns: p + sp * step, sp = 0 ..
// splits - 1, added in that order.  `deep`: up to 8 loads are in flight before the first add, for the
// small reductions (a few MiB spread over every CU) that are bound by latency alone; large ones
// are faster with one block at a time (8 streams several MiB apart: 41 -> 43 us at 256 x 8192 x 8).
__device__ __forceinline__ f32x4 splitk_sum4(const float* p, int64_t step, int splits, bool deep) {
  f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (!deep) {
    for (int sp = 0; sp < splits; ++sp) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(p + sp * step);
      v[0] += t[0]; v[1] += t[1]; v[2] += t[2]; v[3] += t[3];
    }
    return v;
  }
  int sp = 0;
  for (; sp + 8 <= splits; sp += 8) {
    f32x4 t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = *reinterpret_cast<const f32x4*>(p + (sp + u) * step);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      v[0] += t[u][0]; v[1] += t[u][1]; v[2] += t[u][2]; v[3] += t[u][3];
    }
  }
  for (; sp < splits; ++sp) {
    const f32x4 t = *reinterpret_cast<const f32x4*>(p + sp * step);
    v[0] += t[0]; v[1] += t[1]; v[2] += t[2]; v[3] += t[3];
  }
  return v;
}

// Workgroup size of a reduce kernel over `groups` 4-column groups: one wave per workgroup while
// that still gives every CU only a few of them (decode batches up to 32 rows of 8192), else 256.
static inline int reduce_block(int64_t groups) { return groups <= 64 * 1024 ? 64 : 256; }

// One output element, any alignment (edge tiles and the generic kernels).
template <int DT>
__device__ __forceinline__ void epilogue1(const GemmArgs& g, int m, int n, float x) {
  const int64_t off = (int64_t)m * g.ldc + n;
  x *= g.alpha;
  if (g.flags & LH_GEMM_ACCUMULATE_C)
    x += (g.out_dt == LH_F32) ? reinterpret_cast<const float*>(g.c)[off] : load_as_f32<DT>(g.c, off);
  if (g.flags & LH_GEMM_HAS_BIAS)
    x += (g.bias_dt == LH_F32) ? reinterpret_cast<const float*>(g.bias)[n] : load_as_f32<DT>(g.bias, n);
  if (g.flags & LH_GEMM_HAS_GELU) x = gelu_tanh(x);
  if (g.flags & LH_GEMM_HAS_RELU) x = relu_nan(x);
  if (g.out_dt == LH_F32) reinterpret_cast<float*>(g.out)[off] = x;
  else store_from_f32<DT>(g.out, off, x);
}

// epilogue4 for columns n .. n + 3 of row m, of which those below N exist; any alignment.  The bias and accumulator input of the
// call are in `bias` and `c`.
template <int DT>
__device__ __forceinline__ void epilogue4_loaded(const GemmArgs& g, int m, int n, const f32x4& acc, const f32x4& bias, const f32x4& c) {
  float v[4] = {acc[0] * g.alpha, acc[1] * g.alpha, acc[2] * g.alpha, acc[3] * g.alpha};
  const int64_t off = (int64_t)m * g.ldc + n;
  const int left = g.N - n;
  if (g.flags & LH_GEMM_ACCUMULATE_C) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += c[e];
  }
  if (g.flags & LH_GEMM_HAS_BIAS) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += bias[e];
  }
  if (g.flags & LH_GEMM_HAS_GELU) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
  }
  if (g.flags & LH_GEMM_HAS_RELU) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = relu_nan(v[e]);
  }
  const f32x4 o = {v[0], v[1], v[2], v[3]};
  if (g.out_dt == LH_F32) store4_any<LH_F32>(g.out, off, o, left);
  else store4_any<DT>(g.out, off, o, left);
}
// ... loaded here.
template <int DT>
__device__ __forceinline__ void epilogue4_any(const GemmArgs& g, int m, int n, const f32x4& acc) {
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 bias = zero, c = zero;
  if (g.flags & LH_GEMM_ACCUMULATE_C) {
    const int64_t off = (int64_t)m * g.ldc + n;
    c = g.out_dt == LH_F32 ? load4_any<LH_F32>(g.c, off, g.N - n) : load4_any<DT>(g.c, off, g.N - n);
  }
  if (g.flags & LH_GEMM_HAS_BIAS) bias = bias4<DT, true>(g, n);
  epilogue4_loaded<DT>(g, m, n, acc, bias, c);
}

// Results so large that they push the operands out of the memory-side cache (256 MB, of which reads and writes both take) leave
// past the caches.  256 x 256 tiles, K = 768 bf16, plain and past the caches: 8192 x 50432 654 and 563 us (main loop of a tile
// 23.6 and 17.7), f32 797 and 763; 8192 x 16392 234 and 206; 8192 x 8200 x 2048 252 either way; fp8 8192^3 407 and 401.
// Smaller ones, which the next kernel reads, lose as often as they gain: nanoGPT blocks of 2048 rows 88 and 93 us, of 4096
// rows 138 and 135.5.  What counts is what is written, not the rows that it lies in: 2560 columns of a buffer of 65536, M = 4096,
// K = 1024, and a product that reads them 53 plain and 62 past the caches.
static inline bool large_result(const GemmArgs& g) { return (int64_t)g.M * g.N * (g.out_dt == LH_F32 ? 4 : 2) >= 128000000; }

int gemm16(const GemmArgs& g, int ab_dtype, hipStream_t s);
// Estimated time of a 16-bit product with few tiles, untransposed and aligned, not cut along K, in us.
double gemm16_us(const GemmArgs& g, int ab_dtype);
int gemm32(const GemmArgs& g, hipStream_t s);
int gemm8(const GemmArgs& g, hipStream_t s);
// Kernels for problems with few output tiles (gemm_small.hip): the tile they would use (-1: none fits the
// problem) with an estimate of its time in us, and the launch.  They need no temporary memory and take any
// alignment; a workspace query (planning()) does not ask, so that its figure is an upper bound that does
// not depend on which kernel is the faster one.
double gemm_small_choose(const GemmArgs& g, int dtype, int* tile);
// They are taken where their estimate is below the other kernels' by more than the two estimates' error: in a tie
// the tile kernels stay, which add up k in one order whatever the tile.
constexpr double kSmallMargin = 1.08;
int gemm_small(const GemmArgs& g, int dtype, int tile, hipStream_t s);

// LayerNorm of x and up to three products of its result, side by side in the output, in one launch (gemm_small_norm.hip).
struct NormedGemm {
  // a: x, f32; N: columns of one product; ldc: of all of them; flags: of every product.  Its b and bias are those of no product:
  // the kernel puts the group's bias there.
  GemmArgs g;
  const float *gamma, *beta;
  float eps, inv_n;
  const void* b[3];
  const void* bias[3];
  int groups;
  Touch next;  // what launches after this one read
};
// The tile it would run on; -1: the LayerNorm and the products on their own are the faster way, or it does not take them.
int gemm_normed_choose(const NormedGemm& n, int dtype);
int gemm_normed(const NormedGemm& n, int dtype, int tile, hipStream_t s);

}  // namespace lh
