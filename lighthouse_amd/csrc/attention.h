// What the attention sources share: the arguments of a launch and the entry of the small-problem kernel.
#pragma once

#include "common.h"

namespace lh {

struct AttnArgs {
  void* out;
  const void* q;
  const void* k;
  const void* v;
  int Z, H, T;
  lh_strides3 so, sq, sk, sv;
  float scale_log2e;  // scale * log2(e)
  float scale;
  int causal;
  int cus;  // compute units of the device (causal launch order)
  int request = 0;  // LH_ATTN_ROWS_* | LH_ATTN_STAGES_* bits of the call (0: the library chooses)
  bool scale_f32 = false;  // LH_ATTN_SCALE_F32: Q stays as stored and the scores are scaled in f32
  int d = 0;        // head dimension of the call (the padded kernels mask the columns from d on)
  // Key range split between workgroups (few query blocks, long sequences): `kv_groups` workgroups
  // per query block each take a contiguous share of its key tiles and leave (unnormalised output,
  // offset, row sum) in `part`; attention16_merge combines them.  1: one workgroup per query block.
  int kv_groups = 1;
  float* part = nullptr;
  // Causal launches of up to a third more query blocks than fit the CUs at once (32 rows per wave,
  // three workgroups per CU): the grid is `chain` = 3 x CUs workgroups, all resident, and the first
  // third of them take a second query block each (see attention16_kernel).  0: one block per workgroup.
  int chain = 0;
  // 64 rows per wave, two workgroups per CU: of every 8 key tiles, the number for which the younger
  // workgroup's waves hold the higher priority (0: the two take turns tile by tile).
  int pair_bias = 0;
  bool allow_grid_split = true;  // the caller lets the launch take temporary memory for it
  Scratch* ws = nullptr;         // where that memory comes from: a caller workspace, or (nullptr) the stream's pool
};

// The small-problem kernel (16-bit tensors, head dimension 64, 16-byte aligned rows): 16-row query tiles per
// workgroup that it should run `a` with, 0 if the other kernels are the faster ones.
int attention_small_tiles(const AttnArgs& a);
int attention_small(const AttnArgs& a, int dtype, int tiles, hipStream_t s);

}  // namespace lh
