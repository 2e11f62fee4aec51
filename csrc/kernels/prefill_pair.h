// Launch of prefill_pair.hip, which attention.hip's prefill entry points choose.
#pragma once
#include "common.h"

struct PairArgs {
  const bf16* q;
  int64_t q_stride;
  const void *k_cache, *v_cache;
  const int* block_tables;
  int bt_stride;
  const int *cu_q, *kv_lens, *items;   // items: (sequence, row), or of split ranges (sequence, row, first key, part)
  int listed, chunk;                   // as ome_paged_prefill_split has them
  float *part_o, *part_ml;
  bf16* out;
  int64_t out_stride;
  int Hkv;
  float mul, v_scale;                  // of scores, to the base 2
  const float* sinks;
};

// split 0: a workgroup an item; 1: a workgroup a piece; 2: a workgroup a run of pieces.  grid: those times Hkv
void ome_prefill_pair(const PairArgs& a, int kv_fmt, int split, int grid, hipStream_t stream);
