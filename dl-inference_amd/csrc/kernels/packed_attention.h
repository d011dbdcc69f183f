#pragma once

// Arguments of the packed-row attention kernels (packed_attention.hip), shared by the host launch
// code and the kernels.
#include <stdint.h>

namespace dk {

constexpr int kPackedTileK = 64;  // keys per tile

struct PackedAttentionArgs {
  const void* q;  // [B, Hq, Sq, D]
  const void* k;  // [B, Hkv, keys, D], or the key pool [block, Hkv, block_size, D]
  const void* v;  // [B, Hkv, keys, D], or the value pool [block, Hkv, D, block_size]
  const int32_t* block_table;  // paged: [B, max_blocks]
  const void* positions;       // paged: tokens cached before the queries, per sequence, or NULL
  void* out;                   // [B, Hq, Sq, D]
  float* part_ml;              // splits > 1: [splits][B Hkv][rows] of (max, sum)
  float* part_o;               // splits > 1: [splits][B Hkv][rows][D]
  int64_t past;                // paged: tokens cached before the queries when positions is NULL
  int64_t max_blocks;
  int32_t pos64, block_size, q_heads, kv_heads, seq_q;
  int32_t keys;  // Sk, or the cache's capacity per sequence
  int32_t causal, splits;
  float scale_log2;  // the softmax scale times log2(e)
};

}  // namespace dk
