// Arguments and launcher of the query-tile attention kernel
// (hexkv_prefill.hip), which hexkv_attend runs for calls of several query
// rows per sequence.
#pragma once

#include "hexkv_common.h"

namespace hexkv {

struct TileArgs {
  const void *q;
  int64_t q_bs, q_rs;  // elements
  const void *cache;
  int64_t c_bs, c_ps, c_kv;  // elements
  void *out;
  int64_t o_bs, o_rs;  // elements
  const int32_t *seqlens;
  int32_t bias, q_len, causal;
  int32_t q_heads, kv_heads, group;  // group: query heads per KV head
  int32_t part, max_parts;           // positions per key partition, partitions of the longest row
  int32_t max_seqlen;                // every row length is clamped to it
  int32_t pairs, tiles;              // (sequence, KV head) pairs; row tiles of one pair
  float scale_log2;
  float *ws_o, *ws_ml;   // split rows: partials as the decode kernels store them
  unsigned int *status;  // HEXKV_STATUS_* word, or nullptr
};

// Whether the kernel is compiled for these types and sizes.
bool tiles_support(int dtype, int head_dim);

// Query rows of one pair (q_len * group of them) per workgroup: 32 for each of
// its four waves.
constexpr int kTileRows = 128;

// One launch over every tile (and key partition); a.pairs, a.q_len, a.group
// and a.max_parts set, a.tiles filled here.
int launch_tiles(TileArgs a, int dtype, int head_dim, int64_t batch, hipStream_t stream, const char *what);

}  // namespace hexkv
