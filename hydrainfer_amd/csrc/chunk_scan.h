// chunk_scan.h — portions of prompts through a recurrence with a matrix state per head, sixteen tokens at a time
// (chunk_scan.hip); the entries of state_scan.hip and gated_recurrence.hip choose it.
#pragma once
#include "hx_common.h"

namespace hxm {

enum ChunkForm {
  kChunkDecay = 0,        // S <- a S + k (s v)^T;  o = S^T q
  kChunkDelta = 1,        // S <- a S;  S <- S + k (b (v - S^T k))^T;  o = S^T q       (a one per head)
  kChunkBonus = 2,        // o = (S + diag(u) k v^T)^T q;  S <- diag(a) S + k v^T      (a one per key channel)
  kChunkGated = 3,        // f = low + (1 - low) sigmoid(k + f_bias), S <- diag(f) S + (1 - f) v^T, o = S^T silu(q)
};

struct ChunkScanArgs {
  float* out;             // [n_tokens][heads * V]
  const void *q, *k, *v;
  int64_t q_stride, k_stride, v_stride;
  int32_t q_dtype, k_dtype, v_dtype;      // HX_F32 or HX_BF16
  int32_t form, per_channel;              // per_channel: decay [n_tokens][heads * K], else [n_tokens][heads]
  const float *decay, *vscale, *beta, *bonus, *f_bias, *low;
  float* state;
  int64_t slot_stride;
  const int32_t *slots, *q_cu, *positions;
  int32_t n_seq, heads, qk_heads, K, V;
  int64_t n_tokens;
  int32_t longest;        // the longest portion, 0: not known
  float* made;            // chunk_scan_workspace floats on a multiple of 16 bytes: what chunks need is made in a launch ahead; or NULL
  int32_t segment;        // chunk_chain.hip's own: chunks a segment of a portion (0: a portion is one chain), and what the segments leave for each other
  float* segments;
};

// true if chunk_scan serves these sizes
bool chunk_scan_fits(const ChunkScanArgs& a);
// floats of workspace with which it goes faster; 0: none
int64_t chunk_scan_workspace(const ChunkScanArgs& a);
int chunk_scan(const ChunkScanArgs& a, hipStream_t s);
int chunk_chain(const ChunkScanArgs& a, hipStream_t s);      // with a.made
int chunk_head(const ChunkScanArgs& a, hipStream_t s);       // one decay per token and head, without it: the delta rule with more than 64 key channels, the decayed sum of bfloat16 q and k

}  // namespace hxm
