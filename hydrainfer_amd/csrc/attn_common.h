// attn_common.h — MFMA wrappers and parameter block shared by the attention kernels.
#pragma once
#include "hx_common.h"

namespace hx {

template <typename T> struct Mfma;
template <> struct Mfma<F16> {
  // D[16x16] += A[16x32] * B[32x16]; lane l: A[row l&15][k 8(l>>4)+j], B[k 8(l>>4)+j][col l&15]
  static __device__ __forceinline__ f32x4 mma(u16x8 a, u16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma<BF16> {
  static __device__ __forceinline__ f32x4 mma(u16x8 a, u16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// ds_read_b64_tr_b16: lane (g = l>>4, c = l&15) of a [16 rows][16 cols] 2-byte tile whose rows
// start at lds_ptr(row-group base) receives column-major data suitable as an MFMA A operand of
// the transposed tile (see attn_fwd.hip for the addressing used with it).
typedef short hx_s16x4_t __attribute__((__vector_size__(4 * sizeof(short))));
__device__ __forceinline__ u16x4 lds_tr_read(const char* lds_ptr) {
  typedef __attribute__((address_space(3))) hx_s16x4_t lds_s4;
  hx_s16x4_t r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)lds_ptr);
  return __builtin_bit_cast(u16x4, r);
}

// Finite "minus infinity" for running maxima: keeps exp2(m_old - m_new) == 1 when a
// lane group has not seen any unmasked key yet (no NaN from inf - inf).
#define HX_NEG_BIG (-1.0e30f)

// key index -> (page slot in the block table, row inside the page)
__device__ __forceinline__ int page_slot(int key, int block_size, int block_shift) {
  return block_shift >= 0 ? key >> block_shift : key / block_size;
}
__device__ __forceinline__ int page_row(int key, int block_size, int block_shift) {
  return block_shift >= 0 ? key & (block_size - 1) : key % block_size;
}

// The least value over the wave, uniform (the vector ALU alone: four DPP steps and two swaps)
template <int CTRL>
__device__ __forceinline__ int dpp_int(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true); }
__device__ __forceinline__ int wave_min_int(int v) {
  v = min(v, dpp_int<0xB1>(v));       // lane ^ 1
  v = min(v, dpp_int<0x4E>(v));       // lane ^ 2
  v = min(v, dpp_int<0x141>(v));      // the half row's mirror image
  v = min(v, dpp_int<0x140>(v));      // the row's
  const auto a = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
  v = min((int)a[0], (int)a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
  return __builtin_amdgcn_readfirstlane(min((int)b[0], (int)b[1]));
}
__device__ __forceinline__ int wave_max_int(int v) { return -wave_min_int(-v); }

__device__ __forceinline__ float halves_max(float v) {      // with lane ^ 32, without the LDS crossbar
  const auto a = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  const unsigned a0 = a[0], a1 = a[1];
  return fmaxf(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1));
}
__device__ __forceinline__ float groups_max(float v) {      // over the four lanes with the same lane % 16
  const auto a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  const unsigned a0 = a[0], a1 = a[1];
  v = fmaxf(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1));
  const auto b = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  const unsigned b0 = b[0], b1 = b[1];
  return fmaxf(__builtin_bit_cast(float, b0), __builtin_bit_cast(float, b1));
}

// The slot-th (sequence, tile of TQ rows) pair of a batch whose sequences bring (cu[i + 1] - cu[i]) * per rows: sequences in groups of
// four, of every group the last tile of each — it sees the most keys —, then the one before it of each, ...; row tiles end with
// the portion, so that a partial tile is the first.  false: a spare slot.  Every lane counts one group's tiles: one round of loads
// for 256 sequences (walked a group at a time, a decode of 32 waited for eight).
template <int TQ, typename P>
__device__ __forceinline__ bool find_row_tile(P cu, int n_seq, int per, int slot, int& b, int& tile, int& q0, int& n_rows) {
  const int lane = threadIdx.x & 63;
  for (int base = 0; base < n_seq; base += 256) {
    int cq[5], tl[4], upto = 0, most = 0;
#pragma unroll
    for (int i = 0; i < 5; ++i) cq[i] = cu[min(base + 4 * lane + i, n_seq)];
#pragma unroll
    for (int i = 0; i < 4; ++i) upto += ((cq[i + 1] - cq[i]) * per + TQ - 1) / TQ;      // (0 past the last sequence: its offsets repeat)
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(upto, off, 64);
      if (lane >= off) upto += v;
    }
    const uint64_t past = __builtin_amdgcn_ballot_w64(upto > slot);
    if (!past) { slot -= __builtin_amdgcn_readlane(upto, 63); continue; }
    const int at = __builtin_ctzll(past), g0 = base + 4 * at;
    if (at > 0) slot -= __builtin_amdgcn_readlane(upto, at - 1);
#pragma unroll
    for (int i = 0; i < 5; ++i) cq[i] = __builtin_amdgcn_readlane(cq[i], at);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      tl[i] = ((cq[i + 1] - cq[i]) * per + TQ - 1) / TQ;
      most = max(most, tl[i]);
    }
    // the last rank with at most `slot` tiles in front of it (walked rank by rank a prompt's hundreds took microseconds)
    auto before = [&](int rank) { return (min(tl[0], rank) + min(tl[1], rank)) + (min(tl[2], rank) + min(tl[3], rank)); };
    int lo = 0, hi = most;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (before(mid) <= slot) lo = mid;
      else hi = mid;
    }
    // (turned from rank to rank: dealt round robin, the eight XCDs would else keep a sequence each, long or short)
    const int there = (tl[0] > lo) + (tl[1] > lo) + (tl[2] > lo) + (tl[3] > lo);
    slot = (slot - before(lo) + (lo >> 1)) % there;
    b = -1;
    tile = q0 = n_rows = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (b < 0 && tl[i] > lo) {
        if (slot == 0) {
          b = g0 + i;
          tile = tl[i] - 1 - lo;
          q0 = cq[i];
          n_rows = (cq[i + 1] - cq[i]) * per;
        }
        --slot;
      }
    }
    b = __builtin_amdgcn_readfirstlane(b);
    return true;
  }
  return false;
}

struct AttnParams {
  void* out;
  const void* q;
  const void* k;
  const void* v;
  const int32_t* cu_q;
  const int32_t* cu_k;
  const int32_t* block_table;
  const int32_t* cu_block_lens;
  int64_t q_row_stride, o_row_stride;
  int64_t k_block_stride, k_row_stride, k_head_stride;
  int64_t v_block_stride, v_row_stride, v_head_stride;
  int32_t n_heads, group;   // group = n_heads / n_kv_heads
  int32_t batch;            // number of sequences
  int64_t total_q;          // query rows over all sequences
  int32_t block_size;       // paged: tokens per page (multiple of 16)
  int32_t block_shift;      // log2(block_size) when it is a power of two, else -1 (runtime integer
                            // division costs ~30 VALU instructions; the kernels do two per key row)
  int32_t causal;
  int32_t window_left, window_right;   // local attention (general kernel only): -1 = unbounded
  float softcap_scale;                 // softmax_scale / softcap when softcap > 0 (then scale_log2 = softcap * log2 e), else 0
  int32_t xcd_remap;        // prefill kernel: renumber workgroups so that one head's query tiles share an XCD
  int32_t wg_priority;      // prefill kernel (32x32 form): the two workgroups of a CU run at different priorities
  unsigned long long* stamps;   // EXPERIMENTS builds: time stamps of the persistent prefill kernel (null otherwise)
  int32_t max_seqlen_k;     // the caller's bound on a sequence's keys (host side: chooses between the forms of the prefill kernel)
  int32_t cu_pairing;       // prefill kernel, persistent form: the second workgroup of a CU takes a round's items from the short end
  int32_t unit_mode;        // prefill kernel, persistent form: deal units (the k-th longest + k-th shortest tile of a sequence)
  int32_t seq_group;        // prefill kernel, persistent form: sequences per deal group, 1 / 2 / 4 (set by its launcher)
  int32_t n_cus;            // prefill kernel, persistent form: CUs of the device (set by its launcher)
  int32_t n_tile_slots;     // prefill kernel, persistent form: upper bound of the (sequence, query tile) pairs (set by its launcher)
  float scale_log2;         // softmax_scale * log2(e)
  int32_t n_splits;
  float* ws_o;              // [batch, n_heads, n_splits, D] unnormalised partial outputs
  float* ws_ml;             // [batch, n_heads, n_splits, 2] (max, sum)
  // fused RoPE + cache append (decode only; all null/0 otherwise)
  const void* k_new;        // [batch, n_kv_heads, D] un-rotated key of the new token
  const void* v_new;        // [batch, n_kv_heads, D]
  int64_t kn_row_stride, vn_row_stride;
  const int32_t* positions; // [batch] rotary position of the new token
  const void* cos_sin;      // [max_pos, 2, D/2] in T
  const int32_t* new_slots; // [batch] cache slot of the new token
  // optional: q / k_new / v_new arrive as split-K fp32 slabs of the fused qkv projection
  const float* qkv_partial; // [n_splits][batch][(n_heads + 2*n_kv_heads) * D]
  int32_t qkv_splits;
  int64_t qkv_slab_stride;  // batch * row length
  int64_t qkv_row;          // (n_heads + 2*n_kv_heads) * D
  const int32_t* rank_desc; // decode kernel, RANKED form: [0] ragged?, [1 + r] the sequence with the r-th most keys (null: static grid)
};

}  // namespace hx
