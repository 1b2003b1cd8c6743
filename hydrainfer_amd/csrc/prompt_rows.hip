// prompt_rows.hip — the rows of a batch of prompts that are sampled, taken out in front of the last layer's queries (extends
// hydrainfer/model/model_forward.py, where they are taken out in front of its feed-forward): behind that layer's keys and values no other row is used.
#include "hx_common.h"
#include "../../include/hydra_hip.h"

namespace hx {
namespace {

struct PromptRows {
  const void* rows;               // [n] int32 or int64; negative ones count from the end
  int32_t wide, n, n_tokens, n_seq;
  const int32_t *q_cu, *kv_cu, *cu_blocks, *positions;
  const u16 *x, *h;
  u16 *x_out, *h_out;
  int32_t row_bytes;
  int32_t *position_out, *q_cu_out, *kv_cu_out, *cu_blocks_out;
};

__device__ __forceinline__ int prompt_row(const PromptRows& p, int i) {
  const int64_t r = p.wide ? ((const int64_t*)p.rows)[i] : ((const int32_t*)p.rows)[i];
  const int64_t at = r < 0 ? r + p.n_tokens : r;
  return (int)(at < 0 ? 0 : at >= p.n_tokens ? p.n_tokens - 1 : at);
}

// Workgroup i < n: row i of both; the last one: each row as a sequence of one query, with the keys that it sees.
__global__ __launch_bounds__(256) void prompt_rows_kernel(PromptRows p) {
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < p.n) {
    const int64_t from = (int64_t)prompt_row(p, blockIdx.x) * p.row_bytes, to = (int64_t)blockIdx.x * p.row_bytes;
    for (int c = 16 * tid; c < p.row_bytes; c += 16 * 256) {
      *reinterpret_cast<u32x4*>((char*)p.x_out + to + c) = *reinterpret_cast<const u32x4*>((const char*)p.x + from + c);
      *reinterpret_cast<u32x4*>((char*)p.h_out + to + c) = *reinterpret_cast<const u32x4*>((const char*)p.h + from + c);
    }
    return;
  }
  __shared__ int32_t sums[4];
  int32_t run = 0;                // keys of the rows in front
  for (int i0 = 0; i0 < p.n; i0 += 256) {
    const int i = i0 + tid;
    int32_t keys = 0;
    if (i < p.n) {
      const int r = prompt_row(p, i);
      int lo = 0, hi = p.n_seq - 1;                        // the last sequence that starts at or before row r
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (p.q_cu[mid] <= r) lo = mid;
        else hi = mid - 1;
      }
      keys = p.kv_cu[lo + 1] - p.kv_cu[lo] - (p.q_cu[lo + 1] - 1 - r);
      p.position_out[i] = p.positions[r];
      p.q_cu_out[i] = i;
      p.cu_blocks_out[i] = p.cu_blocks[lo];
    }
    int32_t up_to = keys;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t v = __shfl_up(up_to, d, 64);
      if ((tid & 63) >= d) up_to += v;
    }
    if ((tid & 63) == 63) sums[tid >> 6] = up_to;
    __syncthreads();
    for (int w = 0; w < 4; ++w) {
      if (w < tid >> 6) up_to += sums[w];
    }
    if (i < p.n) p.kv_cu_out[i] = run + up_to - keys;
    run += sums[0] + sums[1] + sums[2] + sums[3];
    __syncthreads();
  }
  if (tid == 0) {
    p.q_cu_out[p.n] = p.n;
    p.kv_cu_out[p.n] = run;
    p.cu_blocks_out[p.n] = p.cu_blocks[p.n_seq];
  }
}

}  // namespace
}  // namespace hx

using namespace hx;

extern "C" int hx_prompt_rows(const void* rows, int32_t rows_are_int64, int64_t n, int64_t n_tokens, int64_t n_seq, const int32_t* q_cu, const int32_t* kv_cu, const int32_t* cu_blocks,
                              const int32_t* positions, const void* x, const void* h, void* x_out, void* h_out, int64_t row_bytes, int32_t* tables, hx_stream stream) {
  if (n < 0 || n > 65535 || n_tokens < 1 || n_tokens > INT32_MAX || n_seq < 1 || n_seq > 65535 || row_bytes < 16 || row_bytes % 16 || row_bytes > (1 << 20)) return HX_ERR_SHAPE;
  if (n == 0) return HX_OK;
  if (!rows || !q_cu || !kv_cu || !cu_blocks || !positions || !x || !h || !x_out || !h_out || !tables) return HX_ERR_NULL;
  if (!aligned16(x) || !aligned16(h) || !aligned16(x_out) || !aligned16(h_out)) return HX_ERR_STRIDE;
  PromptRows p;
  p.rows = rows; p.wide = rows_are_int64 != 0; p.n = (int32_t)n; p.n_tokens = (int32_t)n_tokens; p.n_seq = (int32_t)n_seq;
  p.q_cu = q_cu; p.kv_cu = kv_cu; p.cu_blocks = cu_blocks; p.positions = positions;
  p.x = (const u16*)x; p.h = (const u16*)h; p.x_out = (u16*)x_out; p.h_out = (u16*)h_out; p.row_bytes = (int32_t)row_bytes;
  p.q_cu_out = tables; p.kv_cu_out = tables + (n + 1); p.cu_blocks_out = tables + 2 * (n + 1); p.position_out = tables + 3 * (n + 1);
  hx::launcher(prompt_rows_kernel, dim3((unsigned)(n + 1)), dim3(256), 0, (hipStream_t)stream)(p);
  return check_launch();
}

namespace {

// The scratch of a last layer, in the order in which it is laid out.
struct LastLayerScratch {
  int32_t* tables;
  char *h, *q, *o, *act, *sums, *attn;
  int64_t sums_bytes, attn_bytes, bytes;
};

int64_t most(int64_t a, int64_t b) { return a > b ? a : b; }

// The layer's attention: the sampled rows as sequences of one query; the tables as hx_prompt_rows leaves them.
hx_attn_args last_attention(const hx_prompt_last& a, const LastLayerScratch& s) {
  hx_attn_args t = a.attn;
  const int64_t width = (int64_t)t.n_heads * t.head_dim;
  t.q = s.q; t.out = s.o;
  t.cu_seqlens_q = s.tables; t.cu_seqlens_k = s.tables + (a.n + 1); t.cu_block_lens = s.tables + 2 * (a.n + 1);
  t.batch = t.total_q = (int32_t)a.n;
  t.max_seqlen_q = 1;
  t.q_row_stride = t.o_row_stride = width;
  t.workspace = s.attn_bytes ? s.attn : nullptr;
  t.workspace_bytes = s.attn_bytes;
  return t;
}

int lay_out(const hx_prompt_last& a, LastLayerScratch* s) {
  const int64_t n = a.n, width = (int64_t)a.attn.n_heads * a.attn.head_dim;
  if (n < 1 || n > 64 || a.hidden < 256 || a.hidden % 256 || a.inter < 256 || a.inter % 256 || width < 256 || width % 256) return HX_ERR_SHAPE;
  if (a.attn.dtype != HX_F16 && a.attn.dtype != HX_BF16) return HX_ERR_DTYPE;
  if (a.attn.n_kv_heads < 1 || a.attn.n_heads % a.attn.n_kv_heads || !a.attn.block_table) return HX_ERR_SHAPE;
  char* const base = a.scratch ? (char*)a.scratch : (char*)256;       // (where only the size is asked for, addresses that are not null)
  char* at = base;
  auto take = [&](int64_t bytes) { char* p = at; at += (bytes + 255) / 256 * 256; return p; };
  s->tables = (int32_t*)take(4 * (4 * n + 3));
  s->h = take(2 * n * a.hidden);
  s->q = take(2 * n * width);
  s->o = take(2 * n * width);
  s->act = take(2 * n * a.inter);
  s->sums_bytes = most(most(hx_linear_decode_workspace_bytes(n, width, a.hidden), hx_linear_decode_workspace_bytes(n, a.hidden, width)),
                       most(hx_linear_decode_workspace_bytes(n, 2 * a.inter, a.hidden), hx_linear_decode_workspace_bytes(n, a.hidden, a.inter)));
  s->sums = take(s->sums_bytes);
  s->attn_bytes = 0;
  const hx_attn_args t = last_attention(a, *s);
  s->attn_bytes = hx_mha_varlen_fwd_workspace_bytes(&t);
  if (s->attn_bytes < 0) return (int)s->attn_bytes;
  s->attn = take(s->attn_bytes);
  s->bytes = at - base;
  return HX_OK;
}

}  // namespace

extern "C" int64_t hx_prompt_last_scratch_bytes(const hx_prompt_last* layer) {
  if (!layer) return HX_ERR_NULL;
  LastLayerScratch s;
  const int rc = lay_out(*layer, &s);
  return rc != HX_OK ? rc : s.bytes;
}

// The layer's launches from one call: from Python each took 8 - 14 us of the caller.  300 tokens through one layer of width 2048, us a call: 198 with
// these launches issued from Python, 182 with all rows through the layer (fewer launches), 126 this way.
extern "C" int hx_prompt_last_layer(const hx_prompt_last* layer, hx_stream stream) {
  if (!layer) return HX_ERR_NULL;
  const hx_prompt_last& a = *layer;
  LastLayerScratch s;
  int rc = lay_out(a, &s);
  if (rc != HX_OK) return rc;
  if (!a.scratch || !a.kv || !a.wq || !a.wo || !a.w_gate_up || !a.w_down || !a.norm_mlp || !a.norm_next || !a.cos_sin || !a.new_cache_slots || !a.out) return HX_ERR_NULL;
  if (a.scratch_bytes < s.bytes) return HX_ERR_WORKSPACE;
  const hx_attn_args t = last_attention(a, s);
  const int dt = t.dtype;
  const int64_t n = a.n, D = t.head_dim, width = (int64_t)t.n_heads * D, keys = (int64_t)t.n_kv_heads * D;
  float* sums = (float*)s.sums;
  u16* kv = (u16*)a.kv;
  rc = hx_prompt_rows(a.rows, a.rows_are_int64, n, a.n_tokens, a.n_seq, a.attn.cu_seqlens_q, a.attn.cu_seqlens_k, a.attn.cu_block_lens, a.positions, a.x, a.h, a.out, s.h,
                      2 * a.hidden, s.tables, stream);
  if (rc != HX_OK) return rc;
  rc = hx_rope_set_kv_cache(kv, kv, kv + keys, a.positions, a.cos_sin, a.new_cache_slots, (void*)t.k, (void*)t.v, a.n_tokens, 0, t.n_kv_heads, D, D, 2 * keys,
                            2 * keys, 2 * keys, t.block_size, t.k_block_stride, t.v_block_stride, dt, stream);
  if (rc != HX_OK) return rc;
  rc = hx_linear_decode(s.q, a.out, a.wq, n, width, a.hidden, a.hidden, a.ld_wq, width, sums, s.sums_bytes, dt, stream);
  if (rc != HX_OK) return rc;
  rc = hx_apply_rotary_pos_emb(s.q, s.q, s.tables + 3 * (n + 1), a.cos_sin, n, t.n_heads, 0, D, D, width, width, 0, dt, stream);
  if (rc != HX_OK) return rc;
  rc = hx_mha_varlen_fwd(&t, stream);
  if (rc != HX_OK) return rc;
  int slabs = hx_linear_decode_partial(sums, s.o, a.wo, n, a.hidden, width, width, a.ld_wo, s.sums_bytes, dt, stream);
  if (slabs < 0) return slabs;
  rc = hx_add_rms_norm_slabs(a.out, s.h, sums, slabs, a.norm_mlp, a.epsilon, n, a.hidden, dt, stream);
  if (rc != HX_OK) return rc;
  slabs = hx_linear_decode_partial(sums, a.out, a.w_gate_up, n, 2 * a.inter, a.hidden, a.hidden, a.ld_gate_up, s.sums_bytes, dt, stream);
  if (slabs < 0) return slabs;
  rc = hx_silu_and_mul_slabs(s.act, sums, slabs, n, a.inter, dt, stream);
  if (rc != HX_OK) return rc;
  slabs = hx_linear_decode_partial(sums, s.act, a.w_down, n, a.hidden, a.inter, a.inter, a.ld_down, s.sums_bytes, dt, stream);
  if (slabs < 0) return slabs;
  return hx_add_rms_norm_slabs(a.out, s.h, sums, slabs, a.norm_next, a.epsilon, n, a.hidden, dt, stream);
}

namespace {

// The scratch of a layer of a few hundred rows.  false: some product of it is not made in the tiles of gemm_rows.hip.
struct LayerScratch {
  int o_splits, down_splits;
  char *o, *act, *sums, *attn;
  int64_t attn_bytes, bytes;
};
hx_attn_args layer_attention(const hx_prompt_layer& a, const LayerScratch& s) {
  hx_attn_args t = a.attn;
  t.q = a.qkv; t.out = s.o;
  t.total_q = (int32_t)a.n_tokens;
  t.q_row_stride = (int64_t)(t.n_heads + 2 * t.n_kv_heads) * t.head_dim;
  t.o_row_stride = (int64_t)t.n_heads * t.head_dim;
  t.workspace = s.attn_bytes ? s.attn : nullptr;
  t.workspace_bytes = s.attn_bytes;
  return t;
}
int lay_out(const hx_prompt_layer& a, LayerScratch* s) {
  const int64_t n = a.n_tokens, width = (int64_t)a.attn.n_heads * a.attn.head_dim;
  if (n < 1 || n > 1 << 20 || a.hidden < 1 || a.inter < 1 || width < 1 || a.attn.n_kv_heads < 1 || a.attn.n_heads % a.attn.n_kv_heads || a.attn.batch < 1) return HX_ERR_SHAPE;
  if (a.attn.dtype != HX_F16 && a.attn.dtype != HX_BF16) return HX_ERR_DTYPE;
  if (!a.attn.block_table) return HX_ERR_NULL;
  s->o_splits = hx_linear_rows_splits(n, a.hidden, width);
  s->down_splits = hx_linear_rows_splits(n, a.hidden, a.inter);
  if (s->o_splits < 1 || s->down_splits < 1 || hx_gate_up_silu_few_rows_supported(n, a.inter, a.hidden) != 1 || a.hidden < 128) return HX_ERR_UNSUPPORTED;
  char* const base = a.scratch ? (char*)a.scratch : (char*)256;       // (where only the size is asked for, addresses that are not null)
  char* at = base;
  auto take = [&](int64_t bytes) { char* p = at; at += (bytes + 255) / 256 * 256; return p; };
  auto sum_bytes = [&](int splits) { return n * a.hidden * (splits > 1 ? (int64_t)4 * splits : 2); };
  s->o = take(2 * n * width);
  s->act = take(2 * n * a.inter);
  s->sums = take(most(sum_bytes(s->o_splits), sum_bytes(s->down_splits)));
  s->attn_bytes = 0;
  const hx_attn_args t = layer_attention(a, *s);
  s->attn_bytes = hx_mha_varlen_fwd_workspace_bytes(&t);
  if (s->attn_bytes < 0) return (int)s->attn_bytes;
  s->attn = take(s->attn_bytes);
  s->bytes = at - base;
  return HX_OK;
}

// h += x w^T, out = rms_norm(h)
int product_add_norm(void* out, void* h, char* sums, int splits, const void* x, int64_t k, const void* w, int64_t ldw, const void* norm, const hx_prompt_layer& a, hx_stream stream) {
  const int dt = a.attn.dtype;
  int rc = hx_linear_rows(splits > 1 ? nullptr : sums, splits > 1 ? (float*)sums : nullptr, splits, x, w, a.n_tokens, a.hidden, k, k, ldw, dt, stream);
  if (rc != HX_OK) return rc;
  return splits > 1 ? hx_add_rms_norm_slabs(out, h, (const float*)sums, splits, norm, a.epsilon, a.n_tokens, a.hidden, dt, stream)
                    : hx_add_rms_norm(out, h, sums, norm, a.epsilon, a.n_tokens, a.hidden, dt, stream);
}

}  // namespace

extern "C" int64_t hx_prompt_layer_scratch_bytes(const hx_prompt_layer* layer) {
  if (!layer) return HX_ERR_NULL;
  LayerScratch s;
  const int rc = lay_out(*layer, &s);
  return rc != HX_OK ? rc : s.bytes;
}

// A layer's seven launches behind its qkv product from one call: from Python they take 75 us of the caller, more than the GPU needs for a hundred tokens of width 2048.  Issued
// from Python and this way, width 2048, us a call: two layers, 4 prompts of 23 - 106 tokens 218 188, one of 70 196 159, 3 of 60 - 200 201 199; six layers, 3 of 19 - 58 529 440, 3 of
// 60 - 200 617 617; width 4096, where the GPU bounds, 319 319.
extern "C" int hx_prompt_layer_step(const hx_prompt_layer* layer, hx_stream stream) {
  if (!layer) return HX_ERR_NULL;
  const hx_prompt_layer& a = *layer;
  LayerScratch s;
  int rc = lay_out(a, &s);
  if (rc != HX_OK) return rc;
  if (!a.scratch || !a.qkv || !a.x || !a.h || !a.wo || !a.w_gate_up || !a.w_down || !a.norm_mlp || !a.norm_next || !a.cos_sin || !a.positions || !a.new_cache_slots) return HX_ERR_NULL;
  if (a.scratch_bytes < s.bytes) return HX_ERR_WORKSPACE;
  const hx_attn_args t = layer_attention(a, s);
  const int dt = t.dtype;
  const int64_t n = a.n_tokens, D = t.head_dim, width = (int64_t)t.n_heads * D, keys = (int64_t)t.n_kv_heads * D, row = width + 2 * keys;
  u16* qkv = (u16*)a.qkv;
  rc = hx_rope_set_kv_cache(qkv, qkv + width, qkv + width + keys, a.positions, a.cos_sin, a.new_cache_slots, (void*)t.k, (void*)t.v, n, t.n_heads, t.n_kv_heads, D, D, row, row, row,
                            t.block_size, t.k_block_stride, t.v_block_stride, dt, stream);
  if (rc != HX_OK) return rc;
  rc = hx_mha_varlen_fwd(&t, stream);
  if (rc != HX_OK) return rc;
  rc = product_add_norm(a.x, a.h, s.sums, s.o_splits, s.o, width, a.wo, a.ld_wo, a.norm_mlp, a, stream);
  if (rc != HX_OK) return rc;
  rc = hx_gate_up_silu_rows(s.act, a.x, a.w_gate_up, n, a.inter, a.hidden, a.hidden, a.ld_gate_up, dt, stream);
  if (rc != HX_OK) return rc;
  return product_add_norm(a.x, a.h, s.sums, s.down_splits, s.act, a.inter, a.w_down, a.ld_down, a.norm_next, a, stream);
}
