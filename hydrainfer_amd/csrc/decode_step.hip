// decode_step.hip — a layer of a decode step issued by one call: the launches of hx_linear_decode_ex, hx_decode_attention_fused,
// hx_norm_gate_up_silu_xreg, hx_norm_linear_decode_xreg and hx_add_rms_norm_slabs_ex in the order in which a caller would issue them
// (and recorded in a launch plan as theirs).  One row through four layers of width 2048 is 195 us of kernels, and 26 calls from Python
// took 265 us (8 - 10 us each, of which 3 are the launch); this way 199.  A layer a call and not all of them: the first layer runs while
// the caller fills in the next one's arguments.
#include "hx_common.h"

extern "C" int hx_decode_layer_step(const hx_decode_layer* layer, int32_t qkv_slabs, hx_stream stream) {
  if (!layer) return HX_ERR_NULL;
  const hx_decode_layer& a = *layer;
  if (!a.h || !a.x || !a.x_frag || !a.act || !a.ws || !a.ws_qkv || !a.sync) return HX_ERR_NULL;
  if (qkv_slabs < 1) return HX_ERR_SHAPE;
  hx_fused_decode_args fused = a.fused;
  fused.qkv_partial = a.ws_qkv;
  fused.qkv_splits = qkv_slabs;
  int rc = hx_decode_attention_fused(&a.attn, &fused, stream);
  if (rc != HX_OK) return rc;
  int slabs = hx_linear_decode_ex(a.ws, a.ws_bytes, a.attn.out, (int64_t)a.attn.n_heads * a.attn.head_dim, 0, &a.o, a.rows, stream);
  if (slabs < 0) return slabs;
  rc = hx_norm_gate_up_silu_xreg(a.act, a.h, a.ws, slabs, a.norm_mlp, a.epsilon, a.x_frag, a.gate_up, a.rows, a.inter, a.hidden, a.sync, a.dtype, stream);
  if (rc != HX_OK) return rc;
  slabs = hx_linear_decode_ex(a.ws, a.ws_bytes, a.act, a.inter, 1, &a.down, a.rows, stream);
  if (slabs < 0) return slabs;
  const hx_decode_weight& next = a.next_qkv;
  if (!next.packed) return hx_add_rms_norm_slabs_ex(a.x, a.h, a.ws, slabs, a.norm_next, a.epsilon, a.rows, a.hidden, a.dtype, 0, stream);
  if (a.norm_in_qkv)
    return hx_norm_linear_decode_xreg(a.ws_qkv, a.h, a.ws, slabs, a.norm_next, a.epsilon, a.x_frag, next.packed, a.rows, next.N, next.K,
                                      a.sync + HX_XREG_SYNC_WORDS, a.ws_qkv_bytes, a.dtype, stream);
  rc = hx_add_rms_norm_slabs_ex(a.x_frag, a.h, a.ws, slabs, a.norm_next, a.epsilon, a.rows, a.hidden, a.dtype, 1, stream);
  return rc != HX_OK ? rc : hx_linear_decode_ex(a.ws_qkv, a.ws_qkv_bytes, a.x_frag, a.hidden, 1, &next, a.rows, stream);
}
