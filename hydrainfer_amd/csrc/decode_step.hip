// decode_step.hip — the layers of a decode step issued by one call: the launches of hx_linear_decode_ex, hx_decode_attention_fused,
// hx_norm_gate_up_silu_xreg, hx_norm_linear_decode_xreg and hx_add_rms_norm_slabs_ex in the order in which a caller would issue them
// (and recorded in a launch plan as theirs).  One row through four layers of width 2048 is 210 us of kernels, and 26 calls from Python
// took 270 us (8 - 10 us each, of which 3 are the launch); this way 221.
#include "hx_common.h"

extern "C" int64_t hx_decode_layers_workspace_bytes(const hx_decode_layer* layers, int32_t n_layers) {
  int64_t bytes = 0;
  for (int32_t l = 0; layers && l < n_layers; ++l) {
    const int64_t b = hx_mha_varlen_fwd_workspace_bytes(&layers[l].attn);
    if (b < 0) return b;
    bytes = b > bytes ? b : bytes;
  }
  return bytes;
}

extern "C" int hx_decode_layers(const hx_decode_layers_args* args, const hx_decode_layer* layers, int32_t n_layers, hx_stream stream) {
  if (!args || !layers) return HX_ERR_NULL;
  const hx_decode_layers_args& a = *args;
  if (n_layers < 1) return HX_ERR_SHAPE;
  if (!a.h || !a.x || !a.x_frag || !a.act || !a.ws || !a.ws_qkv || !a.sync) return HX_ERR_NULL;
  int slabs = hx_linear_decode_ex(a.ws_qkv, a.ws_qkv_bytes, a.x, a.hidden, 0, &layers[0].qkv, a.rows, stream);
  if (slabs < 0) return slabs;
  for (int32_t l = 0; l < n_layers; ++l) {
    const hx_decode_layer& L = layers[l];
    int32_t* sync = a.sync + (int64_t)l * 2 * HX_XREG_SYNC_WORDS;
    hx_fused_decode_args fused = L.fused;
    fused.qkv_partial = a.ws_qkv;
    fused.qkv_splits = slabs;
    int rc = hx_decode_attention_fused(&L.attn, &fused, stream);
    if (rc != HX_OK) return rc;
    slabs = hx_linear_decode_ex(a.ws, a.ws_bytes, L.attn.out, (int64_t)L.attn.n_heads * L.attn.head_dim, 0, &L.o, a.rows, stream);
    if (slabs < 0) return slabs;
    rc = hx_norm_gate_up_silu_xreg(a.act, a.h, a.ws, slabs, L.norm_mlp, a.epsilon, a.x_frag, L.gate_up, a.rows, a.inter, a.hidden, sync, a.dtype, stream);
    if (rc != HX_OK) return rc;
    slabs = hx_linear_decode_ex(a.ws, a.ws_bytes, a.act, a.inter, 1, &L.down, a.rows, stream);
    if (slabs < 0) return slabs;
    if (l + 1 == n_layers) return hx_add_rms_norm_slabs_ex(a.x, a.h, a.ws, slabs, L.norm_next, a.epsilon, a.rows, a.hidden, a.dtype, 0, stream);
    const hx_decode_weight& next = layers[l + 1].qkv;
    if (a.norm_in_qkv) {
      slabs = hx_norm_linear_decode_xreg(a.ws_qkv, a.h, a.ws, slabs, L.norm_next, a.epsilon, a.x_frag, next.packed, a.rows, next.N, next.K,
                                         sync + HX_XREG_SYNC_WORDS, a.ws_qkv_bytes, a.dtype, stream);
    } else {
      rc = hx_add_rms_norm_slabs_ex(a.x_frag, a.h, a.ws, slabs, L.norm_next, a.epsilon, a.rows, a.hidden, a.dtype, 1, stream);
      if (rc != HX_OK) return rc;
      slabs = hx_linear_decode_ex(a.ws_qkv, a.ws_qkv_bytes, a.x_frag, a.hidden, 1, &next, a.rows, stream);
    }
    if (slabs < 0) return slabs;
  }
  return HX_OK;
}
