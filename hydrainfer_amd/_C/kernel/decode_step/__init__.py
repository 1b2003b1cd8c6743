"""The layers of a decode step, each in one native call (csrc/decode_step.hip, hx_decode_layer_step): the launches that
gemm.linear_decode_ex, flash_attn.decode_attention_fused, gemm.norm_gate_up_silu_xreg, gemm.norm_linear_decode_xreg and
norm.add_rms_norm_slabs issue one by one, in the same order with the same arguments.  And layers of a batch of prompts (csrc/prompt_rows.hip)."""
import ctypes
from typing import Iterable, NamedTuple, Optional

import torch
from torch import Tensor

from hydrainfer_amd import _lib
from hydrainfer_amd._C.kernel.gemm import DecodeWeight, XREG_SYNC_WORDS, fragment_major_elems


class DecodeLayer(NamedTuple):
    key_cache: Tensor               # [n_blocks, block_size, kv_heads, head_dim]
    value_cache: Tensor
    new_cache_slots: Tensor         # int32 [rows], as are the next four (see flash_attn.decode_attention_fused)
    cu_seqlens_q: Tensor
    cu_seqlens_k: Tensor
    block_table: Tensor
    cu_block_lens: Tensor
    max_seqlen_k: int
    rank_desc: Optional[Tensor]
    next_qkv: Optional[DecodeWeight]      # of the next layer, xreg layout as is down
    o: DecodeWeight
    down: DecodeWeight
    gate_up: Tensor                 # pack_weight_xreg(W [2 * inter, hidden], interleave_halves=True)
    norm_mlp: Tensor                # [hidden]
    norm_next: Tensor               # [hidden]: the next layer's first norm, or the final one


def decode_layers(h: Tensor, x: Tensor, x_frag: Tensor, act: Tensor, ws: Tensor, ws_qkv: Tensor, sync: Tensor, inter: int, n_heads: int,
                  head_dim: int, positions: Tensor, cos_sin: Tensor, softmax_scale: float, epsilon: float, norm_in_qkv: bool, qkv_slabs: int,
                  layers: Iterable[DecodeLayer]) -> None:
    """h [rows <= 32, hidden] residual (updated); x [rows, hidden] receives the final norm's output; qkv_slabs of the first layer's qkv
    product stand in ws_qkv; x_frag, act: fragment-major scratch of hidden and inter; ws, ws_qkv: float32 slabs (two buffers with norm_in_qkv, the qkv
    product taking the norm of the layer before); sync: zeroed int32 [layers, 2, XREG_SYNC_WORDS].  layers may be a generator: the first
    layer runs while the caller puts the next one together."""
    _lib.require_gpu(h, x, x_frag, act, ws, ws_qkv, sync, positions, cos_sin)
    rows, hidden = h.shape
    dt = h.dtype
    if dt not in (torch.float16, torch.bfloat16) or cos_sin.dtype != dt or any(t.dtype != dt or not t.is_contiguous() for t in (h, x, x_frag, act)) or x.shape != h.shape \
            or x_frag.numel() < fragment_major_elems(rows, hidden) or act.numel() < fragment_major_elems(rows, inter):
        raise _lib.HydraHipError("decode_layers: h, x [rows, hidden] and fragment-major scratch, contiguous and of one dtype (fp16 / bf16)")
    if any(t.dtype != torch.float32 or not t.is_contiguous() for t in (ws, ws_qkv)) or (norm_in_qkv and ws.data_ptr() == ws_qkv.data_ptr()):
        raise _lib.HydraHipError("decode_layers: slabs must be contiguous float32, of their own for the qkv product that takes the norm")
    if sync.dtype != torch.int32 or not sync.is_contiguous():
        raise _lib.HydraHipError("decode_layers: sync must be [layers, 2, XREG_SYNC_WORDS] contiguous int32 (zeroed)")
    if positions.dtype != torch.int32 or not positions.is_contiguous() or positions.numel() < rows:
        raise _lib.HydraHipError("decode_layers: positions must be contiguous int32 [rows]")
    q_size = n_heads * head_dim
    o = torch.empty((rows, q_size), dtype=dt, device=h.device)
    lib, stream = _lib.lib(), _lib.current_stream()
    c = _lib.hx_decode_layer()
    a, f = c.attn, c.fused
    a.out = a.q = o.data_ptr()                                    # (q, k_new and v_new are read from the slabs)
    a.batch, a.n_heads, a.head_dim, a.max_seqlen_q, a.total_q = rows, n_heads, head_dim, 1, rows
    a.q_row_stride = a.o_row_stride = q_size
    a.softmax_scale, a.causal, a.dtype, a.window_left, a.window_right = float(softmax_scale), 1, _lib.dtype_code(h), -1, -1
    f.k_new = f.v_new = a.out
    f.k_new_row_stride = f.v_new_row_stride = q_size
    f.positions, f.cos_sin, f.rotary_dim = positions.data_ptr(), cos_sin.data_ptr(), head_dim
    c.h, c.x, c.x_frag, c.act, c.ws, c.ws_qkv = (t.data_ptr() for t in (h, x, x_frag, act, ws, ws_qkv))
    c.ws_bytes, c.ws_qkv_bytes, c.rows, c.hidden, c.inter = 4 * ws.numel(), 4 * ws_qkv.numel(), rows, hidden, inter
    c.epsilon, c.norm_in_qkv, c.dtype = float(epsilon), int(norm_in_qkv), a.dtype
    slabs, attn_ws, first_sync, no_weight = int(qkv_slabs), None, sync.data_ptr(), _lib.hx_decode_weight()
    for l, p in enumerate(layers):
        k, v, ints = p.key_cache, p.value_cache, p[2:7]
        if sync.numel() < (l + 1) * 2 * XREG_SYNC_WORDS:
            raise _lib.HydraHipError("decode_layers: sync has no words left for this layer")
        _lib.require_gpu(k, v, *ints, p.rank_desc, p.gate_up, p.norm_mlp, p.norm_next)
        if k.dtype != dt or v.dtype != dt or k.dim() != 4 or v.shape != k.shape:
            raise _lib.HydraHipError("decode_layers: caches [n_blocks, block_size, kv_heads, head_dim] of the activations' dtype")
        for t in ints:
            if t.dtype != torch.int32 or not t.is_contiguous():
                raise _lib.HydraHipError("decode_layers: slots, lengths and block tables must be contiguous int32")
        n_kv, nq = k.size(2), p.next_qkv
        qkv_n = (n_heads + 2 * n_kv) * head_dim
        if ws_qkv.numel() < slabs * rows * qkv_n:
            raise _lib.HydraHipError("decode_layers: ws_qkv must hold the qkv product's slabs")
        if p.cu_seqlens_q.numel() != rows + 1:
            raise _lib.HydraHipError("decode_layers needs exactly one query token per sequence")
        if p.rank_desc is not None and (p.rank_desc.dtype != torch.int32 or not p.rank_desc.is_contiguous() or p.rank_desc.numel() < rows + 1):
            raise _lib.HydraHipError("decode_layers: rank_desc must be a contiguous int32 device tensor [1 + rows]")
        if (p.o.N, p.o.K, p.down.N, p.down.K) != (hidden, q_size, hidden, inter) or (nq is not None and ((nq.N, nq.K) != (qkv_n, hidden) or nq.packed.dtype != dt)) \
                or p.o.packed.dtype != dt or p.down.packed.dtype != dt or p.gate_up.dtype != dt or p.gate_up.numel() != 2 * inter * hidden:
            raise _lib.HydraHipError("decode_layers: packed weights do not match the activations")
        for w in (p.norm_mlp, p.norm_next):
            if w.dtype != dt or w.numel() != hidden or not w.is_contiguous():
                raise _lib.HydraHipError("decode_layers: norm weights [hidden] of the activations' dtype")
        c.o, c.down, c.next_qkv = p.o.desc, p.down.desc, no_weight if nq is None else nq.desc
        c.gate_up, c.norm_mlp, c.norm_next = p.gate_up.data_ptr(), p.norm_mlp.data_ptr(), p.norm_next.data_ptr()
        c.sync = first_sync + 4 * 2 * XREG_SYNC_WORDS * l
        a.k, a.v, a.n_kv_heads, a.block_size, a.max_seqlen_k = k.data_ptr(), v.data_ptr(), n_kv, k.size(1), int(p.max_seqlen_k)
        a.k_block_stride, a.k_row_stride, a.k_head_stride = k.stride()[:3]
        a.v_block_stride, a.v_row_stride, a.v_head_stride = v.stride()[:3]
        f.new_cache_slots, a.cu_seqlens_q, a.cu_seqlens_k, a.block_table, a.cu_block_lens = (t.data_ptr() for t in ints)
        f.rank_desc = None if p.rank_desc is None else p.rank_desc.data_ptr()
        need = lib.hx_mha_varlen_fwd_workspace_bytes(ctypes.byref(a))
        if need > (0 if attn_ws is None else attn_ws.numel()):
            attn_ws = torch.empty(need, dtype=torch.uint8, device=h.device)
            a.workspace, a.workspace_bytes = attn_ws.data_ptr(), need
        slabs = lib.hx_decode_layer_step(ctypes.byref(c), slabs, stream)
        if slabs < 0:
            _lib.check(slabs, "decode_layers")


def prompt_last_layer(x: Tensor, h: Tensor, rows: Tensor, kv: Tensor, positions: Tensor, cos_sin: Tensor, key_cache: Tensor, value_cache: Tensor, new_cache_slots: Tensor,
                      cu_seqlens_q: Tensor, cu_seqlens_k: Tensor, block_table: Tensor, cu_block_lens: Tensor, max_seqlen_k: int, wq: Tensor, wo: Tensor,
                      w_gate_up: Tensor, w_down: Tensor, norm_mlp: Tensor, norm_next: Tensor, softmax_scale: float, epsilon: float) -> Tensor:
    """The last layer of a batch of prompts for the rows of x that are sampled (csrc/prompt_rows.hip): kv [n_tokens, keys | values] of x = norm1(h), unrotated,
    goes to the cache (kv's keys are rotated in place).  rms_norm(h[rows] + attention + feed-forward) * norm_next."""
    tensors = (x, h, rows, kv, positions, cos_sin, key_cache, value_cache, new_cache_slots, cu_seqlens_q, cu_seqlens_k, block_table, cu_block_lens, wq, wo, w_gate_up,
               w_down, norm_mlp, norm_next)
    _lib.require_gpu(*tensors)
    (n_tokens, hidden), n, n_kv, D, width, inter, dt = x.shape, rows.shape[0], key_cache.shape[2], key_cache.shape[3], wq.shape[0], w_down.shape[1], x.dtype
    if dt not in (torch.float16, torch.bfloat16) or any(t.dtype != dt for t in (h, kv, cos_sin, key_cache, value_cache, wq, wo, w_gate_up, w_down, norm_mlp, norm_next)):
        raise _lib.HydraHipError("prompt_last_layer: one dtype (fp16 / bf16)")
    if any(t.dtype != torch.int32 or not t.is_contiguous() for t in (positions, new_cache_slots, cu_seqlens_q, cu_seqlens_k, block_table, cu_block_lens)):
        raise _lib.HydraHipError("prompt_last_layer: positions, slots, lengths and block table must be contiguous int32")
    if rows.dim() != 1 or not 1 <= n <= 64 or rows.dtype not in (torch.int32, torch.int64) or any(not t.is_contiguous() for t in (rows, x, h, kv, cos_sin, norm_mlp, norm_next)):
        raise _lib.HydraHipError("prompt_last_layer: 1 to 64 rows, int32 or int64; rows, x, h, kv, cos_sin and norms contiguous")
    if h.shape != x.shape or kv.shape != (n_tokens, 2 * n_kv * D) or positions.numel() != n_tokens or new_cache_slots.numel() != n_tokens or value_cache.shape != key_cache.shape \
            or width % D or wq.shape[1] != hidden or wo.shape != (hidden, width) or w_gate_up.shape != (2 * inter, hidden) or w_down.shape != (hidden, inter) \
            or norm_mlp.numel() != hidden or norm_next.numel() != hidden or cu_seqlens_k.numel() != cu_seqlens_q.numel() or cu_block_lens.numel() < cu_seqlens_q.numel():
        raise _lib.HydraHipError("prompt_last_layer: shape mismatch")
    if any(t.stride(-1) != 1 for t in (wq, wo, w_gate_up, w_down)) or any(c.stride(3) != 1 or c.stride(2) != D or c.stride(1) != n_kv * D for c in (key_cache, value_cache)):
        raise _lib.HydraHipError("prompt_last_layer: rows of weights and of a cache block must be contiguous")
    out = torch.empty((n, hidden), dtype=dt, device=x.device)
    c = _lib.hx_prompt_last()
    a = c.attn
    a.k, a.v, a.block_size = key_cache.data_ptr(), value_cache.data_ptr(), key_cache.shape[1]
    a.k_block_stride, a.k_row_stride, a.k_head_stride = key_cache.stride()[:3]
    a.v_block_stride, a.v_row_stride, a.v_head_stride = value_cache.stride()[:3]
    a.cu_seqlens_q, a.cu_seqlens_k, a.block_table, a.cu_block_lens = (t.data_ptr() for t in (cu_seqlens_q, cu_seqlens_k, block_table, cu_block_lens))
    a.n_heads, a.n_kv_heads, a.head_dim, a.max_seqlen_k = width // D, n_kv, D, int(max_seqlen_k)
    a.softmax_scale, a.causal, a.dtype, a.window_left, a.window_right = float(softmax_scale), 1, _lib.dtype_code(x), -1, -1
    c.x, c.h, c.rows, c.kv, c.positions, c.cos_sin, c.new_cache_slots = (t.data_ptr() for t in (x, h, rows, kv, positions, cos_sin, new_cache_slots))
    c.wq, c.wo, c.w_gate_up, c.w_down, c.norm_mlp, c.norm_next, c.out = (t.data_ptr() for t in (wq, wo, w_gate_up, w_down, norm_mlp, norm_next, out))
    c.ld_wq, c.ld_wo, c.ld_gate_up, c.ld_down = wq.stride(0), wo.stride(0), w_gate_up.stride(0), w_down.stride(0)
    c.n, c.n_tokens, c.n_seq, c.hidden, c.inter = n, n_tokens, cu_seqlens_q.numel() - 1, hidden, inter
    c.epsilon, c.rows_are_int64 = float(epsilon), rows.dtype == torch.int64
    lib = _lib.lib()
    need = lib.hx_prompt_last_scratch_bytes(ctypes.byref(c))
    if need < 0:
        _lib.check(int(need), "prompt_last_layer")
    scratch = torch.empty(need, dtype=torch.uint8, device=x.device)
    c.scratch, c.scratch_bytes = scratch.data_ptr(), need
    _lib.check(lib.hx_prompt_last_layer(ctypes.byref(c), _lib.current_stream()), "prompt_last_layer")
    return out


def prompt_layer(x: Tensor, h: Tensor, qkv: Tensor, positions: Tensor, cos_sin: Tensor, key_cache: Tensor, value_cache: Tensor, new_cache_slots: Tensor, cu_seqlens_q: Tensor,
                 cu_seqlens_k: Tensor, block_table: Tensor, cu_block_lens: Tensor, max_seqlen_q: int, max_seqlen_k: int, n_heads: int, wo: Tensor, w_gate_up: Tensor, w_down: Tensor,
                 norm_mlp: Tensor, norm_next: Tensor, softmax_scale: float, epsilon: float) -> bool:
    """A layer of a batch of prompts behind its qkv product (csrc/prompt_rows.hip), in place: qkv [n_tokens, q | k | v] of x = norm1(h) is rotated, its keys and values go
    to the cache, h += attention and feed-forward, x = rms_norm(h) * norm_next.  False, and nothing done, where a product of it is left to a library."""
    _lib.require_gpu(x, h, qkv, positions, cos_sin, key_cache, value_cache, new_cache_slots, cu_seqlens_q, cu_seqlens_k, block_table, cu_block_lens, wo, w_gate_up, w_down, norm_mlp,
                     norm_next)
    (n, hidden), n_kv, D, inter, dt = x.shape, key_cache.shape[2], key_cache.shape[3], w_down.shape[1], x.dtype
    width = n_heads * D
    if dt not in (torch.float16, torch.bfloat16) or any(t.dtype != dt or not t.is_contiguous() for t in (x, h, qkv, cos_sin, norm_mlp, norm_next)) \
            or any(t.dtype != dt or t.stride(-1) != 1 for t in (key_cache, value_cache, wo, w_gate_up, w_down)):
        raise _lib.HydraHipError("prompt_layer: one dtype (fp16 / bf16); x, h, qkv, cos_sin, norms and rows of weights and caches contiguous")
    if any(t.dtype != torch.int32 or not t.is_contiguous() for t in (positions, new_cache_slots, cu_seqlens_q, cu_seqlens_k, block_table, cu_block_lens)):
        raise _lib.HydraHipError("prompt_layer: positions, slots, lengths and block table must be contiguous int32")
    if h.shape != x.shape or qkv.shape != (n, width + 2 * n_kv * D) or positions.numel() != n or new_cache_slots.numel() != n or value_cache.shape != key_cache.shape \
            or wo.shape != (hidden, width) or w_gate_up.shape != (2 * inter, hidden) or w_down.shape != (hidden, inter) or norm_mlp.numel() != hidden or norm_next.numel() != hidden \
            or cu_seqlens_q.numel() < 2 or cu_seqlens_k.numel() != cu_seqlens_q.numel() or cu_block_lens.numel() < cu_seqlens_q.numel() or D % 8 or D > 256 or key_cache.shape[1] % 16 \
            or any(c.stride(2) != D or c.stride(1) != n_kv * D for c in (key_cache, value_cache)):
        raise _lib.HydraHipError("prompt_layer: shape mismatch")
    c = _lib.hx_prompt_layer()
    a = c.attn
    a.k, a.v, a.block_size = key_cache.data_ptr(), value_cache.data_ptr(), key_cache.shape[1]
    a.k_block_stride, a.k_row_stride, a.k_head_stride = key_cache.stride()[:3]
    a.v_block_stride, a.v_row_stride, a.v_head_stride = value_cache.stride()[:3]
    a.cu_seqlens_q, a.cu_seqlens_k, a.block_table, a.cu_block_lens = cu_seqlens_q.data_ptr(), cu_seqlens_k.data_ptr(), block_table.data_ptr(), cu_block_lens.data_ptr()
    a.batch, a.n_heads, a.n_kv_heads, a.head_dim, a.max_seqlen_q, a.max_seqlen_k = cu_seqlens_q.numel() - 1, n_heads, n_kv, D, int(max_seqlen_q), int(max_seqlen_k)
    a.softmax_scale, a.causal, a.dtype, a.window_left, a.window_right = float(softmax_scale), 1, _lib.dtype_code(x), -1, -1
    c.positions, c.new_cache_slots, c.qkv, c.x, c.h, c.cos_sin = (t.data_ptr() for t in (positions, new_cache_slots, qkv, x, h, cos_sin))
    c.wo, c.w_gate_up, c.w_down, c.norm_mlp, c.norm_next = (t.data_ptr() for t in (wo, w_gate_up, w_down, norm_mlp, norm_next))
    c.n_tokens, c.hidden, c.inter, c.ld_wo, c.ld_gate_up, c.ld_down = n, hidden, inter, wo.stride(0), w_gate_up.stride(0), w_down.stride(0)
    c.epsilon = float(epsilon)
    lib = _lib.lib()
    need = lib.hx_prompt_layer_scratch_bytes(ctypes.byref(c))
    if need == _lib.HX_ERR_UNSUPPORTED:
        return False
    if need < 0:
        _lib.check(int(need), "prompt_layer")
    scratch = torch.empty(need, dtype=torch.uint8, device=x.device)
    c.scratch, c.scratch_bytes = scratch.data_ptr(), need
    _lib.check(lib.hx_prompt_layer_step(ctypes.byref(c), _lib.current_stream()), "prompt_layer")
    return True
