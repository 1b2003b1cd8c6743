"""The mixers' calls by way of csrc/front.cpp give what they give in Python (the same library, the same bytes), with every optional operand and
without, as views, with splits and workspaces and without; and what Python refuses is refused by the same words."""
from unittest import mock

import pytest
import torch

pytestmark = pytest.mark.gpu
BLOCK = 16


def both(f):
    """f() by way of the native side, and with something else in the library's place, which goes through Python alone."""
    from hydrainfer_amd import _lib
    lib = _lib.mix_lib()

    class StandIn:
        def __getattr__(self, name):
            return getattr(lib, name)

    calls = mock.Mock(wraps=_lib._front)
    with mock.patch.object(_lib, "_front", calls):
        native = f()
        assert calls.method_calls
        taken = len(calls.method_calls)
        with mock.patch.object(_lib, "_mix", StandIn()):
            plain = f()
        assert len(calls.method_calls) == taken
    native, plain = ([r] if isinstance(r, torch.Tensor) else list(r) for r in (native, plain))
    assert len(native) == len(plain)
    for a, b in zip(native, plain):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)


def batch(new, kv):
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    nb = [(n + BLOCK - 1) // BLOCK for n in kv]
    cu = lambda v: i([sum(v[:s]) for s in range(len(v) + 1)])
    seq = [s for s, n in enumerate(new) for _ in range(n)]
    pos = [p for n, k in zip(new, kv) for p in range(k - n, k)]
    return dict(seq=i(seq), pos=i(pos), q_cu=cu(new), table=i(list(range(sum(nb)))), blocks=cu(nb), n_blocks=sum(nb))


def rand(*shape, dtype=torch.bfloat16):
    return torch.randn(shape, device="cuda").to(dtype)


@pytest.mark.parametrize("new, kv", [([1, 1, 1], [700, 3, 50]), ([20, 1], [20, 300])])
@pytest.mark.parametrize("extra", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_attention(new, kv, extra, dtype):
    from hydrainfer_amd._C.kernel.biased_attn import biased_attention
    from hydrainfer_amd._C.kernel.latent_attn import latent_attention
    torch.manual_seed(1)
    b, T, H = batch(new, kv), sum(new), 8
    q, cache, sinks, gate = rand(H, T, 128, dtype=dtype).transpose(0, 1), rand(b["n_blocks"], BLOCK, 1, 136, dtype=dtype), rand(H, dtype=torch.float32), rand(T, H + 3, dtype=dtype)
    out = torch.empty((T, H, 128), dtype=dtype, device="cuda")
    both(lambda: latent_attention(q, cache, b["seq"], b["pos"], b["q_cu"], b["table"], b["blocks"], 0.1, 300 if extra else None, max(new),
                                  max_kv_len=max(kv), **(dict(gate_pre=gate, sinks=sinks, out=out) if extra else {})).clone())
    q, k, v = rand(T, H, 64, dtype=dtype), rand(b["n_blocks"], BLOCK, 4, 64, dtype=dtype), rand(b["n_blocks"], BLOCK, 4, 64, dtype=dtype)
    more = dict(slopes=sinks.abs(), mask="window", mask_size=200, softcap=30, head_scale=sinks.abs() + 1, sinks=sinks, kv_heads=2) if extra else {}
    both(lambda: biased_attention(q, k, v, 64, b["seq"], b["pos"], b["q_cu"], b["table"], b["blocks"], 0.125, max_q_len=max(new), max_kv_len=max(kv), **more))


@pytest.mark.parametrize("lens", [[1, 1, 1], [400, 3, 150]])
@pytest.mark.parametrize("mode", ["decay", "bonus", "delta"])
def test_recurrences(lens, mode):
    from hydrainfer_amd._C.kernel.recurrence import gated_recurrence
    from hydrainfer_amd._C.kernel.seq_mix import state_scan
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    torch.manual_seed(2)
    b, T, H, G, K, V, f32 = batch(lens, lens), sum(lens), 4, 2, 64, 32, torch.float32
    qk, decay = rand(T, 2 * G * K), torch.rand((T, H), device="cuda")
    if mode == "bonus":
        decay = torch.rand((T, H * K), device="cuda")
    more = dict(vscale=rand(T, H, dtype=f32), beta=torch.rand((T, H), device="cuda"), bonus=rand(H * K, dtype=f32))
    state = rand(5, 2, H * K * V + 8, dtype=f32)
    slots = torch.tensor([3, 0, 4], dtype=torch.int32, device="cuda")

    def scan():
        seq = SequenceState(state.clone(), slots, b["seq"])
        return state_scan(mode, qk[:, :G * K], qk[:, G * K:], rand_v, decay, seq, 12, b["q_cu"], b["pos"], H, G, K, V, **more), seq.state

    rand_v = rand(T, H * V, dtype=f32)
    both(scan)
    p = rand(T, H * (2 * K + V))

    def gated():
        seq = SequenceState(state.clone(), slots, b["seq"])
        return gated_recurrence(p[:, :H * K], p[:, H * K:2 * H * K], p[:, 2 * H * K:], more["bonus"], 0.9 * torch.sigmoid(more["bonus"]), rand_w, 1e-5, seq, 1,
                                b["q_cu"], b["pos"], H, K, V, max_q_len=max(lens)), seq.state

    rand_w = rand(V, dtype=f32)
    both(gated)


@pytest.mark.parametrize("T", [1, 300])
@pytest.mark.parametrize("act", ["none", "relu2", "glu"])
def test_experts(T, act):
    from hydrainfer_amd._C.kernel.moe_mix import grouped_linear, moe_combine, moe_plan, router_topk
    torch.manual_seed(3)
    E, W, top, f32 = 6, 64, 2, torch.float32
    x, w, bias = rand(T, W, dtype=f32), rand(E, W, dtype=f32), rand(E, dtype=f32)
    both(lambda: router_topk(x, w, bias if act == "glu" else None, top))
    weights, experts = router_topk(x, w, None, top)
    both(lambda: moe_plan(experts, E)[0])      # (the order of rows within an expert is nobody's)
    seg, row_of, src = moe_plan(experts, E)
    h, up = rand(T, W), rand(E, 96, W)
    both(lambda: grouped_linear(h, up, seg, T * top, src=src, act=act, limit=7.0, alpha=1.5, up_shift=1))
    y, shared, gate = rand(T * top, W), rand(T, W), rand(T, 3, dtype=f32)
    both(lambda: moe_combine(y, row_of, weights))
    both(lambda: moe_combine(y, row_of, weights, shared=shared, shared_gate=gate[:, 1], identity=h if act == "glu" else None))


def refused(call):
    """call() is refused, and by way of the native side in the words that Python has by itself."""
    from hydrainfer_amd import _lib
    lib = _lib.mix_lib()
    assert _lib.front() is not None

    class StandIn:
        def __getattr__(self, name):
            return getattr(lib, name)

    said = []
    for stand_in in (lib, StandIn()):
        with mock.patch.object(_lib, "_mix", stand_in), pytest.raises(Exception) as e:
            call()
        said.append((e.type, str(e.value)))
    assert said[0] == said[1] and issubclass(said[0][0], (_lib.HydraHipError, KeyError)), said


def test_what_is_refused_stays_refused():
    from hydrainfer_amd import _lib
    from hydrainfer_amd._C.kernel.latent_attn import latent_attention
    from hydrainfer_amd._C.kernel.moe_mix import grouped_linear, moe_combine, moe_plan, router_topk
    b = batch([1, 1], [20, 3])
    q, cache = rand(2, 4, 64), rand(b["n_blocks"], BLOCK, 1, 64)
    args = dict(q=q, cache=cache, tok_seq=b["seq"], positions=b["pos"], q_cu=b["q_cu"], block_table=b["table"], cu_block_lens=b["blocks"], scale=0.1, window=None,
                max_q_len=1)
    latent_attention(**args)
    for wrong in (dict(q=q.half(), cache=cache.half()), dict(cache=cache.float()), dict(tok_seq=b["seq"].long()), dict(positions=b["pos"][:1]), dict(q=q.transpose(1, 2)),
                  dict(cache=cache[..., :32]), dict(sinks=rand(4)), dict(gate_pre=rand(2, 3)), dict(out=rand(2, 4, 32)), dict(q=q.cpu()), dict(max_q_len=0)):
        with pytest.raises(_lib.HydraHipError):
            latent_attention(**{**args, **wrong})
        refused(lambda: latent_attention(**{**args, **wrong}))
    x, w = rand(2, 64, dtype=torch.float32), rand(4, 64, dtype=torch.float32)
    for call in (lambda: router_topk(x.bfloat16(), w, None, 2), lambda: router_topk(x, w, None, 9), lambda: moe_plan(b["seq"], 4), lambda: moe_plan(b["seq"][:, None].long(), 4),
                 lambda: grouped_linear(q[0], rand(1, 32, 64), b["q_cu"][:2], 9), lambda: moe_combine(q[0], b["seq"][:, None], x)):
        with pytest.raises(_lib.HydraHipError):
            call()
        refused(call)


def test_attention_refuses_in_the_same_words():
    from hydrainfer_amd._C.kernel.biased_attn import biased_attention
    b = batch([1, 1], [20, 3])
    q, k, v = rand(2, 8, 64), rand(b["n_blocks"], BLOCK, 4, 64), rand(b["n_blocks"], BLOCK, 4, 64)
    args = dict(q=q, key_cache=k, value_cache=v, vdim=64, tok_seq=b["seq"], positions=b["pos"], q_cu=b["q_cu"], block_table=b["table"], cu_block_lens=b["blocks"],
                scale=0.125, max_q_len=1, max_kv_len=20)
    biased_attention(**args)
    for wrong in (dict(q=q.float()), dict(q=q[:, :, :32]), dict(value_cache=v.float()), dict(value_cache=v.transpose(1, 2)), dict(kv_heads=3), dict(kv_heads=16), dict(vdim=65),
                  dict(vdim=0), dict(tok_seq=b["seq"][:1]), dict(positions=b["pos"].long()), dict(q_cu=b["q_cu"].float()), dict(block_table=b["table"].long()),
                  dict(cu_block_lens=b["blocks"][:2]), dict(slopes=rand(8)), dict(slopes=rand(7, dtype=torch.float32)), dict(head_scale=rand(8)),
                  dict(sinks=rand(16, dtype=torch.float32)[::2]), dict(mask="window"), dict(mask="none"), dict(mask="chunk", mask_size=-1), dict(form="other"), dict(q=q.cpu()),
                  dict(key_cache=k[:, :8], value_cache=v[:, :8]), dict(q=q.half(), key_cache=k.half(), value_cache=v.half())):
        refused(lambda: biased_attention(**{**args, **wrong}))


def test_recurrences_refuse_in_the_same_words():
    from hydrainfer_amd._C.kernel.recurrence import gated_recurrence
    from hydrainfer_amd._C.kernel.seq_mix import state_scan
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    b, T, H, G, K, V, f32 = batch([4, 3], [4, 3]), 7, 4, 2, 16, 8, torch.float32
    state, slots = rand(3, 2, H * K * V + 4, dtype=f32), torch.tensor([2, 0], dtype=torch.int32, device="cuda")
    seq = SequenceState(state, slots, b["seq"])
    other = lambda **x: SequenceState(**{**dict(state=state, slots=slots, tok_seq=b["seq"]), **x})
    q, k, v, decay, beta = rand(T, G * K), rand(T, G * K), rand(T, H * V), torch.rand((T, H), device="cuda"), torch.rand((T, H), device="cuda")
    args = dict(mode="delta", q=q, k=k, v=v, decay=decay, seq=seq, offset=4, q_cu=b["q_cu"], positions=b["pos"], heads=H, qk_heads=G, dim=K, vdim=V, beta=beta)
    state_scan(**args)
    for wrong in (dict(mode="other"), dict(beta=None), dict(mode="bonus"), dict(q=q.half()), dict(q=q[:, 1:]), dict(q=q.t().contiguous().t()), dict(k=k[:3]), dict(v=v[:, ::2]),
                  dict(decay=decay.bfloat16()), dict(decay=decay[:, :2]), dict(beta=beta[:2]), dict(vscale=rand(T, H)), dict(bonus=rand(H, dtype=f32)),
                  dict(offset=-1), dict(offset=2 * state.shape[2]), dict(q_cu=b["q_cu"].long()), dict(positions=b["pos"][:3]), dict(seq=other(slots=slots[:1])),
                  dict(seq=other(slots=slots.long())), dict(seq=other(tok_seq=b["seq"][:2])), dict(seq=other(state=state.bfloat16())), dict(seq=other(state=state[:, :, 1:])),
                  dict(seq=other(state=state.cpu())), dict(v=v.cpu()), dict(heads=3), dict(qk_heads=3), dict(dim=300)):
        refused(lambda: state_scan(**{**args, **wrong}))
    p, bias, low, norm = rand(T, H * (2 * K + V)), rand(H * K, dtype=f32), torch.rand(H * K, device="cuda"), rand(V, dtype=f32)
    args = dict(q_pre=p[:, :H * K], f_pre=p[:, H * K:2 * H * K], v=p[:, 2 * H * K:], f_bias=bias, low=low, norm_w=norm, eps=1e-5, seq=seq, state_row=1, q_cu=b["q_cu"],
                positions=b["pos"], heads=H, dim=K, vdim=V, max_q_len=4)
    gated_recurrence(**args)
    for wrong in (dict(q_pre=args["q_pre"].half()), dict(q_pre=args["q_pre"].float()), dict(f_pre=args["f_pre"][:, 1:]), dict(v=args["v"][:2]), dict(f_bias=bias.bfloat16()),
                  dict(low=low[1:]), dict(norm_w=norm[:3]), dict(state_row=2), dict(state_row=-1), dict(seq=other(state=state[:, :, :64].contiguous())),
                  dict(seq=other(state=state.double())), dict(seq=other(slots=slots[:1])), dict(q_cu=b["q_cu"].long()), dict(positions=b["pos"].long()), dict(positions=b["pos"][:2]),
                  dict(low=low.cpu()), dict(dim=17), dict(vdim=9)):
        refused(lambda: gated_recurrence(**{**args, **wrong}))


def test_experts_refuse_in_the_same_words():
    from hydrainfer_amd._C.kernel.moe_mix import grouped_linear, moe_combine, moe_plan, router_topk
    T, E, W, top, f32 = 5, 4, 64, 2, torch.float32
    x, w = rand(T, W, dtype=f32), rand(E, W, dtype=f32)
    weights, experts = router_topk(x, w, None, top)
    seg, row_of, src = moe_plan(experts, E)
    h, up, y = rand(T, W), rand(E, 96, W), rand(T * top, W)
    refused(lambda: router_topk(x[:, 1:], w, None, top))
    refused(lambda: router_topk(x, w.t(), None, top))
    refused(lambda: router_topk(x, w, rand(E), top))
    refused(lambda: router_topk(x, w, rand(E + 1, dtype=f32), top))
    refused(lambda: router_topk(x, w, None, E + 1))
    refused(lambda: moe_plan(experts.t(), E))
    refused(lambda: moe_plan(experts.long(), E))
    refused(lambda: moe_plan(experts.cpu(), E))
    for wrong in (dict(x=h.float()), dict(x=h[:, 1:]), dict(w=up.transpose(1, 2)), dict(seg=seg[1:]), dict(seg=seg.long()), dict(src=src[1:]), dict(src=src.long()), dict(src=None),
                  dict(act="other"), dict(act="glu", w=rand(E, 80, W)), dict(x=h.half(), w=up.half()), dict(x=h.cpu())):
        refused(lambda: grouped_linear(**{**dict(x=h, w=up, seg=seg, max_rows=T * top, src=src), **wrong}))
    for wrong in (dict(y=y.t()), dict(y=y.half()), dict(row_of=row_of.long()), dict(weights=weights.bfloat16()), dict(weights=weights[:, :1]), dict(shared=h[:3]), dict(shared=h.float()),
                  dict(shared=h, shared_gate=rand(T)), dict(shared=h, shared_gate=rand(T + 1, dtype=f32)), dict(identity=h[:3]), dict(identity=h[:, 1:]), dict(identity=h.float()),
                  dict(shared=h.cpu())):
        refused(lambda: moe_combine(**{**dict(y=y, row_of=row_of, weights=weights), **wrong}))
