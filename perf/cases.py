"""The work that this framework is asked to do, as cases that can be timed and checked: steps and prompts of a Llama decoder,
and the mixers of the other model designs through their operators, each in both of its directions (a batch of prompts, a
batch of single tokens).  Sizes are those of this repository's configurations (widths of 2048, 4096 and 5120, heads of 64
and 128, latents of 64 to 512, 8 to 32 experts) with ragged batches, as a scheduler makes them."""
import math

import torch

BLOCK = 16                    # rows of a cache block
VOCAB = 32064
GLU_ALPHA, GLU_LIMIT = 1.702, 7.0
WIDTHS = {2048: (5632, 16), 4096: (11008, 32), 5120: (13824, 40)}      # width -> inner size, heads of 128


def listed():
    return [
        # one user, one token: a chat's next word from a small decoder.  Launches and latency count.
        dict(name="step_one", kind="step", width=2048, layers=4, rows=1, shortest=705, longest=705, dtype="bfloat16"),
        # the serving batch: 32 conversations of different lengths, four layers of a 7B decoder
        dict(name="step_32_ragged", kind="step", width=4096, layers=4, rows=32, shortest=131, longest=959, dtype="bfloat16"),
        # a batch of prompts under the scheduler's token budget, two layers of the same decoder
        dict(name="prompts_ragged", kind="prompts", width=4096, layers=2, rows=5, shortest=176, longest=901, dtype="bfloat16"),
        # grouped-query attention with a sink per head over the paged cache: prompts, and one token of 32 conversations
        dict(name="attend_prompts", kind="attend", step=False, rows=4, shortest=797, longest=1151, past=0, heads=32, kv_heads=8, dim=128,
             mask="causal", size=0, slopes=False, sinks=True, softcap=0.0),
        dict(name="attend_step", kind="attend", step=True, rows=32, shortest=1025, longest=2047, past=0, heads=32, kv_heads=8, dim=128,
             mask="causal", size=0, slopes=False, sinks=True, softcap=0.0),
        # attention over cached latents: prompts without a window, and one token of 32 conversations under a window
        dict(name="latent_prompts", kind="latent", step=False, rows=4, shortest=797, longest=1151, past=0, heads=32, rank=512, window=0,
             gate=True, sinks=False),
        dict(name="latent_step", kind="latent", step=True, rows=32, shortest=301, longest=1747, past=0, heads=32, rank=512, window=512,
             gate=False, sinks=True),
        # gated delta rule: prompts, some of them continued; state-space duality: one token of 32 conversations
        dict(name="delta_prompts", kind="scan", mode="delta", step=False, rows=4, shortest=797, longest=1151, heads=32, qk_heads=16, dim=128, vdim=128),
        dict(name="decay_step", kind="scan", mode="decay", step=True, rows=32, shortest=1, longest=1, heads=64, qk_heads=8, dim=128, vdim=64),
        # gated linear recurrence: prompts, some of them continued
        dict(name="recurrence_prompts", kind="recurrence", step=False, rows=4, shortest=797, longest=1151, heads=32, dim=128, vdim=128),
        # mixture of experts with a clamped gate and a router in float: a batch of prompts, and one token of 32 conversations
        dict(name="experts_prompts", kind="experts", tokens=3989, width=4096, inner=2752, experts=16, top=4),
        dict(name="experts_step", kind="experts", tokens=32, width=4096, inner=2752, experts=16, top=4),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _two(rng, lo, hi):
    a, b = _log_int(rng, lo, hi), _log_int(rng, lo, hi)
    return min(a, b), max(a, b)


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["step", "prompts", "attend", "attend", "latent", "latent", "scan", "scan", "recurrence", "experts", "experts"])
    step = rng.random() < 0.5
    if kind == "step":
        lo, hi = _two(rng, 17, 2047)
        return dict(kind=kind, width=rng.choice([2048, 4096, 5120]), layers=rng.randint(1, 3), rows=_log_int(rng, 1, 64), shortest=lo, longest=hi,
                    dtype=rng.choice(["bfloat16", "bfloat16", "float16"]))
    if kind == "prompts":
        lo, hi = _two(rng, 17, 901)
        return dict(kind=kind, width=rng.choice([2048, 4096]), layers=rng.randint(1, 2), rows=rng.randint(1, 5), shortest=lo, longest=hi,
                    dtype=rng.choice(["bfloat16", "bfloat16", "float16"]))
    if kind in ("attend", "latent"):
        rows = _log_int(rng, 1, 64) if step else rng.randint(1, 4)
        lo, hi = _two(rng, 17, 2047 if step else 1151)
        out = dict(kind=kind, step=step, rows=rows, shortest=lo, longest=hi, past=0 if step or rng.random() < 0.7 else rng.randint(1, 500))
        if kind == "attend":
            heads = rng.choice([8, 16, 32])
            mask = rng.choice(["causal", "window", "chunk"])
            return dict(out, heads=heads, kv_heads=heads // rng.choice([1, 2, 4, 8]), dim=rng.choice([64, 128, 128]), mask=mask,
                        size=0 if mask == "causal" else rng.choice([128, 500, 512]), slopes=rng.random() < 0.3, sinks=rng.random() < 0.5,
                        softcap=rng.choice([0.0, 0.0, 30.0]))
        return dict(out, heads=rng.choice([8, 16, 32]), rank=rng.choice([64, 128, 256, 320, 512]), window=rng.choice([0, 500, 512]),
                    gate=rng.random() < 0.5, sinks=rng.random() < 0.5)
    if kind in ("scan", "recurrence"):
        rows = _log_int(rng, 1, 32) if step else rng.randint(1, 4)
        lo, hi = (1, 1) if step else _two(rng, 17, 1151)
        out = dict(kind=kind, step=step, rows=rows, shortest=lo, longest=hi)
        if kind == "recurrence":
            return dict(out, heads=rng.choice([8, 16, 32]), dim=rng.choice([64, 128]), vdim=rng.choice([64, 128]))
        mode = rng.choice(["decay", "bonus", "delta"])
        heads, dim = rng.choice([8, 16, 32]), rng.choice([64, 128])
        return dict(out, mode=mode, heads=heads, qk_heads=heads if mode == "bonus" else heads // rng.choice([1, 2, 4]), dim=dim,
                    vdim=dim if mode == "bonus" else rng.choice([64, 128]))
    width = rng.choice([1024, 2048, 4096])
    experts = rng.choice([8, 16, 32])
    return dict(kind=kind, tokens=_log_int(rng, 1, 3989), width=width, inner=rng.choice([704, 1408]) if width < 4096 or experts > 16 else 2752,
                experts=experts, top=rng.choice([1, 2, 4]))


# ------------------------------------------------------------------------------------------------------------ inputs
def _lens(case):
    """The batch's lengths: from the shortest to the longest, every other one from the far end."""
    n, lo, hi = case["rows"], case["shortest"], case["longest"]
    v = [lo + (hi - lo) * i // max(n - 1, 1) for i in range(n)] if n > 1 else [hi]
    return [v[i // 2] if i % 2 == 0 else v[n - 1 - i // 2] for i in range(n)]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + 13)


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def _batch(new, kv, seed):
    """Index tensors of a ragged batch over a paged cache: sequence s brings its last new[s] of kv[s] tokens; its blocks lie
    anywhere in the pool."""
    n_blocks = [(k + BLOCK - 1) // BLOCK for k in kv]
    perm = torch.randperm(sum(n_blocks), generator=torch.Generator().manual_seed(seed)).tolist()
    cu_blocks, cu_q, cu_k = [0], [0], [0]
    for n, q, k in zip(n_blocks, new, kv):
        cu_blocks.append(cu_blocks[-1] + n)
        cu_q.append(cu_q[-1] + q)
        cu_k.append(cu_k[-1] + k)
    pos = [p for q, k in zip(new, kv) for p in range(k - q, k)]
    seq = [s for s, q in enumerate(new) for _ in range(q)]
    slots = [perm[cu_blocks[s] + p // BLOCK] * BLOCK + p % BLOCK for s, p in zip(seq, pos)]
    return dict(n_blocks=sum(n_blocks), table=_i32(perm), cu_blocks=_i32(cu_blocks), q_cu=_i32(cu_q), k_cu=_i32(cu_k), pos=_i32(pos),
                seq=_i32(seq), slots=_i32(slots), last=torch.tensor([c - 1 for c in cu_q[1:]], device="cuda"), new=new, kv=kv)


def _portions(case):
    """(tokens a sequence brings, tokens it holds with them)"""
    lens = _lens(case)
    if case.get("step", case["kind"] == "step"):
        return [1] * len(lens), lens
    return lens, [n + case.get("past", 0) for n in lens]


def _decoder_inputs(case, seed):
    g = _gen(seed)
    dt = getattr(torch, case["dtype"])
    W, (inner, H), D = case["width"], WIDTHS[case["width"]], 128
    w = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=dt).mul_(0.02)
    norm = lambda: (1 + 0.1 * torch.randn(W, generator=g, device="cuda")).to(dt)
    state = {"embed": w(VOCAB, W), "lm_head": w(VOCAB, W), "norm": norm()}
    for l in range(case["layers"]):
        state.update({f"l{l}.wqkv": w(3 * H * D, W), f"l{l}.wo": w(W, H * D), f"l{l}.wgu": w(2 * inner, W), f"l{l}.wdown": w(W, inner),
                      f"l{l}.norm1": norm(), f"l{l}.norm2": norm()})
    new, kv = _portions(case)
    b = _batch(new, kv, seed)
    caches = [[torch.randn((b["n_blocks"], BLOCK, H, D), generator=g, device="cuda", dtype=dt) for _ in range(2)] for _ in range(case["layers"])]
    ids = torch.randint(0, VOCAB, (sum(new),), generator=g, device="cuda", dtype=torch.int64)
    return state, b, caches, ids, (inner, H, D, dt)


def _attend_inputs(case, seed):
    g = _gen(seed)
    H, G, D = case["heads"], case["kv_heads"], case["dim"]
    b = _batch(*_portions(case), seed)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)], device="cuda") if case["slopes"] else None
    sinks = torch.randn(H, generator=g, device="cuda") if case["sinks"] else None
    return b, r(sum(b["new"]), H, D), r(b["n_blocks"], BLOCK, G, D), r(b["n_blocks"], BLOCK, G, D), slopes, sinks


def _latent_inputs(case, seed):
    g = _gen(seed)
    H, R = case["heads"], case["rank"]
    b = _batch(*_portions(case), seed)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    T = sum(b["new"])
    q = r(H, T, R).transpose(0, 1)                        # as a batched product over the heads leaves it
    return b, q, r(b["n_blocks"], BLOCK, 1, R), r(T, H) if case["gate"] else None, \
        torch.randn(H, generator=g, device="cuda") if case["sinks"] else None


def _starts(case, lens):
    """Every other portion of prompts continues a sequence; single tokens always do."""
    return [77 if case["step"] or s % 2 else 0 for s in range(len(lens))]


def _scan_inputs(case, seed):
    g = _gen(seed)
    H, G, K, V = case["heads"], case["qk_heads"], case["dim"], case["vdim"]
    lens = _lens(case)
    b = _batch(lens, [n + p for n, p in zip(lens, _starts(case, lens))], seed)
    T = sum(lens)
    f = lambda *s: torch.randn(s, generator=g, device="cuda")
    x = dict(q=f(T, G * K), k=f(T, G * K), v=f(T, H * V).to(torch.bfloat16), vscale=None, beta=None, bonus=None)
    if case["mode"] == "bonus":
        x["decay"] = torch.exp(-torch.exp(f(T, H * K) - 2.0))
        x["bonus"] = f(H * K)
    else:
        step = torch.nn.functional.softplus(f(T, H) - 2.0)
        x["decay"] = torch.exp(-torch.exp(0.3 * f(H)) * step)
        if case["mode"] == "decay":
            x["vscale"] = step
        else:
            x["beta"] = torch.sigmoid(f(T, H))
    if case["mode"] == "delta":                           # unit vectors, in float
        unit = lambda t: torch.nn.functional.normalize(t.view(T, G, K), dim=-1).reshape(T, G * K)
        x["q"], x["k"] = unit(x["q"]) * K ** -0.5, unit(x["k"])
    else:                                                 # views of one projection
        both = torch.cat([x["q"], x["k"]], dim=1).mul_(K ** -0.5).to(torch.bfloat16)
        x["q"], x["k"] = both[:, :G * K], both[:, G * K:]
    x["state"] = 0.1 * f(len(lens), 1, H * K * V)
    return b, x


def _recurrence_inputs(case, seed):
    g = _gen(seed)
    H, K, V = case["heads"], case["dim"], case["vdim"]
    lens = _lens(case)
    b = _batch(lens, [n + p for n, p in zip(lens, _starts(case, lens))], seed)
    T = sum(lens)
    f = lambda *s: torch.randn(s, generator=g, device="cuda")
    return b, dict(proj=f(T, H * (2 * K + V)).to(torch.bfloat16), f_bias=f(H * K), low=0.9 * torch.rand(H * K, generator=g, device="cuda"),
                   norm_w=1 + 0.1 * f(V), state=0.1 * f(len(lens), 1, H * K * V))


def _experts_inputs(case, seed):
    g = _gen(seed)
    T, W, F, E = case["tokens"], case["width"], case["inner"], case["experts"]
    f = lambda *s: torch.randn(s, generator=g, device="cuda")
    w = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=torch.bfloat16)
    x = f(T, W)
    return dict(x=x, h=x.to(torch.bfloat16), router=f(E, W).mul_(W ** -0.5), router_b=0.1 * f(E), gate_up=w(E, 2 * F, W).mul_(W ** -0.5),
                down=w(E, W, F).mul_(F ** -0.5), shared=f(T, W).to(torch.bfloat16))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "prompts"):
        from hydrainfer_amd.layer.causal_attention import AttentionParameters, decode_rank_descriptor
        from hydrainfer_amd.memory.kv_cache import KVCache
        from hydrainfer_amd.model.llama import LanguageModelParameters, LlamaForCausalLM, LlamaShape
        state, b, caches, ids, (inner, H, D, dt) = _decoder_inputs(case, seed)
        model = LlamaForCausalLM(LlamaShape(case["width"], inner, case["layers"], H, H, D, VOCAB), dt, "cuda", state)
        single = kind == "step"
        if single:
            model.prepare_decode(max_rows=case["rows"])
        rank = _i32(decode_rank_descriptor(b["kv"])) if single else None
        params = LanguageModelParameters([AttentionParameters(
            kv_cache=KVCache(k, v), q_cu_seq_lens=b["q_cu"], kv_cu_seq_lens=b["k_cu"], new_cache_slots=b["slots"], block_tables=b["table"],
            cu_blocks_lens=b["cu_blocks"], num_sequences=case["rows"], all_sequences_decode=single, q_max_seq_len=max(b["new"]),
            kv_max_seq_len=max(b["kv"]), decode_rank=rank) for k, v in caches], single, None if single else b["last"])
        return dict(kind=kind, model=model, ids=ids, pos=b["pos"], params=params, caches=caches)
    if kind == "attend":
        b, q, kc, vc, slopes, sinks = _attend_inputs(case, seed)
        return dict(kind=kind, args=(q, kc, vc, case["dim"], b["seq"], b["pos"], b["q_cu"], b["table"], b["cu_blocks"], case["dim"] ** -0.5, slopes,
                                     case["mask"], case["size"]),
                    more=dict(max_q_len=max(b["new"]), max_kv_len=max(b["kv"]), softcap=case["softcap"], sinks=sinks))
    if kind == "latent":
        b, q, cache, gate, sinks = _latent_inputs(case, seed)
        return dict(kind=kind, args=(q, cache, b["seq"], b["pos"], b["q_cu"], b["table"], b["cu_blocks"], case["rank"] ** -0.5, case["window"] or None,
                                     max(b["new"])),
                    more=dict(gate_pre=gate, max_kv_len=max(b["kv"]), sinks=sinks))
    if kind in ("scan", "recurrence"):
        from hydrainfer_amd._C.kernel.stream_ops import SequenceState
        b, x = _scan_inputs(case, seed) if kind == "scan" else _recurrence_inputs(case, seed)
        seq = SequenceState(x["state"], _i32(list(range(case["rows"]))), b["seq"])
        H, K, V = case["heads"], case["dim"], case["vdim"]
        if kind == "scan":
            return dict(kind=kind, seq=seq, args=(case["mode"], x["q"], x["k"], x["v"], x["decay"], seq, 0, b["q_cu"], b["pos"], H, case["qk_heads"], K, V),
                        more=dict(vscale=x["vscale"], beta=x["beta"], bonus=x["bonus"]))
        p = x["proj"]
        return dict(kind=kind, seq=seq, args=(p[:, :H * K], p[:, H * K:2 * H * K], p[:, 2 * H * K:], x["f_bias"], x["low"], x["norm_w"], 1e-5, seq, 0,
                                              b["q_cu"], b["pos"], H, K, V), more=dict(max_q_len=max(b["new"])))
    from hydrainfer_amd._C.kernel.moe_mix import gate_up_turns
    x = _experts_inputs(case, seed)
    F = case["inner"]
    for w in x["gate_up"]:
        w.copy_(gate_up_turns(w[:F], w[F:]))
    return dict(x, kind=kind, top=case["top"])


# --------------------------------------------------------------------------------------------------------------- run
def run(state):
    kind = state["kind"]
    with torch.inference_mode():
        if kind in ("step", "prompts"):
            logits = state["model"].forward_logits(state["ids"], state["pos"], state["params"])
            return {"logits": logits, "caches": state["caches"]}
        if kind == "attend":
            from hydrainfer_amd._C.kernel.biased_attn import biased_attention
            return biased_attention(*state["args"], **state["more"])
        if kind == "latent":
            from hydrainfer_amd._C.kernel.latent_attn import latent_attention
            return latent_attention(*state["args"], **state["more"])
        if kind == "scan":
            from hydrainfer_amd._C.kernel.seq_mix import state_scan
            return {"out": state_scan(*state["args"], **state["more"]), "state": state["seq"].state}
        if kind == "recurrence":
            from hydrainfer_amd._C.kernel.recurrence import gated_recurrence
            return {"out": gated_recurrence(*state["args"], **state["more"]), "state": state["seq"].state}
        from hydrainfer_amd._C.kernel.moe_mix import grouped_linear, moe_combine, moe_plan, router_topk
        T, top, E = state["x"].shape[0], state["top"], state["router"].shape[0]
        weights, experts = router_topk(state["x"], state["router"], state["router_b"], top)
        seg, row_of, src = moe_plan(experts, E)
        inner = grouped_linear(state["h"], state["gate_up"], seg, T * top, src=src, act="glu", limit=GLU_LIMIT, alpha=GLU_ALPHA, up_shift=1.0)
        y = grouped_linear(inner, state["down"], seg, T * top)
        return {"out": moe_combine(y, row_of, weights, state["shared"]), "weights": weights, "experts": experts}


# -------------------------------------------------------------------------------------------------------------- work
def _seen(new, kv, first):
    """Pairs of a query and a key that it sees."""
    return sum(p - first(p) + 1 for q, k in zip(new, kv) for p in range(k - q, k))


def _read(new, kv, first):
    """Cached rows that some query sees."""
    return sum(k - first(k - q) for q, k in zip(new, kv))


def _first(mask, size):
    if mask == "window":
        return lambda p: max(0, p - size + 1)
    if mask == "chunk":
        return lambda p: p // size * size
    return lambda p: 0


def work(case):
    kind = case["kind"]
    if kind in ("step", "prompts"):
        W, (inner, H), D, L = case["width"], WIDTHS[case["width"]], 128, case["layers"]
        new, kv = _portions(case)
        T, n = sum(new), case["rows"]
        layer = 3 * H * D * W + W * H * D + 3 * inner * W
        flops = 2 * L * layer * T + 4 * L * H * D * _seen(new, kv, _first("causal", 0)) + 2 * n * VOCAB * W
        if kind == "prompts":                             # the last layer's feed-forward serves the sampled rows only
            flops -= 2 * 3 * inner * W * (T - n)
        return {"bytes": 2 * (L * layer + VOCAB * W + T * W + n * VOCAB + 2 * L * H * D * sum(kv)), "flops": flops}
    if kind == "attend":
        new, kv = _portions(case)
        H, G, D, first = case["heads"], case["kv_heads"], case["dim"], _first(case["mask"], case["size"])
        return {"bytes": 2 * (2 * sum(new) * H * D + 2 * G * D * _read(new, kv, first)), "flops": 4 * H * D * _seen(new, kv, first)}
    if kind == "latent":
        new, kv = _portions(case)
        H, R, first = case["heads"], case["rank"], _first("window" if case["window"] else "causal", case["window"])
        return {"bytes": 2 * (2 * sum(new) * H * R + R * _read(new, kv, first)), "flops": 4 * H * R * _seen(new, kv, first)}
    if kind in ("scan", "recurrence"):
        H, K, V, T = case["heads"], case["dim"], case["vdim"], sum(_lens(case))
        continued = sum(1 for s in _starts(case, _lens(case)) if s)
        state = 4 * H * K * V * (case["rows"] + continued)
        if kind == "recurrence":
            return {"bytes": state + 2 * T * H * (2 * K + 2 * V), "flops": 5 * T * H * K * V}
        G, e = case["qk_heads"], 4 if case["mode"] == "delta" else 2
        per_token = 2 * e * G * K + 6 * H * V + 4 * H * (K if case["mode"] == "bonus" else 2)
        return {"bytes": state + T * per_token, "flops": {"decay": 5, "bonus": 5, "delta": 7}[case["mode"]] * T * H * K * V}
    T, W, F, E, top = case["tokens"], case["width"], case["inner"], case["experts"], case["top"]
    used = min(E, E * (1 - (1 - top / E) ** T))           # experts that some token chooses
    return {"bytes": 2 * used * 3 * F * W + 4 * E * W + T * W * (4 + 2 + 2 + 2) + 8 * T * top, "flops": 2 * T * top * 3 * F * W + 2 * T * E * W}


def tolerance(case):
    kind = case["kind"]
    if kind in ("step", "prompts"):                       # bfloat16 activations and residual through the layers
        return {"rel": 0.03, "max": 0.3} if case["dtype"] == "bfloat16" else {"rel": 0.01, "max": 0.1}
    if kind == "scan":                                    # float throughout
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "experts":
        return {"rel": 0.01, "max": 0.15, "differ": 0.001}
    return {"rel": 0.01, "max": 0.15}                     # one rounding to bfloat16 of weights and results


# -------------------------------------------------------------------------------------------------- the same in 64 bits
def _rows_of(cache, b, s):
    """Sequence s's cached rows [keys, heads, size]."""
    lo, hi = int(b["cu_blocks"][s]), int(b["cu_blocks"][s + 1])
    rows = cache[b["table"][lo:hi].long()]
    return rows.reshape(-1, *rows.shape[2:])[:b["kv"][s]]


def _softmax_attention(q, k, v, pos, first, scale, slopes=None, sinks=None, softcap=0.0):
    """q [n, H, D], k / v [keys, G, .] in double, queries at positions pos: [n, H, V]."""
    n, H, D = q.shape
    G = k.shape[1]
    q = q.transpose(0, 1).contiguous()                                           # [H, n, D]
    k, v = (x.transpose(0, 1).repeat_interleave(H // G, dim=0) for x in (k, v))
    s = torch.bmm(q, k.transpose(1, 2).contiguous()) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    j = torch.arange(k.shape[1], device="cuda")
    far = (pos.long()[:, None] - j[None, :]).double()
    if slopes is not None:
        s = s - slopes.double()[:, None, None] * far
    lo = torch.tensor([first(int(p)) for p in pos.tolist()], device="cuda")
    s = s.masked_fill(((far < 0) | (j[None, :] < lo[:, None]))[None], -math.inf)
    if sinks is not None:
        s = torch.cat([s, sinks.double()[:, None, None].expand(H, n, 1)], dim=2)
    p = torch.softmax(s, dim=2)[:, :, :k.shape[1]].contiguous()
    return torch.bmm(p, v.contiguous()).transpose(0, 1)


def _exact_decoder(case, seed):
    st, b, caches, ids, (inner, H, D, dt) = _decoder_inputs(case, seed)
    w = lambda n: st[n].double()
    norm = lambda x, n: x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + 1e-5) * w(n)
    inv = 1.0 / torch.pow(10000.0, torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D)
    ang = b["pos"].double()[:, None] * inv[None, :]
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]

    def turn(x):
        x1, x2 = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], dim=-1)

    h = st["embed"][ids].double()
    slots, q_cu, out = b["slots"].long(), b["q_cu"].tolist(), []
    for l in range(case["layers"]):
        q, k, v = (norm(h, f"l{l}.norm1") @ w(f"l{l}.wqkv").t()).view(-1, 3, H, D).unbind(1)
        q, k = turn(q), turn(k)
        pair = []
        for cache, rows in zip(caches[l], (k, v)):
            c = cache.double()
            c.view(-1, H, D)[slots] = rows
            pair.append(c)
        o = torch.cat([_softmax_attention(q[q_cu[s]:q_cu[s + 1]], _rows_of(pair[0], b, s), _rows_of(pair[1], b, s), b["pos"][q_cu[s]:q_cu[s + 1]],
                                          lambda p: 0, D ** -0.5) for s in range(case["rows"])])
        out.append(pair)
        h = h + o.reshape(-1, H * D) @ w(f"l{l}.wo").t()
        if case["kind"] == "prompts" and l == case["layers"] - 1:
            h = h[b["last"]]
        gu = norm(h, f"l{l}.norm2") @ w(f"l{l}.wgu").t()
        h = h + (torch.nn.functional.silu(gu[:, :inner]) * gu[:, inner:]) @ w(f"l{l}.wdown").t()
    return {"logits": norm(h, "norm") @ w("lm_head").t(), "caches": out}


def _exact_attend(case, seed):
    if case["kind"] == "attend":
        b, q, kc, vc, slopes, sinks = _attend_inputs(case, seed)
        gate, first, scale, cap = None, _first(case["mask"], case["size"]), case["dim"] ** -0.5, case["softcap"]
    else:
        b, q, kc, gate, sinks = _latent_inputs(case, seed)
        vc, slopes, cap, first, scale = kc, None, 0.0, _first("window" if case["window"] else "causal", case["window"]), case["rank"] ** -0.5
    q_cu = b["q_cu"].tolist()
    out = torch.cat([_softmax_attention(q[q_cu[s]:q_cu[s + 1]].double(), _rows_of(kc, b, s).double(), _rows_of(vc, b, s).double(),
                                        b["pos"][q_cu[s]:q_cu[s + 1]], first, scale, slopes, sinks, cap) for s in range(case["rows"])])
    return out if gate is None else out * torch.sigmoid(gate.double())[:, :, None]


def _padded(t, b, fill=0.0):
    """[tokens, ...] -> double [sequences, longest portion, ...]"""
    q_cu = b["q_cu"].tolist()
    out = torch.full((len(b["new"]), max(b["new"]), *t.shape[1:]), fill, dtype=torch.float64, device="cuda")
    for s, n in enumerate(b["new"]):
        out[s, :n] = t[q_cu[s]:q_cu[s] + n].double()
    return out


def _exact_scan(case, seed):
    H, K, V, rows = case["heads"], case["dim"], case["vdim"], case["rows"]
    hgrn = case["kind"] == "recurrence"
    if hgrn:
        b, x = _recurrence_inputs(case, seed)
        p = x["proj"].double()
        f = x["low"].double() + (1 - x["low"].double()) * torch.sigmoid(p[:, H * K:2 * H * K] + x["f_bias"].double())
        x.update(q=torch.nn.functional.silu(p[:, :H * K]), k=1 - f, v=p[:, 2 * H * K:], decay=f)
        mode, G = "decay", H
    else:
        b, x = _scan_inputs(case, seed)
        mode, G = case["mode"], case["qk_heads"]
    q, k = (_padded(x[n], b).view(rows, -1, G, K).repeat_interleave(H // G, dim=2) for n in ("q", "k"))
    v = _padded(x["v"], b).view(rows, -1, H, V)
    a = _padded(x["decay"], b, 1.0).view(rows, v.shape[1], H, -1, 1)             # (a token past the portion changes nothing)
    if x.get("vscale") is not None:
        v = v * _padded(x["vscale"], b)[..., None]
    beta = _padded(x["beta"], b)[..., None, None] if mode == "delta" else None
    S = x["state"].double().view(rows, H, K, V).clone()
    for s, start in enumerate(_starts(case, b["new"])):
        if start == 0:
            S[s] = 0
    out = torch.empty_like(v)
    for t in range(v.shape[1]):
        qt, kt, vt = q[:, t, :, None, :], k[:, t, :, :, None], v[:, t, :, None, :]
        if mode == "bonus":
            kv = kt * vt
            out[:, t] = torch.matmul(qt, S + x["bonus"].double().view(H, K, 1) * kv)[:, :, 0]
            S = a[:, t] * S + kv
        else:
            S = a[:, t] * S
            if mode == "delta":
                vt = beta[:, t] * (vt - torch.matmul(kt.transpose(2, 3), S))
            S = S + kt * vt
            out[:, t] = torch.matmul(qt, S)[:, :, 0]
    out = torch.cat([out[s, :n] for s, n in enumerate(b["new"])])
    if hgrn:
        out = out / torch.sqrt((out * out).mean(dim=-1, keepdim=True) + 1e-5) * x["norm_w"].double()
    return {"out": out.reshape(-1, H * V), "state": S.reshape(rows, 1, -1)}


def _exact_experts(case, seed):
    x = _experts_inputs(case, seed)
    F, E = case["inner"], case["experts"]
    z, experts = torch.topk(x["x"].double() @ x["router"].double().t() + x["router_b"].double(), case["top"], dim=1)
    weights = torch.softmax(z, dim=1)
    out = x["shared"].double()
    for e in range(E):
        t, k = (experts == e).nonzero(as_tuple=True)
        gu = x["h"][t].double() @ x["gate_up"][e].double().t()
        g, u = gu[:, :F].clamp(max=GLU_LIMIT), gu[:, F:].clamp(-GLU_LIMIT, GLU_LIMIT)
        out.index_add_(0, t, weights[t, k][:, None] * ((g * torch.sigmoid(GLU_ALPHA * g) * (u + 1.0)) @ x["down"][e].double().t()))
    return {"out": out, "weights": weights, "experts": experts.to(torch.int32)}


def exact(case, seed):
    with torch.inference_mode():
        kind = case["kind"]
        if kind in ("step", "prompts"):
            return _exact_decoder(case, seed)
        if kind in ("attend", "latent"):
            return _exact_attend(case, seed)
        return _exact_scan(case, seed) if kind in ("scan", "recurrence") else _exact_experts(case, seed)
