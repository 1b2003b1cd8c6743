"""G8: tiny Llama end-to-end (prefill two requests, then greedy decode) — the oracle model on
CPU and the HIP-backed LlamaForCausalLM on GPU against logits/tokens produced by the
reference's own LlamaForCausalLM (tests/golden/generate_goldens.py::gen_tiny_llama)."""
import numpy as np
import pytest
import torch

from tests.golden import cases as C
from tests.util import load_golden

BS = C.TINY_BLOCK_SIZE


def _shape():
    from hydrainfer_amd.model.llama import LlamaShape
    t = C.TINY_LLAMA
    return LlamaShape(**t)


def _scenario(step_fn):
    """Drives `step_fn(ids, positions, meta(dict of lists), select)` -> logits [2, vocab] fp32
    through prefill + decode, greedy-feeding its own tokens.  Returns (tokens, logits)."""
    tables = C.tiny_block_tables()
    lens = [0, 0]
    toks, logs = [], []
    new = [C.tiny_prompt_ids(0), C.tiny_prompt_ids(1)]
    for _ in range(C.TINY_DECODE_STEPS):
        ids, pos, sel, slots, bt, cu_q, cu_k, cu_b = [], [], [], [], [], [0], [0], [0]
        for r, n in enumerate(new):
            slots += [tables[r][p // BS] * BS + p % BS for p in range(lens[r], lens[r] + len(n))]
            pos += list(range(lens[r], lens[r] + len(n)))
            lens[r] += len(n)
            t = tables[r][: (lens[r] + BS - 1) // BS]
            bt += t
            ids += n
            cu_q.append(cu_q[-1] + len(n))
            cu_k.append(cu_k[-1] + lens[r])
            cu_b.append(cu_b[-1] + len(t))
            sel.append(cu_q[-1] - 1)
        meta = dict(q_cu=cu_q, kv_cu=cu_k, slots=slots, bt=bt, cu_b=cu_b, q_lens=[len(n) for n in new],
                    kv_lens=list(lens), tables=[tables[r][: (lens[r] + BS - 1) // BS] for r in range(2)])
        logits = step_fn(ids, pos, meta, sel)
        nxt = logits.argmax(-1).tolist()
        toks.append(nxt)
        logs.append(logits)
        new = [[nxt[0]], [nxt[1]]]
    return np.array(toks), torch.stack(logs).numpy()


def _pool(dt):
    t = C.TINY_LLAMA
    gen = torch.Generator().manual_seed(77)
    return torch.randn((t["num_hidden_layers"], 2, C.TINY_BLOCKS, BS, t["num_key_value_heads"],
                        t["head_dim"]), generator=gen).to(dt)


def _margin_ok(ref_logits, tol):
    """top-1 margin of the reference logits vs the comparison tolerance: greedy-token identity
    is only asserted where the margin exceeds twice the tolerance."""
    srt = np.sort(ref_logits, axis=-1)
    return (srt[..., -1] - srt[..., -2]) > 2 * tol


@pytest.mark.parametrize("dname", ["fp16", "bf16"])
def test_oracle_model_matches_reference(dname):
    from oracle.model import OracleAttnMeta, OracleLlama
    g = load_golden("g8_tiny_llama")
    dt = C.DTYPES[dname]
    pool = _pool(dt)
    assert C.checksum(pool) == str(g[f"tiny_{dname}_pool_chk"])
    model = OracleLlama(_shape(), C.tiny_llama_state_dict(dt), dt)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)

    def step(ids, pos, m, sel):
        meta = OracleAttnMeta(i32(m["q_cu"]), i32(m["kv_cu"]), i32(m["slots"]), i32(m["bt"]), i32(m["cu_b"]))
        caches = [(pool[l, 0], pool[l, 1]) for l in range(pool.shape[0])]
        select = torch.tensor(sel) if any(q > 1 for q in m["q_lens"]) else None
        return model.forward_logits(i32(ids), i32(pos), meta, caches, select).float()

    toks, logs = _scenario(step)
    np.testing.assert_array_equal(toks, g[f"tiny_{dname}_tokens"])
    assert C.checksum(pool) == str(g[f"tiny_{dname}_pool_end_chk"])  # KV cache bit-exact
    # same ops, same machine class: logits agree to T round-off of the last linear
    np.testing.assert_allclose(logs, g[f"tiny_{dname}_logits"], atol=2e-2 if dname == "bf16" else 4e-3, rtol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("dname", ["fp16", "bf16"])
def test_hip_model_matches_reference(dname):
    from hydrainfer_amd.layer.causal_attention import AttentionParametersBuilder
    from hydrainfer_amd.memory.kv_cache import KVCache
    from hydrainfer_amd.model.llama import LanguageModelParameters, LlamaForCausalLM
    g = load_golden("g8_tiny_llama")
    dt = C.DTYPES[dname]
    dev = torch.device("cuda:0")
    shape = _shape()
    model = LlamaForCausalLM.from_reference_state_dict(shape, C.tiny_llama_state_dict(dt), dt, dev)
    pool = _pool(dt).to(dev)
    L = shape.num_hidden_layers

    def step(ids, pos, m, sel):
        b = AttentionParametersBuilder(shape.num_attention_heads, shape.num_key_value_heads,
                                       shape.head_dim, BS, dev)
        off = 0
        for r in range(2):
            ql = m["q_lens"][r]
            b.add_request(ql, m["kv_lens"][r], m["slots"][off: off + ql], m["tables"][r])
            off += ql
        for l in range(L):
            b.add_kv_cache(KVCache(pool[l, 0], pool[l, 1]))
        ap = b.build_attention_parameters()
        for f in ("q_cu_seq_lens", "kv_cu_seq_lens", "new_cache_slots", "block_tables", "cu_blocks_lens"):
            key = {"q_cu_seq_lens": "q_cu", "kv_cu_seq_lens": "kv_cu", "new_cache_slots": "slots",
                   "block_tables": "bt", "cu_blocks_lens": "cu_b"}[f]
            assert getattr(ap[0], f).tolist() == m[key]   # integer metadata bit-exact
        prefill = any(q > 1 for q in m["q_lens"])
        params = LanguageModelParameters(attention_params=ap, all_sequences_decode=not prefill,
                                         selected_token_ids=torch.tensor(sel, device=dev) if prefill else None)
        logits = model.forward_logits(torch.tensor(ids, dtype=torch.int32, device=dev),
                                      torch.tensor(pos, dtype=torch.int32, device=dev), params)
        return logits.float().cpu()

    toks, logs = _scenario(step)
    ref_logits, ref_toks = g[f"tiny_{dname}_logits"], g[f"tiny_{dname}_tokens"]
    # stated tolerance on logits vs the reference's CPU path: fp16 2e-2, bf16 1.5e-1 absolute
    # (logit scale ~ +-6; reference's own model bar is atol=rtol=0.2, tests/model/test_llama.py:57)
    tol = 1.5e-1 if dname == "bf16" else 2e-2
    same_path = (toks == ref_toks).all(axis=1).cumprod() == 1   # steps before any divergence
    n_same = int(same_path.sum())
    assert n_same >= 1
    err = np.abs(logs[:n_same] - ref_logits[:n_same]).max()
    assert err <= tol, f"logits max abs err {err} > {tol}"
    # greedy tokens identical wherever the reference's top-1 margin exceeds 2*tol
    ok = _margin_ok(ref_logits, tol)
    for s in range(C.TINY_DECODE_STEPS):
        if not ok[s].all():
            break   # a near-tie: later steps legitimately depend on the tie-break
        assert (toks[s] == ref_toks[s]).all(), f"greedy token mismatch at step {s}"
    else:
        assert (toks == ref_toks).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(4096, 11008, 32, 32), (5120, 13824, 40, 40), (2048, 5632, 16, 4)],
                         ids=["7b-mha", "13b-mha", "gqa-16q-4kv"])
def test_7b_shaped_two_layer_model_matches_oracle(dims):
    """BASELINE layer shapes (7B: hidden 4096, 32 heads x 128, inter 11008; 13B = configs[2]: hidden
    5120, 40 heads, inter 13824; vocab 32064) with 2 layers: prefill + 4 greedy decode steps on the
    HIP path (decode GEMMs on the weight-streaming kernel with packed weights, fused attention)
    against the CPU oracle model on the same weights; and a grouped-query shape (16 query / 4 KV
    heads), whose decode steps run the grouped-query attention kernel."""
    from hydrainfer_amd.layer.causal_attention import AttentionParametersBuilder
    from hydrainfer_amd.memory.kv_cache import KVCache
    from hydrainfer_amd.model.llama import LanguageModelParameters, LlamaForCausalLM, LlamaShape
    from oracle.model import OracleAttnMeta, OracleLlama
    dt, dev = torch.float16, torch.device("cuda:0")
    hidden, inter, H, HK = dims
    shape = LlamaShape(hidden, inter, 2, H, HK, 128, 32064)
    model = LlamaForCausalLM.random_init(shape, dt, dev, seed=3, std=0.02)
    assert model.fuse_decode_attention == (H == HK)
    sd = model.to_reference_state_dict()
    oracle = OracleLlama(shape, sd, dt)
    bs, n_blocks = 16, 16
    gen = torch.Generator().manual_seed(5)
    pool = torch.randn((2, 2, n_blocks, bs, HK, 128), generator=gen).to(dt)
    pool_d = pool.to(dev)
    prompts = [torch.randint(0, 32000, (50,), generator=gen).tolist(), torch.randint(0, 32000, (33,), generator=gen).tolist()]
    tables = [[15, 14, 13, 12], [11, 10, 9]]
    lens = [0, 0]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)
    new = prompts
    n_checked = 0
    for step in range(5):
        ids, pos, sel, slots, bt, cu_q, cu_k, cu_b = [], [], [], [], [], [0], [0], [0]
        b = AttentionParametersBuilder(H, HK, 128, bs, dev)
        for r, x in enumerate(new):
            sl = [tables[r][p // bs] * bs + p % bs for p in range(lens[r], lens[r] + len(x))]
            pos += list(range(lens[r], lens[r] + len(x)))
            lens[r] += len(x)
            tb = tables[r][: (lens[r] + bs - 1) // bs]
            b.add_request(len(x), lens[r], sl, tb)
            slots += sl; bt += tb; ids += x
            cu_q.append(cu_q[-1] + len(x)); cu_k.append(cu_k[-1] + lens[r]); cu_b.append(cu_b[-1] + len(tb))
            sel.append(cu_q[-1] - 1)
        for l in range(2):
            b.add_kv_cache(KVCache(pool_d[l, 0], pool_d[l, 1]))
        prefill = step == 0
        params = LanguageModelParameters(attention_params=b.build_attention_parameters(),
                                         all_sequences_decode=not prefill,
                                         selected_token_ids=torch.tensor(sel, device=dev) if prefill else None)
        got = model.forward_logits(torch.tensor(ids, dtype=torch.int64, device=dev),
                                   torch.tensor(pos, dtype=torch.int32, device=dev), params).float().cpu()
        meta = OracleAttnMeta(i32(cu_q), i32(cu_k), i32(slots), i32(bt), i32(cu_b))
        ref = oracle.forward_logits(i32(ids), i32(pos), meta, [(pool[l, 0], pool[l, 1]) for l in range(2)],
                                    torch.tensor(sel) if prefill else None).float()
        err = (got - ref).abs().max().item()
        assert err <= 3e-2, f"step {step}: logits max abs err {err}"       # stated tolerance (fp16)
        srt = ref.sort(dim=-1).values
        margin_ok = (srt[:, -1] - srt[:, -2]) > 6e-2
        gt, rt = got.argmax(-1), ref.argmax(-1)
        assert (gt[margin_ok] == rt[margin_ok]).all(), f"step {step}: greedy token differs despite a clear margin"
        n_checked += int(margin_ok.sum())
        new = [[int(rt[0])], [int(rt[1])]]          # both sides follow the oracle's tokens
    # the KV pool written by the HIP path equals the oracle's up to T round-off of the projections
    assert (pool_d.cpu().float() - pool.float()).abs().max().item() <= 2e-2


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_decode_with_norm_fused_launches_equals_separate_launches(dt):
    """A 3-layer 7B-width model, 24 decode steps: the 5-launch layer (add+norm folded into the gate|up and
    qkv launches, in-kernel hand-over over the same buffers every layer and step) == the 7-launch layer:
    sampled tokens and the whole KV pool bit-identical, no hand-over gave up."""
    from hydrainfer_amd.model.llama import LlamaForCausalLM, LlamaShape
    from hydrainfer_amd.model.runner import DecodeRunner, RunnerConfig
    DEV = torch.device("cuda:0")
    sh = LlamaShape(1024, 2816, 3, 8, 8, 128, 2048)
    outs = []
    for fuse in (False, True):
        model = LlamaForCausalLM.random_init(sh, dt, DEV, seed=3)
        model.fuse_norm = fuse
        r = DecodeRunner(model, RunnerConfig(batch=5, prompt_len=40, n_generate=32, use_graph=fuse), seed=4)
        g = torch.Generator().manual_seed(0)
        r.prefill(torch.randint(5, 2000, (5, 40), generator=g).to(DEV))
        for _ in range(24):
            r.step()
        torch.cuda.synchronize()
        if fuse:
            assert model.xreg_sync is not None and int(model.xreg_sync[:, :, 1].abs().sum()) == 0
        outs.append((r.generated(), r.pool.clone()))
    assert torch.equal(outs[0][0], outs[1][0])
    assert torch.equal(outs[0][1], outs[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("hidden, inter, layers, batch", [(1024, 2816, 3, 1), (1024, 2816, 1, 32), (2048, 5632, 3, 5)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_layers_in_one_call_each_equal_the_launches_one_by_one(hidden, inter, layers, batch, dt):
    """The next layer's norm inside its qkv product (width 1024) and as a launch of its own (width 2048, two K splits): sampled
    tokens and the KV pool bit-identical, eager steps and replayed graphs."""
    from hydrainfer_amd.model import llama
    from hydrainfer_amd.model.runner import DecodeRunner, RunnerConfig
    sh = llama.LlamaShape(hidden, inter, layers, hidden // 128, hidden // 128, 128, 2048)
    outs, calls = [], []
    for one_call, graph in ((False, False), (True, False), (True, True)):
        model = llama.LlamaForCausalLM.random_init(sh, dt, torch.device("cuda:0"), seed=3)
        model.one_call = one_call
        r = DecodeRunner(model, RunnerConfig(batch=batch, prompt_len=40, n_generate=16, use_graph=graph), seed=4)
        g = torch.Generator().manual_seed(0)
        r.prefill(torch.randint(5, 2000, (batch, 40), generator=g).cuda())
        whole = llama.decode_layers
        llama.decode_layers = lambda *a: calls.append(one_call) or whole(*a)
        try:
            for _ in range(12):
                r.step()
        finally:
            llama.decode_layers = whole
        torch.cuda.synchronize()
        outs.append((r.generated(), r.pool.clone()))
    assert calls and all(calls)
    for tokens, pool in outs[1:]:
        assert torch.equal(outs[0][0], tokens) and torch.equal(outs[0][1], pool)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [33, 40, 64])
def test_wide_steps_of_a_narrow_model_equal_two_halves(rows):
    """Width 2048, more than 32 rows: the qkv product of the second layer leaves two slabs, and its norm is a launch of its own."""
    from hydrainfer_amd.layer.causal_attention import AttentionParametersBuilder
    from hydrainfer_amd.memory.kv_cache import KVCache
    from hydrainfer_amd.model.llama import LanguageModelParameters, LlamaForCausalLM, LlamaShape
    dt, dev, L, H = torch.float16, torch.device("cuda:0"), 2, 16
    model = LlamaForCausalLM.random_init(LlamaShape(2048, 5632, L, H, H, 128, 2048), dt, dev, seed=3)
    model.prepare_decode(max_rows=rows)
    g = torch.Generator().manual_seed(rows)
    start, ids = torch.randn((L, 2, 4 * rows, 16, H, 128), generator=g).to(dt), torch.randint(0, 2048, (rows,), generator=g)
    kv = [1 + (13 * r) % 60 for r in range(rows)]

    def step(some):
        pool, b = start.to(dev), AttentionParametersBuilder(H, H, 128, 16, dev)
        for r in some:
            b.add_request(1, kv[r], [64 * r + kv[r] - 1], [4 * r + i for i in range((kv[r] + 15) // 16)])
        for l in range(L):
            b.add_kv_cache(KVCache(pool[l, 0], pool[l, 1]))
        return model.forward_logits(ids[list(some)].to(dev), torch.tensor([kv[r] - 1 for r in some], dtype=torch.int32, device=dev),
                                    LanguageModelParameters(b.build_attention_parameters(), True)).float()

    whole, halves = step(range(rows)), torch.cat([step(range(rows // 2)), step(range(rows // 2, rows))])
    assert model._decode_plan(rows, dt)["wide"]
    # (either is within 3e-2 of the oracle, as above)
    assert bool(torch.isfinite(whole).all()) and float((whole - halves).abs().max()) <= 6e-2


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 16, 17])
@pytest.mark.parametrize("vocab", [2048, 2050])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_logits_of_few_rows(rows, vocab, dt, monkeypatch):
    """On both sides of the 16 rows that the weight-streaming product takes, and with outputs that it does not take."""
    from hydrainfer_amd.model import llama
    from hydrainfer_amd.model.llama import LanguageModelParameters, LlamaForCausalLM, LlamaShape
    monkeypatch.setattr(llama, "MEMORY_SIDE_CACHE", 0)            # (a head of any size comes from memory)
    streamed = []
    monkeypatch.setattr(llama.hip_gemm, "linear_decode", lambda *a, whole=llama.hip_gemm.linear_decode: streamed.append(1) or whole(*a))
    model = LlamaForCausalLM.random_init(LlamaShape(1024, 2816, 1, 8, 8, 128, vocab), dt, torch.device("cuda:0"), seed=3)
    x = torch.randn((rows, 1024), generator=torch.Generator().manual_seed(rows)).to(dt).cuda()
    model.forward_hidden = lambda *a: x
    got, want = model.forward_logits(x, None, LanguageModelParameters([], False)).float(), x.float() @ model.state["lm_head"].float().t()
    assert len(streamed) == (rows <= 16 and vocab % 16 == 0)
    # sums in float (1024 products, a unit of 2^-24 of the sum of their sizes each at worst), rounded once to dt
    unit = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    size = x.float().abs() @ model.state["lm_head"].float().abs().t()
    assert got.shape == (rows, vocab) and bool(((got - want).abs() <= unit * want.abs() + 1024 * 2.0 ** -24 * size + 1e-7).all())


@pytest.mark.parametrize("off", range(9))
def test_a_head_off_sixteen_bytes_is_left_to_the_library(off, monkeypatch):
    from hydrainfer_amd.model import llama
    calls = []
    model = llama.LlamaForCausalLM.random_init(llama.LlamaShape(256, 512, 1, 2, 2, 128, 160), torch.bfloat16, "cpu")
    model.state["lm_head"] = torch.zeros(160 * 256 + 8, dtype=torch.bfloat16)[off:off + 160 * 256].view(160, 256)
    monkeypatch.setattr(llama, "MEMORY_SIDE_CACHE", 0)            # (a head of any size comes from memory)
    monkeypatch.setattr(llama.hip_gemm, "linear_decode", lambda x, w: calls.append(1) or torch.matmul(x, w.t()))
    model.forward_hidden = lambda *a: torch.zeros((3, 256), dtype=torch.bfloat16)
    model.forward_logits(torch.zeros(3, dtype=torch.int64), None, llama.LanguageModelParameters([], False))
    assert bool(calls) == (off % 8 == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 16])
def test_logits_of_a_head_off_sixteen_bytes(rows, monkeypatch):
    """A head that is a view into a flat buffer: the same logits as from a head of its own, behind prompts as in steps."""
    from hydrainfer_amd.model import llama
    from hydrainfer_amd.model.llama import LanguageModelParameters, LlamaForCausalLM, LlamaShape
    monkeypatch.setattr(llama, "MEMORY_SIDE_CACHE", 0)            # (a head of any size comes from memory)
    model = LlamaForCausalLM.random_init(LlamaShape(1024, 2816, 1, 8, 8, 128, 2048), torch.bfloat16, torch.device("cuda:0"), seed=3)
    x, head = torch.randn((rows, 1024), generator=torch.Generator().manual_seed(rows)).bfloat16().cuda(), model.state["lm_head"]
    model.forward_hidden = lambda *a: x
    flat = torch.empty(head.numel() + 1, dtype=head.dtype, device=head.device)
    model.state["lm_head"] = flat[1:].view_as(head).copy_(head)
    for step in (False, True):
        got, want = model.forward_logits(x, None, LanguageModelParameters([], step)).float(), x.float() @ head.float().t()
        # sums in float (1024 products, a unit of 2^-24 of the sum of their sizes each at worst), rounded once
        bound = 2.0 ** -8 * want.abs() + 1024 * 2.0 ** -24 * (x.float().abs() @ head.float().abs().t()) + 1e-7
        assert bool(((got - want).abs() <= bound).all())


@pytest.mark.parametrize("rows, tokens, step, head_fits, all_fit, streams", [
    (16, 1000, False, True, False, True), (17, 1000, False, True, False, False), (5, 65, False, True, False, True), (5, 64, False, True, False, False),
    (5, 1000, False, True, True, False), (1, 1, True, True, False, False), (16, 16, True, True, False, False), (16, 16, True, False, False, True),
    (1, 17, False, False, False, True), (17, 17, True, False, False, False)])
def test_which_product_makes_the_logits(rows, tokens, step, head_fits, all_fit, streams, monkeypatch):
    """The streaming product where the head comes from memory: larger than the memory-side cache, or pushed out of it by the library's
    products of more than 64 tokens."""
    from hydrainfer_amd.model import llama
    calls = []
    model = llama.LlamaForCausalLM.random_init(llama.LlamaShape(256, 512, 2, 2, 2, 128, 160), torch.bfloat16, "cpu")
    head, layer = model.state["lm_head"], sum(model.state[f"l0.{n}"].numel() for n in ("wqkv", "wo", "wgu", "wdown"))
    assert model.linear_bytes == 2 * (head.numel() + 2 * layer)
    monkeypatch.setattr(llama, "MEMORY_SIDE_CACHE", model.linear_bytes if all_fit else 2 * head.numel() - (not head_fits))
    monkeypatch.setattr(llama.hip_gemm, "linear_decode", lambda x, w: calls.append(1) or torch.matmul(x, w.t()))
    model.forward_hidden = lambda *a: torch.zeros((rows, 256), dtype=torch.bfloat16)
    assert model.forward_logits(torch.zeros(tokens, dtype=torch.int64), None, llama.LanguageModelParameters([], step)).shape == (rows, 160)
    assert bool(calls) == streams
