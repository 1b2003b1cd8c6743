"""The last layer of a batch of prompts, whose queries are made of the sampled rows only (csrc/prompt_rows.hip, model/llama.py), against all rows
through it and the sampled ones taken out behind its attention."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BLOCK = 16


def _batch(new, kv, seed):
    n_blocks = [(k + BLOCK - 1) // BLOCK for k in kv]
    perm = torch.randperm(sum(n_blocks), generator=torch.Generator().manual_seed(seed)).tolist()
    cu_b, cu_q, cu_k = [0], [0], [0]
    for b, q, k in zip(n_blocks, new, kv):
        cu_b.append(cu_b[-1] + b)
        cu_q.append(cu_q[-1] + q)
        cu_k.append(cu_k[-1] + k)
    pos = [p for q, k in zip(new, kv) for p in range(k - q, k)]
    seq = [s for s, q in enumerate(new) for _ in range(q)]
    slots = [perm[cu_b[s] + p // BLOCK] * BLOCK + p % BLOCK for s, p in zip(seq, pos)]
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    return dict(n=sum(n_blocks), table=i(perm), cu_blocks=i(cu_b), q_cu=i(cu_q), k_cu=i(cu_k), pos=i(pos), seq=seq, slots=i(slots))


@pytest.mark.parametrize("new, kv", [([100], [100]), ([3, 0, 70, 1], [40, 9, 70, 33]), ([65] * 3, [65, 300, 129])])
@pytest.mark.parametrize("rows", [[0], [-1, 5, 5, 64], list(range(0, 64))], ids=lambda r: f"{len(r)} rows")
@pytest.mark.parametrize("wide", [True, False])
def test_prompt_rows(new, kv, rows, wide):
    from hydrainfer_amd import _lib
    b, T = _batch(new, kv, 1), sum(new)
    g = torch.Generator(device="cuda").manual_seed(T)
    x, h = (torch.randn(T, 264, generator=g, device="cuda").bfloat16() for _ in range(2))
    at = torch.tensor(rows, dtype=torch.int64 if wide else torch.int32, device="cuda")
    m = len(rows) + 1
    xs, hs, tables = torch.empty(len(rows), 264, dtype=x.dtype, device="cuda"), torch.empty(len(rows), 264, dtype=x.dtype, device="cuda"), torch.empty(4 * m - 1, dtype=torch.int32, device="cuda")
    _lib.check(_lib.lib().hx_prompt_rows(at.data_ptr(), int(wide), len(rows), T, len(new), b["q_cu"].data_ptr(), b["k_cu"].data_ptr(), b["cu_blocks"].data_ptr(), b["pos"].data_ptr(),
                                         x.data_ptr(), h.data_ptr(), xs.data_ptr(), hs.data_ptr(), 2 * 264, tables.data_ptr(), _lib.current_stream()), "prompt_rows")
    q_cu, kv_cu, cu_blocks, pos = tables[:m], tables[m:2 * m], tables[2 * m:3 * m], tables[3 * m:]
    want = [r % T for r in rows]
    assert torch.equal(xs, x[want]) and torch.equal(hs, h[want]) and torch.equal(pos, b["pos"][want])
    assert q_cu.tolist() == list(range(len(rows) + 1))
    keys = [int(b["pos"][r]) + 1 for r in want]
    assert kv_cu.tolist() == [sum(keys[:i]) for i in range(len(keys) + 1)]
    assert cu_blocks.tolist()[:-1] == [int(b["cu_blocks"][b["seq"][r]]) for r in want]


# sequences that begin and that continue, one of them without a sampled row, one sampled in its middle too; as many key heads as heads and fewer
@pytest.mark.parametrize("new, kv, rows", [([70], [70], [69]), ([40, 3, 30, 1], [40, 90, 333, 17], [39, 42, 73]), ([65, 66], [65, 200], [130, 64, 10])])
@pytest.mark.parametrize("heads, kv_heads", [(4, 4), (8, 2)])
@pytest.mark.parametrize("layers, dt", [(1, torch.bfloat16), (2, torch.float16)])
def test_sampled_rows_of_the_last_layer(new, kv, rows, heads, kv_heads, layers, dt):
    from hydrainfer_amd.layer.causal_attention import AttentionParameters
    from hydrainfer_amd.memory.kv_cache import KVCache
    from hydrainfer_amd.model.llama import LanguageModelParameters, LlamaForCausalLM, LlamaShape
    W, inner, D, vocab = 512, 1024, 128, 320
    g = torch.Generator(device="cuda").manual_seed(sum(new) + heads)
    w = lambda *s: torch.randn(s, generator=g, device="cuda").mul_(s[-1] ** -0.5).to(dt)
    state = {"embed": w(vocab, W), "lm_head": w(vocab, W), "norm": torch.ones(W, device="cuda", dtype=dt)}
    for l in range(layers):
        state.update({f"l{l}.wqkv": w((heads + 2 * kv_heads) * D, W), f"l{l}.wo": w(W, heads * D), f"l{l}.wgu": w(2 * inner, W), f"l{l}.wdown": w(W, inner),
                      f"l{l}.norm1": torch.ones(W, device="cuda", dtype=dt), f"l{l}.norm2": torch.ones(W, device="cuda", dtype=dt)})
    model = LlamaForCausalLM(LlamaShape(W, inner, layers, heads, kv_heads, D, vocab), dt, "cuda", state)
    b = _batch(new, kv, 3)
    ids = torch.randint(0, vocab, (sum(new),), generator=g, device="cuda")
    pool = torch.randn(layers, 2, b["n"], BLOCK, kv_heads, D, generator=g, device="cuda").to(dt)

    def through(sampled_only, rows):
        caches = pool.clone()
        model._sampled_rows_only = (lambda *a: took.append(LlamaForCausalLM._sampled_rows_only(model, *a)) or took[-1]) if sampled_only else lambda *a: False
        params = [AttentionParameters(kv_cache=KVCache(c[0], c[1]), q_cu_seq_lens=b["q_cu"], kv_cu_seq_lens=b["k_cu"], new_cache_slots=b["slots"], block_tables=b["table"],
                                      cu_blocks_lens=b["cu_blocks"], num_sequences=len(new), all_sequences_decode=False, q_max_seq_len=max(new), kv_max_seq_len=max(kv)) for c in caches]
        with torch.inference_mode():
            return model.forward_logits(ids, b["pos"], LanguageModelParameters(params, False, torch.tensor(rows, device="cuda"))), caches

    took = []
    got, got_caches = through(True, rows)
    assert took == [True]
    want, want_caches = through(False, rows)
    # the keys and values of every token: the same sums in another product's order, rounded
    half = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    assert float((got_caches.float() - want_caches.float()).norm() / want_caches.float().norm()) < half
    # attention and three products behind it, rounded each: 8 times half a unit in the last place
    assert float((got.float() - want.float()).norm() / want.float().norm()) < 8 * half


# the smallest and largest number of tokens that go this way, ragged portions with an empty one, as many key heads as heads and fewer, slabs of several splits and of none
@pytest.mark.parametrize("new, kv", [([65], [65]), ([40, 3, 0, 61], [40, 90, 17, 333]), ([300, 212], [300, 500])])
@pytest.mark.parametrize("heads, kv_heads, W, inner", [(4, 4, 512, 1024), (8, 2, 512, 640), (16, 16, 2048, 5632)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_layer_by_one_call(new, kv, heads, kv_heads, W, inner, dt):
    from hydrainfer_amd.layer.causal_attention import AttentionParameters
    from hydrainfer_amd.memory.kv_cache import KVCache
    from hydrainfer_amd.model.llama import LanguageModelParameters, LlamaForCausalLM, LlamaShape
    D, vocab, layers = 128, 320, 3
    g = torch.Generator(device="cuda").manual_seed(sum(new) + heads)
    w = lambda *s: torch.randn(s, generator=g, device="cuda").mul_(s[-1] ** -0.5).to(dt)
    norm = lambda: (1 + 0.1 * torch.randn(W, generator=g, device="cuda")).to(dt)
    state = {"embed": w(vocab, W), "lm_head": w(vocab, W), "norm": norm()}
    for l in range(layers):
        state.update({f"l{l}.wqkv": w((heads + 2 * kv_heads) * D, W), f"l{l}.wo": w(W, heads * D), f"l{l}.wgu": w(2 * inner, W), f"l{l}.wdown": w(W, inner), f"l{l}.norm1": norm(), f"l{l}.norm2": norm()})
    model = LlamaForCausalLM(LlamaShape(W, inner, layers, heads, kv_heads, D, vocab), dt, "cuda", state)
    b = _batch(new, kv, 3)
    ids = torch.randint(0, vocab, (sum(new),), generator=g, device="cuda")
    pool = torch.randn(layers, 2, b["n"], BLOCK, kv_heads, D, generator=g, device="cuda").to(dt)

    def through(one_call):
        caches = pool.clone()
        model._layer_of_few_prompts = (lambda *a: took.append(LlamaForCausalLM._layer_of_few_prompts(model, *a)) or took[-1]) if one_call else lambda *a: False
        params = [AttentionParameters(kv_cache=KVCache(c[0], c[1]), q_cu_seq_lens=b["q_cu"], kv_cu_seq_lens=b["k_cu"], new_cache_slots=b["slots"], block_tables=b["table"],
                                      cu_blocks_lens=b["cu_blocks"], num_sequences=len(new), all_sequences_decode=False, q_max_seq_len=max(new), kv_max_seq_len=max(kv)) for c in caches]
        with torch.inference_mode():
            return model.forward_logits(ids, b["pos"], LanguageModelParameters(params, False, torch.tensor([0, sum(new) - 1], device="cuda"))), caches

    took = []
    got, got_caches = through(True)
    assert took == [True] * (layers - 1)
    want, want_caches = through(False)
    assert torch.equal(got, want) and torch.equal(got_caches, want_caches)      # (the same launches)


def test_layer_that_the_call_does_not_take():
    from hydrainfer_amd._C.kernel.decode_step import prompt_layer
    n, W, inner, D, H = 600, 512, 1024, 128, 4                   # (more tokens than o is made of in these tiles)
    b = _batch([n], [n], 1)
    t = lambda *s: torch.randn(s, device="cuda").bfloat16()
    x, h, qkv, kc, vc = t(n, W), t(n, W), t(n, 3 * H * D), t(b["n"], BLOCK, H, D), t(b["n"], BLOCK, H, D)
    held = [y.clone() for y in (x, h, qkv, kc)]
    assert not prompt_layer(x, h, qkv, b["pos"], t(1024, 2, D // 2), kc, vc, b["slots"], b["q_cu"], b["k_cu"], b["table"], b["cu_blocks"], n, n, H, t(W, H * D), t(2 * inner, W), t(W, inner), t(W), t(W), D ** -0.5, 1e-5)
    assert all(torch.equal(y, z) for y, z in zip(held, (x, h, qkv, kc)))
