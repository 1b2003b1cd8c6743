"""Latent attention over portions of prompts (csrc/latent_attn.hip, the wide forms: 64 to 320 columns, 384 and 512) at the edges of
their tiles — 128 or 64 rows of token and head, 64 or 32 keys — with windows, sinks, gates, a negative scale, queries and results
as views of other layouts; and over single tokens, whose keys are dealt to several workgroups.  Every case says which form it is for."""
import math
from unittest import mock

import pytest
import torch

pytestmark = pytest.mark.gpu

BLOCK = 16
WIDE32, WIDE16 = 2, 3           # 32 rows a wave, 16 rows a wave
# (tokens brought, tokens held) of every sequence
BATCHES = [[(2, 2)], [(33, 33), (2, 100)], [(5, 70), (1, 200), (32, 32)], [(129, 129)], [(40, 400), (5, 5), (16, 64), (31, 63), (17, 17)]]


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("R", [64, 128, 192, 256, 320, 384, 512])
@pytest.mark.parametrize("H, window, extra", [(32, 0, "plain"), (3, 1, "plain"), (32, 31, "sinks"), (3, 0, "negative"), (32, 64, "sinks and gate")])
def test_wide_forms(batch, R, H, window, extra):
    new, kv = [a for a, _ in batch], [b for _, b in batch]
    if max(new) * H < 64:
        new[0], kv[0] = 22, max(22, kv[0])
    check(new, kv, R, H, window, extra, WIDE16)


# enough rows for 32 a wave (up to 192 columns), and for row tiles of 16 a wave that follow the largest score: several tiles a portion,
# whole ones and partial ones, portions of one tile beside them
MANY = [(130, 130), (1, 40), (129, 300), (128, 128), (131, 400), (97, 97), (133, 133), (64, 90)]


@pytest.mark.parametrize("R", [64, 128, 192, 256, 320])
@pytest.mark.parametrize("window, extra", [(0, "plain"), (1, "plain"), (64, "sinks and gate"), (31, "negative"), (0, "gate")])
def test_wide_forms_of_many_rows(R, window, extra):
    check([a for a, _ in MANY], [b for _, b in MANY], R, 32, window, extra, WIDE32 if R <= 192 else WIDE16)


# keys shared by two groups of waves (up to 320 columns, few row tiles): an odd and an even number of tiles, portions of one tile beside
# others, tiles that only one group's rows or neither's see
@pytest.mark.parametrize("batch", [[(150, 257)], [(160, 224), (70, 300), (1, 20)], [(400, 700)]], ids=lambda b: f"{len(b)}x{max(b)}")
@pytest.mark.parametrize("R", [64, 128, 192, 256, 320, 384])
@pytest.mark.parametrize("window, extra", [(0, "plain"), (0, "sinks and gate"), (200, "negative"), (160, "sinks")])
def test_two_groups_of_waves(batch, R, window, extra):
    check([a for a, _ in batch], [b for _, b in batch], R, 32, window, extra, WIDE16)


# single tokens: one tile and a split's edge, splits that get no tile (one sequence far shorter than another), more sequences than a
# round of the row tiles' search holds
STEPS = [[64], [129, 1, 32, 33], [2000, 3], [700] * 5, [40] * 260 + [130]]


@pytest.mark.parametrize("kv", STEPS, ids=lambda v: f"{len(v)}x{max(v)}")
@pytest.mark.parametrize("R", [64, 448, 512])
@pytest.mark.parametrize("H, window, extra", [(1, 0, "plain"), (16, 0, "negative"), (16, 300, "sinks and gate"), (65, 300, "plain")])
def test_single_tokens(kv, R, H, window, extra):
    check([1] * len(kv), kv, R, H, window, extra, WIDE32 if R <= 192 and len(kv) >= 256 else WIDE16)


# more keys in all than the form of single tokens takes: row tiles again, in three splits and in two
@pytest.mark.parametrize("kv", [[700] * 189 + [3], [450] * 299 + [64]], ids=lambda v: f"{len(v)}x{max(v)}")
@pytest.mark.parametrize("R, H, window, extra", [(256, 17, 0, "plain"), (320, 8, 0, "sinks and gate"), (512, 32, 400, "plain")])
def test_many_single_tokens(kv, R, H, window, extra):
    check([1] * len(kv), kv, R, H, window, extra, WIDE16)


# Rows that no token of a portion sees are never read: pages left of a window may have been given back, and the rows of the last page
# behind the last token hold anything.
@pytest.mark.parametrize("new, kv", [([1, 3, 1], [700, 1101, 40]), ([33, 20], [700, 90]), ([300, 41, 761], [700, 2005, 800])])
@pytest.mark.parametrize("R", [64, 320, 512])
@pytest.mark.parametrize("window", [300, 0])
def test_rows_that_nobody_sees(new, kv, R, window):
    check(new, kv, R, 32, window, "plain", WIDE32 if R <= 192 and max(new) > 700 else WIDE16, unseen=True)


@pytest.mark.parametrize("R, H", [(64, 32), (320, 16), (512, 32)])
@pytest.mark.parametrize("window", [300, 0])
def test_rows_that_no_single_token_sees(R, H, window):
    check([1] * 4, [700, 1101, 40, 1], R, H, window, "plain", WIDE16, unseen=True)


def hide(cache, table, first, last):
    """What lies outside of keys first .. last of a sequence becomes NaN; its pages there the last block of the cache, all NaN."""
    cache[-1] = math.nan
    for i, page in enumerate(table.tolist()):
        keys = torch.arange(i * BLOCK, (i + 1) * BLOCK)
        if i < first // BLOCK or i > last // BLOCK:
            table[i] = cache.shape[0] - 1
        else:
            cache[page, (keys < first) | (keys > last)] = math.nan


class Spy:
    """The library, noting which form every call takes."""
    def __init__(self, lib):
        self.lib, self.forms = lib, []

    def __getattr__(self, name):
        return getattr(self.lib, name)

    def hxm_latent_attention(self, args, stream):
        self.forms.append(self.lib.hxm_latent_attention_form(args))
        return self.lib.hxm_latent_attention(args, stream)


def check(new, kv, R, H, window, extra, form, unseen=False):
    from hydrainfer_amd import _lib
    from hydrainfer_amd._C.kernel.latent_attn import latent_attention
    g = torch.Generator().manual_seed(R * 100 + H + window + sum(new) + sum(kv))
    nb = [(n + BLOCK - 1) // BLOCK for n in kv]
    T, perm = sum(new), torch.randperm(sum(nb) + (0 if unseen else 1), generator=g)
    cache = torch.randn((sum(nb) + 1, BLOCK, 1, R + 8), generator=g).bfloat16()      # rows wider than the latent
    q = torch.randn((H, T, R), generator=g).bfloat16()
    q[0, 0] *= 20                 # a row whose weights sit on one key
    scale = (-1.0 if extra == "negative" else 1.0) * R ** -0.5
    sinks = 2 * torch.randn(H, generator=g) if "sinks" in extra else None
    gate = torch.randn((T, H + 5), generator=g).bfloat16() if "gate" in extra else None
    cu_b, cu_q = torch.tensor([0] + nb).cumsum(0).int(), torch.tensor([0] + new).cumsum(0).int()
    pos = [p for a, b in zip(new, kv) for p in (range(b - a, b) if a % 2 else torch.randint(0, b, (a,), generator=g).tolist())]      # (even portions: in no order)
    seq = torch.tensor([s for s, a in enumerate(new) for _ in range(a)], dtype=torch.int32)
    table = perm[:sum(nb)].int()
    c = lambda t: None if t is None else t.cuda()
    shown, pages = cache.clone(), table.clone()
    if unseen:
        for s in range(len(new)):
            rows = pos[int(cu_q[s]):int(cu_q[s + 1])]
            hide(shown, pages[int(cu_b[s]):int(cu_b[s + 1])], max(0, min(rows) - window + 1) if window else 0, max(rows))
    out = torch.full((H, T, R), 7.0, dtype=torch.bfloat16, device="cuda")
    spy = Spy(_lib.mix_lib())
    with mock.patch.object(_lib, "mix_lib", lambda: spy):
        latent_attention(c(q).transpose(0, 1), c(shown), c(seq), c(torch.tensor(pos, dtype=torch.int32)), c(cu_q), c(pages), c(cu_b), scale, window or None,
                         max(new), gate_pre=c(gate), out=out.transpose(0, 1), max_kv_len=max(kv), sinks=c(sinks))
    assert spy.forms == [form]
    got = out.double().cpu()
    for s in range(len(new)):
        lo, hi = int(cu_q[s]), int(cu_q[s + 1])
        k = cache[table[int(cu_b[s]):int(cu_b[s + 1])].long()].reshape(-1, R + 8)[:kv[s], :R].double()
        z = torch.matmul(q[:, lo:hi].double(), k.t()) * scale
        far = torch.tensor(pos[lo:hi])[:, None] - torch.arange(kv[s])[None, :]
        z = z.masked_fill(((far < 0) | (far >= window if window else far < 0))[None], -math.inf)
        if sinks is not None:
            z = torch.cat([z, sinks.double()[:, None, None].expand(-1, hi - lo, 1)], dim=2)
        p = torch.softmax(z, dim=2)[:, :, :kv[s]]
        f = torch.sigmoid(gate[lo:hi, :H].double()).t()[:, :, None] if gate is not None else 1.0
        want, size = torch.matmul(p, k) * f, torch.matmul(p, k.abs()) * f
        # the weights and the result are rounded to bfloat16 once each: eight significant bits, so by up to 2^-8 of themselves; 1e-6 of what
        # is summed for the float arithmetic
        bound = 2.0 ** -8 * want.abs() + (2.0 ** -8 + 1e-6) * size + 1e-6
        off = (got[:, lo:hi] - want).abs()
        assert bool((off <= bound).all()), (s, float((off - bound).max()))


@pytest.mark.parametrize("R, tokens", [(64, 1100), (512, 30), (512, 1)])
def test_a_scale_that_is_no_number_shows(R, tokens):
    from hydrainfer_amd._C.kernel.latent_attn import latent_attention
    H, nb = 32, (tokens + 200 + BLOCK - 1) // BLOCK
    g = torch.Generator().manual_seed(R)
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    out = latent_attention(torch.randn((tokens, H, R), generator=g).bfloat16().cuda(), torch.randn((nb, BLOCK, 1, R), generator=g).bfloat16().cuda(), i([0] * tokens),
                           i(list(range(200, 200 + tokens))), i([0, tokens]), i(list(range(nb))), i([0, nb]), math.nan, None, tokens, max_kv_len=200 + tokens)
    assert torch.isnan(out).all()


@pytest.mark.parametrize("R, n", [(512, 1), (64, 1100)])
def test_a_sequence_without_keys(R, n):
    # its tokens stand in front of its first key (position -1) and it has no pages: nothing is looked up for it
    from hydrainfer_amd._C.kernel.latent_attn import latent_attention
    H, nb = 32, (n + 500) // BLOCK
    g = torch.Generator().manual_seed(n)
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    q, cache = torch.randn((2 * n, H, R), generator=g).bfloat16().cuda(), torch.randn((nb, BLOCK, 1, R), generator=g).bfloat16().cuda()
    table, sinks = i(list(range(nb))), torch.randn(H, generator=g).cuda()
    run = lambda q, pos, q_cu, blocks, seq: latent_attention(q, cache, i(seq), i(pos), i(q_cu), table, i(blocks), R ** -0.5, None, n, max_kv_len=n + 400, sinks=sinks)
    own = list(range(400, 400 + n))
    got = run(q, [-1] * n + own, [0, n, 2 * n], [0, 0, nb], [0] * n + [1] * n)
    alone = run(q[n:], own, [0, n], [0, nb], [0] * n)
    assert (got[:n] == 0).all()                                   # the sink takes all the weight
    assert float((got[n:].double() - alone.double()).norm() / alone.double().norm()) < 2.0 ** -7      # (keys may be dealt out otherwise)


def test_rows_past_max_q_len_have_no_place_in_the_workspace():
    import ctypes
    from hydrainfer_amd import _lib
    H, R, new, kv = 32, 512, 3, 1000
    nb = (kv + BLOCK - 1) // BLOCK
    g = torch.Generator().manual_seed(1)
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    q, cache = torch.randn((new, H, R), generator=g).bfloat16().cuda(), torch.randn((nb, BLOCK, 1, R), generator=g).bfloat16().cuda()
    out = torch.empty_like(q)
    ints = dict(tok_seq=i([0] * new), positions=i(list(range(kv - new, kv))), q_cu=i([0, new]), block_table=i(list(range(nb))), cu_block_lens=i([0, nb]))
    a = _lib.hxm_latent_attn_args(out=out.data_ptr(), q=q.data_ptr(), cache=cache.data_ptr(), q_token_stride=H * R, q_head_stride=R, out_token_stride=H * R,
                                  out_head_stride=R, cache_block_stride=BLOCK * R, cache_row_stride=R, block_size=BLOCK, n_tokens=new, n_seq=1, n_heads=H, kv_rank=R,
                                  max_q_len=1, max_kv_len=kv, scale=R ** -0.5, dtype=_lib.dtype_code(q),
                                  **{k: v.data_ptr() for k, v in ints.items()})
    splits, floats = ctypes.c_int32(0), ctypes.c_int64(0)
    _lib.mix_check(_lib.mix_lib().hxm_latent_attention_plan(ctypes.byref(a), ctypes.byref(splits), ctypes.byref(floats)), "plan")
    assert splits.value > 1
    n_o = floats.value // (R + 2) * R
    ws_o, ws_ml = (torch.full((4 * n,), 7.0, device="cuda") for n in (n_o, floats.value - n_o))      # three tokens would fill three quarters
    a.n_splits, a.ws_o, a.ws_ml = splits.value, ws_o.data_ptr(), ws_ml.data_ptr()
    _lib.mix_check(_lib.mix_lib().hxm_latent_attention(ctypes.byref(a), _lib.current_stream()), "latent_attention")
    assert (ws_o[n_o:] == 7.0).all() and (ws_ml[floats.value - n_o:] == 7.0).all()


# (sequences, tokens brought, tokens held)
@pytest.mark.parametrize("n, new, kv", [(2, 60, 60), (8, 140, 300), (64, 1, 900), (4, 16, 516)])
@pytest.mark.parametrize("R", [64, 256, 512])
def test_weights_round_no_more_than_in_the_tile_form(n, new, kv, R):
    # The tile form's weights refer to the largest score so far, 32 keys at a time.  So do the wide forms', and round alike; where the keys
    # are dealt out they refer to the largest of their own 32, and are compared over 2048 rows (two roundings of one row differ by a
    # fifth or so).
    from hydrainfer_amd import _lib
    from hydrainfer_amd._C.kernel.latent_attn import latent_attention
    H, nb = 32, (kv + BLOCK - 1) // BLOCK
    g = torch.Generator().manual_seed(R + n + new + kv)
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    q, cache = torch.randn((n * new, H, R), generator=g).bfloat16(), torch.randn((n * nb, BLOCK, 1, R), generator=g).bfloat16()
    pos = list(range(kv - new, kv))
    seen = torch.tensor(pos)[:, None] >= torch.arange(kv)[None, :]
    want = []
    for s in range(n):
        k = cache[s * nb:(s + 1) * nb].reshape(-1, R)[:kv].double()
        z = torch.matmul(q[s * new:(s + 1) * new].double(), k.t()) * R ** -0.5
        want.append(torch.matmul(torch.softmax(z.masked_fill(~seen[:, None], -math.inf), dim=2), k))
    want, off = torch.cat(want), {}
    try:
        for form in (1, 2):
            _lib.mix_lib().hxm_set_option(b"attn_tile_form", form)
            got = latent_attention(q.cuda(), cache.cuda(), i([s for s in range(n) for _ in pos]), i(pos * n), i([s * new for s in range(n + 1)]), i(list(range(n * nb))),
                                   i([s * nb for s in range(n + 1)]), R ** -0.5, None, new, max_kv_len=kv).double().cpu()
            off[form] = float((got - want).norm() / want.norm())
    finally:
        _lib.mix_lib().hxm_set_option(b"attn_tile_form", 1)
    assert off[1] <= (1.0 if new < 20 else 1.005) * off[2], off


# Batches of single tokens of up to 32 heads: one group of heads and two, tiles in two, three and four places, keys up to a tile's and a group's edge and past it,
# splits of one tile and of several, pages whose size is no power of two, sequences that bring no token, tokens in another order than their sequences.
@pytest.mark.parametrize("kv", [[64, 0, 65, 1], [16, 17, 300, 513], [1040] + [90] * 20], ids=["edges", "few", "splits"])
@pytest.mark.parametrize("R, H, block", [(64, 16, 16), (128, 17, 48), (192, 32, 16), (320, 32, 48), (384, 9, 16), (512, 32, 32)])
@pytest.mark.parametrize("window, extra", [(0, "plain"), (63, "sinks and gate"), (500, "negative")])
def test_steps_of_single_tokens(kv, R, H, block, window, extra):
    from hydrainfer_amd._C.kernel.latent_attn import latent_attention
    g = torch.Generator().manual_seed(R + H + window + sum(kv))
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    seqs = [s for s, n in enumerate(kv) if n]
    if len(seqs) == len(kv):
        seqs.reverse()                            # (q_cu says nothing to these launches but how many sequences there are)
    nb = [(n + block - 1) // block for n in kv]
    cu_b = [sum(nb[:s]) for s in range(len(kv) + 1)]
    cache, q = torch.randn((sum(nb), block, 1, R), generator=g).bfloat16(), torch.randn((len(seqs), H, R), generator=g).bfloat16()
    q[0, 0] *= 20
    table = torch.randperm(sum(nb), generator=g)
    scale = (-1.0 if extra == "negative" else 1.0) * R ** -0.5
    sinks = 2 * torch.randn(H, generator=g) if "sinks" in extra else None
    gate = torch.randn((len(seqs), H), generator=g).bfloat16() if "gate" in extra else None
    q_cu = [sum(1 for s in seqs if s < x) for x in range(len(kv) + 1)]
    c = lambda t: None if t is None else t.cuda()
    got = latent_attention(c(q), c(cache), i(seqs), i([kv[s] - 1 for s in seqs]), i(q_cu), c(table.int()), i(cu_b), scale, window or None, 1, gate_pre=c(gate),
                           max_kv_len=max(kv), sinks=c(sinks)).double().cpu()
    for t, s in enumerate(seqs):
        k = cache[table[cu_b[s]:cu_b[s + 1]]].reshape(-1, R)[:kv[s]].double()[-window if window else 0:]
        z = torch.matmul(q[t].double(), k.t()) * scale
        if sinks is not None:
            z = torch.cat([z, sinks.double()[:, None]], dim=1)
        p = torch.softmax(z, dim=1)[:, :k.shape[0]]
        f = torch.sigmoid(gate[t].double())[:, None] if gate is not None else 1.0
        want, size = torch.matmul(p, k) * f, torch.matmul(p, k.abs()) * f
        # the result is rounded to bfloat16 once, the weights are sums of two bfloat16 numbers (2^-17); 1e-5 of what is summed for that and
        # the float arithmetic
        off = (got[t] - want).abs()
        assert bool((off <= 2.0 ** -8 * want.abs() + 1e-5 * size + 1e-6).all()), (t, float((off - 2.0 ** -8 * want.abs() - 1e-5 * size).max()))
