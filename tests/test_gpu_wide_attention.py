"""Biased attention over portions of prompts with heads of 64 and 128 (csrc/biased_attn.hip, the wide form) at the edges of its
tiles — 128 rows of a key head, 64 keys — under every mask, with slopes, soft caps, temperatures of either sign and of zero,
sinks, and other key than value sizes; and over single tokens and a few (the step form: 16 rows, 32 keys), their keys dealt to several
waves or not."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

BLOCK = 16


def _first(mask, size, p):
    return max(0, p - size + 1) if mask == "window" else p // size * size if mask == "chunk" else 0


def _reference(q, k, v, pos, scale, slopes, mask, size, cap, sinks):
    """(result, bound) for one sequence: q [n, H, D], k [keys, H, D], v [keys, H, V] in double"""
    s = torch.einsum("nhd,khd->hnk", q, k) * scale[:, None, None]
    if cap:
        s = cap * torch.tanh(s / cap)
    j = torch.arange(k.shape[0])
    far = (torch.tensor(pos)[:, None] - j[None, :]).double()
    if slopes is not None:
        s = s - slopes[:, None, None] * far
    seen = (far >= 0) & (j[None, :] >= torch.tensor([_first(mask, size, p) for p in pos])[:, None])
    s = s.masked_fill(~seen[None], -math.inf)
    if sinks is not None:
        s = torch.cat([s, sinks[:, None, None].expand(-1, s.shape[1], 1)], dim=2)
    p = torch.softmax(s, dim=2)[:, :, :k.shape[0]]
    out = torch.einsum("hnk,khv->nhv", p, v)
    # the weights and the result are rounded to bfloat16 once each: eight significant bits, so by up to 2^-8 of themselves (half of the
    # last place, 2^-7, of a number just above a power of two); 1e-6 of what is summed for the float arithmetic
    return out, 2.0 ** -8 * out.abs() + (2.0 ** -8 + 1e-6) * torch.einsum("hnk,khv->nhv", p, v.abs()) + 1e-6


# (tokens brought, tokens held) of every sequence
BATCHES = [[(16, 16)], [(31, 31), (33, 100)], [(64, 65), (1, 200), (32, 32)], [(129, 129)], [(127, 400), (5, 5), (16, 64), (40, 63), (17, 17)]]


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("H, G, D, V", [(4, 1, 128, 128), (32, 8, 64, 64), (6, 2, 128, 64), (16, 16, 64, 128)])
@pytest.mark.parametrize("mask, size, extra", [("causal", 0, "plain"), ("window", 1, "plain"), ("window", 63, "slopes"), ("chunk", 48, "cap"),
                                               ("causal", 0, "cap"), ("chunk", 48, "temperatures and sinks"), ("causal", 0, "temperatures and sinks")])
def test_wide_form(batch, H, G, D, V, mask, size, extra):
    new, kv = [a for a, _ in batch], [b for _, b in batch]
    if max(new) * (H // G) < 64:
        new[0], kv[0] = 64, max(64, kv[0])
    check(new, kv, H, G, D, V, mask, size, extra)


# the same among portions so uneven that the longest one speaks for more row tiles than there are
@pytest.mark.parametrize("H, G, D, V", [(32, 8, 64, 64), (32, 32, 128, 128), (32, 16, 64, 128)])
@pytest.mark.parametrize("mask, size, extra", [("causal", 0, "plain"), ("window", 200, "slopes"), ("chunk", 130, "temperatures and sinks")])
def test_two_groups_of_waves_among_uneven_portions(H, G, D, V, mask, size, extra):
    check([601, 20, 33, 7], [601, 90, 33, 300], H, G, D, V, mask, size, extra)


# equal portions in as many workgroups as there are compute units, and in a few more, which one group of waves each takes
@pytest.mark.parametrize("batch", [[(65, 70)] * 16, [(65, 70)] * 17], ids=lambda b: f"{len(b)}x{max(b)}")
@pytest.mark.parametrize("H, G, D, V, mask, size", [(16, 16, 64, 64, "causal", 0), (32, 16, 128, 128, "window", 66)])
def test_groups_of_waves_by_the_number_of_workgroups(batch, H, G, D, V, mask, size):
    check([a for a, _ in batch], [b for _, b in batch], H, G, D, V, mask, size, "plain")


# keys shared by two groups of waves: one tile, two, three, an odd and an even number of them, tiles that only one group's rows or neither's see
@pytest.mark.parametrize("batch", [[(65, 65)], [(66, 128)], [(100, 129)], [(70, 257), (200, 200), (1, 64)], [(129, 705)]], ids=lambda b: f"{len(b)}x{max(b)}")
@pytest.mark.parametrize("H, G, D, V", [(4, 1, 128, 128), (8, 8, 64, 64), (6, 2, 128, 64), (4, 4, 64, 128)])
@pytest.mark.parametrize("mask, size, extra", [("causal", 0, "plain"), ("window", 70, "slopes"), ("chunk", 128, "cap"), ("window", 3, "temperatures and sinks")])
def test_two_groups_of_waves(batch, H, G, D, V, mask, size, extra):
    check([a for a, _ in batch], [b for _, b in batch], H, G, D, V, mask, size, extra)


# single tokens at the edges of tiles and splits, sequences far shorter than others, two row tiles, more keys in one run than a wave
# holds pages of (1024), sixteen tokens behind many keys
STEPS = [[(1, 1)], [(1, 32), (1, 33), (1, 200), (1, 1025)], [(3, 70), (1, 16), (7, 2300)], [(1, 100)] * 40, [(16, 1500), (2, 40)]]


@pytest.mark.parametrize("batch", STEPS, ids=lambda b: f"{len(b)}x{max(b)}")
@pytest.mark.parametrize("H, G, D, V", [(4, 1, 128, 128), (32, 8, 64, 64), (6, 2, 128, 64), (16, 16, 64, 128), (17, 1, 128, 128)])
@pytest.mark.parametrize("mask, size, extra", [("causal", 0, "plain"), ("window", 63, "slopes"), ("chunk", 48, "cap"), ("causal", 0, "temperatures and sinks")])
@pytest.mark.parametrize("divided", [True, False])
def test_step_form(batch, H, G, D, V, mask, size, extra, divided):
    check([a for a, _ in batch], [b for _, b in batch], H, G, D, V, mask, size, extra, divided)


# two and four runs of keys a workgroup, and three workgroups of four: runs without keys, rows that some of them do not see, partial row tiles
@pytest.mark.parametrize("batch", [[(1, 140), (1, 1), (5, 64)], [(1, 250), (1, 3), (2, 33)], [(1, 511), (3, 40), (1, 129)], [(2, 600), (1, 65), (1, 1)]], ids=lambda b: f"{len(b)}x{max(b)}")
@pytest.mark.parametrize("H, G, D, V", [(4, 1, 128, 128), (32, 8, 64, 64), (6, 2, 128, 64), (16, 16, 64, 128)])
@pytest.mark.parametrize("mask, size, extra", [("causal", 0, "plain"), ("window", 300, "slopes"), ("chunk", 257, "cap"), ("causal", 0, "temperatures and sinks")])
def test_step_form_merged_in_place(batch, H, G, D, V, mask, size, extra):
    check([a for a, _ in batch], [b for _, b in batch], H, G, D, V, mask, size, extra)


# every way that a row tile's splits are dealt out: by twos and fours in one workgroup, two workgroups of four, and single waves with a launch that merges
# (three and four splits of 257 - 383 row tiles, seven of just more than 128)
@pytest.mark.parametrize("kv, H, G, D, V, splits", [
    ([200] * 15 + [1], 32, 8, 128, 128, 4), ([127, 100, 3], 32, 8, 64, 64, 2), ([160, 128], 8, 8, 128, 64, 2), ([700, 512, 33] * 2, 32, 8, 64, 128, 12),
    ([2048] * 3 + [1, 40, 1999] + [500] * 10, 32, 8, 128, 128, 8), ([700] * 39 + [1], 32, 8, 128, 128, 4), ([700] * 46 + [2], 32, 8, 64, 128, 3),
    ([2101] + [700] * 15 + [64], 32, 8, 128, 64, 7), ([2600, 1, 300] + [90] * 15, 16, 8, 64, 64, 7)], ids=lambda v: f"{len(v)}x{max(v)}" if isinstance(v, list) else str(v))
@pytest.mark.parametrize("extra", ["plain", "slopes", "temperatures and sinks"])
def test_step_form_by_its_splits(kv, H, G, D, V, splits, extra):
    import ctypes
    from hydrainfer_amd import _lib
    a = _lib.hxm_biased_attn_args(n_tokens=len(kv), n_seq=len(kv), n_heads=H, kv_heads=G, dim=D, vdim=V, block_size=BLOCK, max_q_len=1, dtype=_lib._DTYPE[torch.bfloat16])
    n, floats = ctypes.c_int32(), ctypes.c_int64()
    assert _lib.mix_lib().hxm_biased_attention_plan(ctypes.byref(a), max(kv), ctypes.byref(n), ctypes.byref(floats)) == 0 and n.value == splits
    check([1] * len(kv), kv, H, G, D, V, "causal", 0, extra)


# Rows that no token of a portion sees are never read: pages left of a window or chunk may have been given back, and the rows of the last
# page behind the last token hold anything.
@pytest.mark.parametrize("batch", [[(64, 700), (33, 1100)], [(129, 333)], [(1, 700), (3, 1101), (1, 40)], [(16, 2005)]], ids=lambda b: f"{len(b)}x{max(b)}")
@pytest.mark.parametrize("H, G, D, V", [(6, 2, 128, 64), (8, 8, 64, 128)])
@pytest.mark.parametrize("mask, size", [("window", 300), ("chunk", 500), ("causal", 0)])
@pytest.mark.parametrize("divided", [True, False])
def test_rows_that_nobody_sees(batch, H, G, D, V, mask, size, divided):
    check([a for a, _ in batch], [b for _, b in batch], H, G, D, V, mask, size, "plain", divided, unseen=True)


def hide(cache, table, first, last):
    """What lies outside of keys first .. last of a sequence becomes NaN; its pages there the last block of the cache, all NaN."""
    cache[-1] = math.nan
    for i, page in enumerate(table.tolist()):
        keys = torch.arange(i * BLOCK, (i + 1) * BLOCK)
        if i < first // BLOCK or i > last // BLOCK:
            table[i] = cache.shape[0] - 1
        else:
            cache[page, (keys < first) | (keys > last)] = math.nan


def check(new, kv, H, G, D, V, mask, size, extra, divided=True, unseen=False):
    from hydrainfer_amd._C.kernel.biased_attn import biased_attention
    g = torch.Generator().manual_seed(H * D + V + size + sum(new) + sum(kv))
    nb = [(n + BLOCK - 1) // BLOCK for n in kv]
    perm = torch.randperm(sum(nb) + (0 if unseen else 1), generator=g)
    r = lambda *s: torch.randn(s, generator=g).bfloat16()
    hs = max(D, V)
    T, kc, vc = sum(new), r(sum(nb) + 1, BLOCK, G, hs), r(sum(nb) + 1, BLOCK, G, hs)
    q = r(T, H, D)
    q[0] *= 20                    # a row whose weights sit on one key
    slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)]) if "slopes" in extra else None
    if "steep" in extra:
        slopes *= 1e5
    cap = 1e5 if extra == "a cap far above the scores" else 4.0 if "cap" in extra else 0.0
    temps = sinks = None
    if "temperatures and sinks" in extra:
        temps, sinks = torch.randn(H, generator=g), 2 * torch.randn(H, generator=g)
        temps[0], sinks[1] = 0.0, -math.inf
    cu_b = torch.tensor([0] + nb).cumsum(0).int()
    cu_q = torch.tensor([0] + new).cumsum(0).int()
    pos = [p for a, b in zip(new, kv) for p in (range(b - a, b) if a % 2 else torch.randint(0, b, (a,), generator=g).tolist())]      # (even portions: in no order)
    seq = torch.tensor([s for s, a in enumerate(new) for _ in range(a)], dtype=torch.int32)
    table = perm[:sum(nb)].int()
    c = lambda t: None if t is None else t.cuda()
    kg, vg, pages = kc.clone(), vc.clone(), table.clone()
    if unseen:
        for s in range(len(new)):
            own, rows = slice(int(cu_b[s]), int(cu_b[s + 1])), pos[int(cu_q[s]):int(cu_q[s + 1])]
            for x, t in ((kg, table[own].clone()), (vg, pages[own])):
                hide(x, t, min(_first(mask, size, p) for p in rows), max(rows))
    got = biased_attention(c(q), c(kg), c(vg), V, c(seq), c(torch.tensor(pos, dtype=torch.int32)), c(cu_q), c(pages), c(cu_b), D ** -0.5, c(slopes), mask,
                           size, max_q_len=max(new), max_kv_len=max(kv) if divided else 0, softcap=cap, head_scale=c(temps), sinks=c(sinks)).double().cpu()
    for s in range(len(new)):
        lo, hi = int(cu_q[s]), int(cu_q[s + 1])
        pages = table[int(cu_b[s]):int(cu_b[s + 1])].long()
        k, v = (x[pages].reshape(-1, G, hs)[:kv[s]].double().repeat_interleave(H // G, dim=1) for x in (kc, vc))
        scale = torch.full((H,), D ** -0.5, dtype=torch.float64) * (temps.double() if temps is not None else 1.0)
        want, bound = _reference(q[lo:hi].double(), k[..., :D], v[..., :V], pos[lo:hi], scale, None if slopes is None else slopes.double(), mask, size, cap,
                                 None if sinks is None else sinks.double())
        off = (got[lo:hi] - want).abs()
        assert bool((off <= bound).all()), (s, float((off - bound).max()))


# slopes, a cap, temperatures and sinks at once; and slopes so steep that the token's own key and the sink share the weights: that key is
# at distance 0, where no slope adds a rounding
@pytest.mark.parametrize("batch", [[(64, 65), (1, 200), (32, 32)], [(129, 129)], [(3, 70), (1, 16), (7, 2300)]], ids=lambda b: f"{len(b)}x{max(b)}")
@pytest.mark.parametrize("H, G, D, V", [(4, 1, 128, 128), (32, 8, 64, 64), (6, 2, 128, 64)])
@pytest.mark.parametrize("mask, size, extra", [("window", 63, "slopes and cap"), ("causal", 0, "slopes, cap, temperatures and sinks"),
                                               ("causal", 0, "steep slopes, temperatures and sinks")])
def test_slopes_with_the_other_extras(batch, H, G, D, V, mask, size, extra):
    check([a for a, _ in batch], [b for _, b in batch], H, G, D, V, mask, size, extra)


# a score is rounded as itself, not as a share of the cap (1e5 / 2^24 would move a weight by 1 %)
@pytest.mark.parametrize("batch", [[(64, 65), (1, 200)], [(300, 1100)] * 8, [(1, 32), (1, 1025)]], ids=lambda b: f"{len(b)}x{max(b)}")
@pytest.mark.parametrize("H, G, D, V", [(4, 1, 128, 128), (32, 8, 64, 64)])
def test_a_cap_far_above_the_scores(batch, H, G, D, V):
    check([a for a, _ in batch], [b for _, b in batch], H, G, D, V, "causal", 0, "a cap far above the scores")


@pytest.mark.parametrize("new, kv", [([40, 16], [40, 300]), ([1, 1], [40, 300])])
@pytest.mark.parametrize("divided", [True, False])
def test_a_temperature_that_is_no_number_shows(new, kv, divided):
    from hydrainfer_amd._C.kernel.biased_attn import biased_attention
    H, G, D = 8, 2, 64
    g = torch.Generator().manual_seed(sum(new))
    r = lambda *s: torch.randn(s, generator=g).bfloat16().cuda()
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    nb = [(n + BLOCK - 1) // BLOCK for n in kv]
    pos = [p for a, b in zip(new, kv) for p in range(b - a, b)]
    temps = torch.rand(H, generator=g) + 0.5
    temps[3] = math.nan
    out = biased_attention(r(sum(new), H, D), r(sum(nb), BLOCK, G, D), r(sum(nb), BLOCK, G, D), D, i([s for s, a in enumerate(new) for _ in range(a)]), i(pos),
                           i([0, new[0], sum(new)]), i(list(range(sum(nb)))), i([0, nb[0], sum(nb)]), D ** -0.5, None, "causal", 0, max_q_len=max(new),
                           max_kv_len=max(kv) if divided else 0, head_scale=temps.cuda()).view(-1, H, D)
    assert torch.isnan(out[:, 3]).all() and torch.isfinite(out[:, [h for h in range(H) if h != 3]]).all()


@pytest.mark.parametrize("n", [1, 40])
@pytest.mark.parametrize("divided", [True, False])
def test_a_sequence_without_keys(n, divided):
    # its tokens stand in front of its first key (position -1) and it has no pages: nothing is looked up for it
    from hydrainfer_amd._C.kernel.biased_attn import biased_attention
    H, G, D = 8, 2, 128
    g = torch.Generator().manual_seed(n)
    r = lambda *s: torch.randn(s, generator=g).bfloat16().cuda()
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    q, kc, vc = r(2 * n, H, D), r(30, BLOCK, G, D), r(30, BLOCK, G, D)
    table, sinks = i(list(range(30))), torch.randn(H, generator=g).cuda()
    run = lambda q, pos, q_cu, blocks, seq: biased_attention(q, kc, vc, D, i(seq), i(pos), i(q_cu), table, i(blocks), D ** -0.5, None, "causal", 0, max_q_len=n,
                                                             max_kv_len=480 if divided else 0, sinks=sinks).view(-1, H, D)
    own = list(range(480 - n, 480))
    got = run(q, [-1] * n + own, [0, n, 2 * n], [0, 0, 30], [0] * n + [1] * n)
    alone = run(q[n:].contiguous(), own, [0, n], [0, 30], [0] * n)
    assert (got[:n] == 0).all()                                   # the sink takes all the weight
    assert float((got[n:].double() - alone.double()).norm() / alone.double().norm()) < 2.0 ** -7      # (keys may be dealt out otherwise)


# (sequences, tokens brought, tokens held)
@pytest.mark.parametrize("n, new, kv", [(2, 64, 64), (2, 250, 300), (1, 200, 700), (64, 1, 900)])
@pytest.mark.parametrize("extra", ["plain", "slopes", "cap"])
def test_weights_round_no_more_than_in_the_tile_form(n, new, kv, extra):
    # The tile form's weights refer to the largest score so far, 32 keys at a time.  So do the wide form's, and round alike; the step
    # form's refer to the largest of their own 32, and are compared over 2048 rows (two roundings of one row differ by a fifth or so).
    from hydrainfer_amd._C.kernel.biased_attn import biased_attention
    H, G, D = 32, 8, 128
    g = torch.Generator().manual_seed(n + new + kv)
    nb = (kv + BLOCK - 1) // BLOCK
    r = lambda *s: torch.randn(s, generator=g).bfloat16()
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    q, kc, vc = r(n * new, H, D), r(n * nb, BLOCK, G, D), r(n * nb, BLOCK, G, D)
    slopes, cap = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)]) if extra == "slopes" else None, 30.0 if extra == "cap" else 0.0
    pos = list(range(kv - new, kv))
    want = []
    for s in range(n):
        k, v = (x[s * nb:(s + 1) * nb].reshape(-1, G, D)[:kv].double().repeat_interleave(H // G, dim=1) for x in (kc, vc))
        want.append(_reference(q[s * new:(s + 1) * new].double(), k, v, pos, torch.full((H,), D ** -0.5, dtype=torch.float64),
                               None if slopes is None else slopes.double(), "causal", 0, cap, None)[0])
    want = torch.cat(want)
    off = {}
    for form in ("auto", "tile"):
        got = biased_attention(q.cuda(), kc.cuda(), vc.cuda(), D, i([s for s in range(n) for _ in pos]), i(pos * n), i([s * new for s in range(n + 1)]), i(list(range(n * nb))),
                               i([s * nb for s in range(n + 1)]), D ** -0.5, None if slopes is None else slopes.cuda(), "causal", 0, max_q_len=new, max_kv_len=kv,
                               softcap=cap, form=form).double().cpu()
        off[form] = float((got - want).norm() / want.norm())
    assert off["auto"] <= (1.0 if new == 1 else 1.005) * off["tile"], off


# What a row adds up: a key weighs 1 and others w, halfway between two bfloat16 numbers, and everything else nothing.  "sum": 31 of them in the
# 32 keys of the one with a value, whose share 1 / (1 + 31 w) shows a denominator of rounded weights (off by up to 2^-8); "share": one of them, with the
# value, in the 32 keys in front, where it is the largest score so far: w / (1 + w), and no rounding of w.  So the result's rounding is all there is.
@pytest.mark.parametrize("what", ["sum", "share"])
@pytest.mark.parametrize("n", [1, 16], ids=["few", "many"])
@pytest.mark.parametrize("D, V", [(64, 64), (128, 128)])
def test_weights_that_no_bfloat16_holds(what, n, D, V):
    from hydrainfer_amd._C.kernel.biased_attn import biased_attention
    H, kv = 8, 256
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    w = torch.tensor([(0.5 if what == "sum" else 2.0 ** -4) * (1 + (2 * h + 1) * 2.0 ** -8) for h in range(H)], dtype=torch.float64)
    temps = -torch.log(w).float()
    k, v, q = torch.zeros((kv, D)), torch.zeros((kv, V)), torch.zeros((n * kv, H, D))
    q[:, :, 0] = 1
    k[:, 0] = -1000
    if what == "sum":
        k[192:224, 0], k[200, 0], v[200] = -1, 0, 1
        want = 1 / (1 + 31 * w)
    else:
        k[197, 0], k[229, 0], v[197] = -1, 0, 1
        want = w / (1 + w)
    pages = lambda x: x.bfloat16()[:, None].expand(-1, H, -1).contiguous().view(kv // BLOCK, BLOCK, H, -1).repeat(n, 1, 1, 1).cuda()
    out = biased_attention(q.bfloat16().cuda(), pages(k), pages(v), V, i([s for s in range(n) for _ in range(kv)]), i(list(range(kv)) * n), i([kv * s for s in range(n + 1)]),
                           i(list(range(n * kv // BLOCK))), i([kv // BLOCK * s for s in range(n + 1)]), 1.0, None, "causal", 0, max_q_len=kv, max_kv_len=kv,
                           head_scale=temps.cuda()).view(n, kv, H, V)[:, 230:].double().cpu()
    # half of a last place of bfloat16, and 1e-5 for the float arithmetic (an exponential of scores up to 3)
    bound = 2.0 ** (torch.floor(torch.log2(want)) - 8) + 1e-5 * want
    off = (out - want[:, None]).abs().amax(dim=(0, 1, 3))
    assert bool((off <= bound).all()), (off / bound).tolist()


# Rows of a group of sixteen are addressed by offsets of 32 bits up to a stride of 2 ** 26 elements (16 rows, in bytes), by pointers past
# it and in groups that reach past the keys that are seen: the same bytes, so the same result to the last bit.
@pytest.mark.parametrize("stride", [2 ** 26 - 8, 2 ** 26], ids=["near", "far"])
@pytest.mark.parametrize("D, V", [(64, 64), (128, 128), (64, 128)])
def test_rows_far_apart(stride, D, V):
    from hydrainfer_amd._C.kernel.biased_attn import biased_attention
    g = torch.Generator().manual_seed(D + V)
    new, nb, H, hs = [40, 30], [3, 2], 4, max(D, V)
    kv = [16 * 3 - 5, 16 * 2]
    r = lambda *s: torch.randn(s, generator=g).bfloat16().cuda()
    i = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    q, k, v = r(sum(new), H, D), r(sum(nb), BLOCK, 1, hs), r(sum(nb), BLOCK, 1, hs)
    table, cu_b, cu_q = torch.randperm(sum(nb), generator=g).int().cuda(), i([0, 3, 5]), i([0, 40, 70])
    pos, seq = i(list(range(kv[0] - 40, kv[0])) + list(range(kv[1] - 30, kv[1]))), i([0] * 40 + [1] * 30)
    call = lambda k, v: biased_attention(q, k, v, V, seq, pos, cu_q, table, cu_b, D ** -0.5, None, "causal", 0, max_q_len=40, max_kv_len=max(kv))
    want = call(k, v)
    room = torch.empty(sum(nb) * BLOCK * stride, dtype=torch.bfloat16, device="cuda")      # (10 GB, of which the rows are touched)
    apart = [room[n * hs:].as_strided(x.shape, (BLOCK * stride, stride, hs, 1)).copy_(x) for n, x in enumerate((k, v))]
    assert torch.equal(call(*apart), want)
