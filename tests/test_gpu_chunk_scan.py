"""Portions of prompts through the recurrences with a matrix state (csrc/chunk_scan.hip) against a token at a time in 64 bits:
portions around the sixteen tokens of a chunk, single tokens beside them, keys and values that fill no tile, every operand
type, rows that cannot be read four elements at a time, decays that vanish."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# 2-norm of the error over that of the result: sums of up to 128 + 16 products and products of up to 16 decays, a unit in the last
# place (2^-24) each at worst a few of them in a row
TOL = 32 * 2.0 ** -24


def _scan(form, q, k, v, decay, vscale, beta, bonus, S, cu, fresh):
    """One token at a time; q, k [T, H, K], v [T, H, V], decay [T, H, K], S [n, H, K, V], all double."""
    out = torch.empty_like(v)
    for s in range(len(cu) - 1):
        X = torch.zeros_like(S[s]) if fresh[s] else S[s]
        for t in range(cu[s], cu[s + 1]):
            kv = lambda w: k[t][:, :, None] * w[:, None, :]
            if form == "bonus":
                out[t] = (q[t][:, None, :] @ (X + bonus[:, :, None] * kv(v[t])))[:, 0]
                X = decay[t][:, :, None] * X + kv(v[t])
            else:
                X = decay[t][:, :, None] * X
                w = v[t] * vscale[t][:, None]
                if form == "delta":
                    w = beta[t][:, None] * (v[t] - (k[t][:, None, :] @ X)[:, 0])
                X = X + kv(w)
                out[t] = (q[t][:, None, :] @ X)[:, 0]
        S[s] = X
    return out, S


def _check(name, got, want, tol=TOL):
    off = (got.double().cpu() - want).norm() / want.norm()
    assert float(off) <= tol, (name, float(off))


LENS = [[17], [16, 1, 33], [1, 15, 31, 2], [48, 5]]
# rows are on their way three chunks ahead and pass through three images in LDS: both come round from the fourth chunk on
LONG = [[64, 113], [65, 300]]


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("K, V", [(64, 64), (128, 128), (12, 20), (100, 130), (65, 7)])
@pytest.mark.parametrize("form, per_channel", [("decay", False), ("decay", True), ("delta", False), ("bonus", True)])
@pytest.mark.parametrize("types", ["bf16", "f32", "mixed"])
def test_portions_through_a_scan(lens, K, V, form, per_channel, types):
    _through_a_scan(lens, K, V, form, per_channel, types, 3)


@pytest.mark.parametrize("lens", LONG)
@pytest.mark.parametrize("K, V, types", [(64, 64, "bf16"), (100, 130, "f32"), (128, 128, "mixed")])
@pytest.mark.parametrize("form, per_channel", [("decay", False), ("decay", True), ("delta", False), ("bonus", True)])
def test_long_portions_through_a_scan(lens, K, V, form, per_channel, types):
    _through_a_scan(lens, K, V, form, per_channel, types, 3)


# portions whose chunks are made in a launch ahead (csrc/chunk_chain.hip): tokens that fill no chunk, sequences without tokens, keys and
# values that fill no tile, keys dealt to four waves and (many sequences) to two
@pytest.mark.parametrize("lens", [[1151], [500, 0, 1, 417], [200] * 22], ids=lambda v: f"{len(v)}x{v[0]}")
@pytest.mark.parametrize("form, per_channel, K, V, types", [
    ("bonus", True, 64, 64, "bf16"), ("bonus", True, 128, 128, "f32"), ("bonus", True, 100, 130, "mixed"), ("decay", True, 128, 64, "bf16"), ("decay", True, 65, 7, "f32"),
    ("decay", True, 64, 68, "mixed"), ("delta", False, 128, 128, "mixed"), ("delta", False, 100, 34, "bf16"), ("decay", False, 128, 96, "f32"),
    ("decay", False, 70, 130, "bf16"), ("decay", False, 40, 64, "mixed")])
def test_chunks_made_ahead(lens, form, per_channel, K, V, types, monkeypatch):
    from hydrainfer_amd import _lib
    lib, asked = _lib.mix_lib(), []

    class Watch:
        def __getattr__(self, name):
            if name != "hxm_state_scan_workspace":
                return getattr(lib, name)
            return lambda a: asked.append(lib.hxm_state_scan_workspace(a)) or asked[-1]

    monkeypatch.setattr(_lib, "_mix", Watch())
    _through_a_scan(lens, K, V, form, per_channel, types, 3)
    # by the rule: short portions of few key channels are left to one launch, and of many sequences those that have many chains for their length
    ahead = {1: True, 4: K > 64, 22: (form, per_channel, K, V) in [("bonus", True, 100, 130), ("decay", True, 128, 64), ("decay", True, 65, 7), ("decay", False, 70, 130)]}
    assert (asked[0] > 0) == ahead[len(lens)]


# the same with more than 256 chains of 32 value channels: the keys of 128 channels go to two waves
MANY = [1003, 901, 930]


@pytest.mark.parametrize("form, per_channel", [("bonus", True), ("decay", True), ("decay", False)])
@pytest.mark.parametrize("K, V, types", [(128, 128, "bf16"), (100, 100, "f32"), (128, 126, "mixed")])
def test_many_chunks_made_ahead(form, per_channel, K, V, types):
    H, n, T = 22, len(MANY), sum(MANY)
    assert n * H * ((V + 31) // 32) > 256
    g = torch.Generator(device="cuda").manual_seed(K + V)
    f = lambda *s: torch.randn(s, generator=g, device="cuda")
    qk_t, v_t = (torch.bfloat16 if types == "bf16" else torch.float32), (torch.float32 if types == "f32" else torch.bfloat16)
    unit = lambda: torch.nn.functional.normalize(f(T, H, K), dim=-1).reshape(T, H * K).to(qk_t)
    x = dict(q=unit(), k=unit(), v=f(T, H * V).to(v_t), decay=torch.rand((T, H * K if per_channel else H), generator=g, device="cuda") ** 0.2,
             vscale=torch.rand((T, H), generator=g, device="cuda") if form == "decay" else None, beta=None, bonus=f(H * K) if form == "bonus" else None,
             state=f(n, 1, H * K * V))
    got, want = _on_the_device(form, MANY, H, K, V, x)
    for name, a, b in zip(("out", "state"), got, want):
        _check(name, a, b)


# numbers that are not finite behind a launch ahead: a chunk's last token, one in a chunk's middle, one in another portion; keys of a value channel in
# two waves (64, and many chains of 128) and in four
# (the delta rule only in four; the bonus form has no number a token and head)
@pytest.mark.parametrize("lens, H, K, V, form, per_channel", [
    (lens, H, K, V, form, per_channel) for lens, H, K, V in (([1151], 2, 64, 64), ([500, 0, 1, 417], 2, 128, 128), (MANY, 22, 128, 128))
    for form, per_channel in (("decay", False), ("decay", True), ("delta", False), ("bonus", True)) if form != "delta" or (K == 128 and H == 2)])
@pytest.mark.parametrize("what, value", [("v", float("inf")), ("v", float("nan")), ("k", float("nan")), ("scalar", float("nan"))])
def test_not_finite_numbers_behind_a_launch_ahead(lens, H, K, V, form, per_channel, what, value):
    if form == "bonus" and what == "scalar":
        what = "v"
    T, n = sum(lens), len(lens)
    g = torch.Generator(device="cuda").manual_seed(K + V)
    f, rand = (lambda *s: torch.randn(s, generator=g, device="cuda")), (lambda *s: torch.rand(s, generator=g, device="cuda"))
    unit = lambda: torch.nn.functional.normalize(f(T, H, K), dim=-1).reshape(T, H * K)
    x = dict(q=unit(), k=unit(), v=f(T, H * V), decay=0.5 + 0.5 * rand(T, H * K if per_channel else H), vscale=rand(T, H) if form == "decay" else None,
             beta=rand(T, H) if form == "delta" else None, bonus=f(H * K) if form == "bonus" else None, state=f(n, 1, H * K * V))
    for t in (271, 470, 700):
        if what == "v":
            x["v"][t, V + 3] = value
        elif what == "k":
            x["k"][t, K + 5] = value
        else:
            (x["beta"] if form == "delta" else x["vscale"])[t, 1] = value
    for got, want in zip(*_on_the_device(form, lens, H, K, V, x)):
        fine = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got).cpu(), fine) and not bool(fine.all()) and bool(fine.any())
        _check("finite", got.cpu()[fine], want[fine])


def _on_the_device(form, lens, H, K, V, x):
    """(result, state) of state_scan, which has to go in two launches, and of a token at a time in 64 bits; every other sequence is continued."""
    from hydrainfer_amd import _lib
    from hydrainfer_amd._C.kernel.seq_mix import state_scan
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    lib, n, T, asked = _lib.mix_lib(), len(lens), sum(lens), []

    class Watch:
        def __getattr__(self, name):
            if name != "hxm_state_scan_workspace":
                return getattr(lib, name)
            return lambda a: asked.append(lib.hxm_state_scan_workspace(a)) or asked[-1]

    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    cu = [sum(lens[:s]) for s in range(n + 1)]
    starts = [0 if s % 2 == 0 else 9 for s in range(n)]
    d = lambda t, *s: t.double().reshape(T, H, *s)
    ones = torch.ones((T, H), dtype=torch.float64, device="cuda")
    want, S = _scan(form, d(x["q"], K), d(x["k"], K), d(x["v"], V), d(x["decay"], -1).expand(T, H, K), ones if x["vscale"] is None else x["vscale"].double(),
                    ones if x["beta"] is None else x["beta"].double(), None if x["bonus"] is None else x["bonus"].double().view(H, K),
                    x["state"].double().view(n, H, K, V).clone(), cu, [p == 0 for p in starts])
    st = x["state"].clone()
    seq = SequenceState(st, i32(list(range(n))), i32([s for s in range(n) for _ in range(lens[s])]))
    _lib._mix = Watch()
    try:
        got = state_scan(form, x["q"], x["k"], x["v"], x["decay"], seq, 0, i32(cu), i32([starts[s] + i for s in range(n) for i in range(lens[s])]), H, H, K, V,
                         vscale=x["vscale"], beta=x["beta"], bonus=x["bonus"])
    finally:
        _lib._mix = lib
    assert asked[0] > 0
    return (got, st.view(n, H, K, V)), (want.reshape(T, H * V).cpu(), S.cpu())


# few chains of long portions: segments of six chunks (96 tokens), whose states a launch ahead makes.  Whole segments, a token more and one less,
# portions of one segment, of one token and of none beside them, a state of an odd number of floats, more columns than a workgroup takes
SEGMENTS = [[288], [289], [383], [700, 0, 96, 480, 1, 97, 1000]]


@pytest.mark.parametrize("lens", SEGMENTS, ids=lambda v: f"{len(v)}x{v[0]}")
@pytest.mark.parametrize("K, V", [(64, 64), (128, 128), (65, 7), (20, 70)])
@pytest.mark.parametrize("form, per_channel, types", [("decay", False, "f32"), ("decay", True, "bf16"), ("bonus", True, "mixed")])
def test_portions_in_segments(lens, K, V, form, per_channel, types, monkeypatch):
    from hydrainfer_amd import _lib
    lib, H, n, T, asked = _lib.mix_lib(), 2, len(lens), sum(lens), []

    class Watch:
        def __getattr__(self, name):
            if name != "hxm_state_scan_workspace":
                return getattr(lib, name)
            return lambda a: asked.append(lib.hxm_state_scan_workspace(a)) or asked[-1]

    monkeypatch.setattr(_lib, "_mix", Watch())
    g = torch.Generator(device="cuda").manual_seed(K + V)
    f, rand = (lambda *s: torch.randn(s, generator=g, device="cuda")), (lambda *s: torch.rand(s, generator=g, device="cuda"))
    qk_t, v_t = (torch.bfloat16 if types == "bf16" else torch.float32), (torch.float32 if types == "f32" else torch.bfloat16)
    unit = lambda: torch.nn.functional.normalize(f(T, H, K), dim=-1).reshape(T, H * K).to(qk_t)
    decay = rand(T, H * K if per_channel else H) ** 0.2
    decay[150:160, 0] = 0.0                                # (nothing is left behind these; what stands there has to vanish, not to turn into NaN)
    x = dict(q=unit(), k=unit(), v=f(T, H * V).to(v_t), decay=decay, vscale=rand(T, H) if form == "decay" else None, beta=None,
             bonus=f(H * K) if form == "bonus" else None, state=f(n, 1, H * K * V))
    got, want = _on_the_device(form, lens, H, K, V, x)
    rest = asked[0] - H * (T // 96 + n) * ((K * V + 1) // 2 * 2 + 2 * K)      # floats of the segments, and those of the chunks
    assert rest > 0 and rest % (H * (T // 16 + n)) == 0
    for name, a, b in zip(("out", "state"), got, want):
        _check(name, a, b)


@pytest.mark.parametrize("lens", SEGMENTS[1:], ids=lambda v: f"{len(v)}x{v[0]}")
@pytest.mark.parametrize("K, V, dtype", [(64, 64, torch.bfloat16), (100, 130, torch.float32), (65, 7, torch.float32)])
def test_gated_portions_in_segments(lens, K, V, dtype):
    _through_the_gated_recurrence(lens, K, V, dtype)


@pytest.mark.parametrize("lens, H", [([1151], 3), ([0, 300, 0, 1, 417, 0], 3), (MANY, 22)], ids=str)
@pytest.mark.parametrize("K, V", [(64, 64), (128, 128), (100, 36), (48, 7)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_gates_made_ahead(lens, H, K, V, dt, monkeypatch):
    from hydrainfer_amd import _lib
    from hydrainfer_amd._C.kernel.recurrence import gated_recurrence
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    lib, T, n = _lib.mix_lib(), sum(lens), len(lens)
    g = torch.Generator(device="cuda").manual_seed(K + V)
    f = lambda *s: torch.randn(s, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    proj, bias, low, w, start = f(T, H * (2 * K + V)).to(dt), f(H * K), 0.9 * torch.rand(H * K, generator=g, device="cuda"), f(V), f(n, 1, H * K * V)
    proj[T // 2, 2 * H * K + 1] = math.inf                        # (a chunk whose sums go in order)
    cu = [sum(lens[:s]) for s in range(n + 1)]
    pos = i32([p + 5 * (s % 2) for s, m in enumerate(lens) for p in range(m)])
    seq_of = i32([s for s, m in enumerate(lens) for _ in range(m)])

    def run():
        st = start.clone()
        return gated_recurrence(proj[:, :H * K], proj[:, H * K:2 * H * K], proj[:, 2 * H * K:], bias, low, w, 1e-5, SequenceState(st, i32(list(range(n))), seq_of), 0,
                                i32(cu), pos, H, K, V, max_q_len=max(lens)), st

    ahead = run()
    assert lib.hxm_gated_recurrence_batch_workspace(n, T, H, K, V, max(lens), _lib._DTYPE[dt]) > lib.hxm_gated_recurrence_workspace(T, H, K, V)

    class Least:
        def __getattr__(self, name):
            return (lambda n, T, H, K, V, m, dt: lib.hxm_gated_recurrence_workspace(T, H, K, V)) if name == "hxm_gated_recurrence_batch_workspace" else getattr(lib, name)

    monkeypatch.setattr(_lib, "_mix", Least())
    for a, b in zip(ahead, run()):
        fine = torch.isfinite(a)
        assert torch.equal(fine, torch.isfinite(b)) and bool(fine.any())
        off = (a[fine].double() - b[fine].double()).norm() / b[fine].double().norm()
        assert float(off) <= (2.0 ** -8 if a.dtype == torch.bfloat16 else 2 * TOL)      # (a unit of a result in bfloat16; TOL for either form)


# out, state: what a token at a time loses in float over the same portions (2-norm, in 1e-7, measured with the form that walks the
# tokens).  Chunks lose no more than that, give or take a twentieth.
@pytest.mark.parametrize("form, K, out, state", [("delta", 128, 1.096, 0.780), ("delta", 64, 1.010, 0.838), ("decay", 128, 1.073, 0.825), ("decay", 64, 1.001, 0.808),
                                                 ("bonus", 128, 0.908, 0.464), ("bonus", 64, 0.832, 0.464)])
def test_chunks_round_no_more_than_single_tokens(form, K, out, state):
    from hydrainfer_amd._C.kernel.seq_mix import state_scan
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    g = torch.Generator().manual_seed(K)
    lens, H, per_channel, bounds = [400, 250], 4, form == "bonus", (1.05e-7 * out, 1.05e-7 * state)
    T, cu = sum(lens), [0, 400, 650]
    f = lambda *s: torch.randn(s, generator=g)
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1).reshape(T, H * K)
    if form == "delta":
        q, k = unit(f(T, H, K)) * K ** -0.5, unit(f(T, H, K))
    else:
        q, k = ((f(T, H * K) * K ** -0.5).bfloat16() for _ in range(2))
    v, step = f(T, H * K).bfloat16(), torch.nn.functional.softplus(f(T, H) - 2)
    decay = torch.exp(-torch.exp(f(T, H * K) - 2)) if per_channel else torch.exp(-torch.exp(0.3 * f(H)) * step)
    beta, bonus, state = torch.sigmoid(f(T, H)), f(H * K), 0.1 * f(2, 1, H * K * K)
    h = lambda x: x.double().view(T, H, K)
    want, S = _scan(form, h(q), h(k), h(v), decay.double().view(T, H, -1).expand(T, H, K), step.double() if form == "decay" else torch.ones((T, H), dtype=torch.float64),
                    beta.double(), bonus.double().view(H, K), state.double().view(2, H, K, K), cu, [False, False])
    c = lambda x: x.cuda()
    st = c(state)
    seq = SequenceState(st, torch.arange(2, dtype=torch.int32, device="cuda"), c(torch.tensor([0] * 400 + [1] * 250, dtype=torch.int32)))
    got = state_scan(form, c(q), c(k), c(v), c(decay), seq, 0, c(torch.tensor(cu, dtype=torch.int32)), c(torch.arange(1, T + 1, dtype=torch.int32)), H, H, K, K,
                     vscale=c(step) if form == "decay" else None, beta=c(beta) if form == "delta" else None, bonus=c(bonus) if form == "bonus" else None)
    _check("out", got, want.reshape(T, H * K), bounds[0])
    _check("state", st.view(2, H, K, K), S, bounds[1])


# batches of as many tokens as sequences (csrc/state_scan.hip, the step form): columns and rows that fill no workgroup, a sequence that
# brings two tokens and one that brings none, slots that start on a multiple of four floats and (the form with a column a lane) not
@pytest.mark.parametrize("lens", [[1], [1, 1, 1, 1, 1], [2, 0, 1]])
@pytest.mark.parametrize("K, V", [(64, 64), (128, 128), (12, 20), (100, 132), (65, 8), (256, 68), (3, 4)])
@pytest.mark.parametrize("form, per_channel", [("decay", False), ("decay", True), ("delta", False), ("bonus", True)])
@pytest.mark.parametrize("types, pad", [("bf16", 4), ("f32", 4), ("mixed", 4), ("mixed", 3)])
def test_single_tokens_through_a_scan(lens, K, V, form, per_channel, types, pad):
    _through_a_scan(lens, K, V, form, per_channel, types, pad)


# portions that may go either way: on both sides of the six tokens a sequence and of the thirteen that the longest may have
@pytest.mark.parametrize("lens", [[12], [13], [5, 6], [6, 6], [1, 13], [7, 1, 10]])
@pytest.mark.parametrize("form, per_channel", [("decay", False), ("decay", True), ("delta", False), ("bonus", True)])
def test_portions_at_the_rule_between_the_forms(lens, form, per_channel):
    _through_a_scan(lens, 40, 20, form, per_channel, "f32", 4)


# portions that go a token at a time: short ones, and the forms and types that have no chunks; with few workgroups (more lanes a column)
# and with many
@pytest.mark.parametrize("lens", [[5], [3, 1, 2], [17, 33], [2] * 40], ids=lambda v: f"{len(v)}x{v[0]}")
@pytest.mark.parametrize("K, V", [(64, 64), (128, 130), (40, 20), (100, 7)])
@pytest.mark.parametrize("form, per_channel, types", [("delta", True, "mixed"), ("bonus", False, "f32"), ("decay", False, "odd"), ("delta", False, "odd")])
def test_portions_a_token_at_a_time(lens, K, V, form, per_channel, types):
    _through_a_scan(lens, K, V, form, per_channel, types, 3)


def _through_a_scan(lens, K, V, form, per_channel, types, pad):
    from hydrainfer_amd._C.kernel.seq_mix import state_scan
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    g = torch.Generator().manual_seed(sum(lens) * 1000 + K + V)
    n, T, H = len(lens), sum(lens), 4
    G = H if form == "bonus" else 2
    qk_t, v_t = (torch.bfloat16 if types in ("bf16", "odd") else torch.float32), (torch.float32 if types in ("f32", "odd") else torch.bfloat16)
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1)
    proj = torch.cat([unit(torch.randn((T, G, K), generator=g)).reshape(T, G * K), unit(torch.randn((T, G, K), generator=g)).reshape(T, G * K),
                      torch.zeros((T, 1))], dim=1).to(qk_t)       # (an odd row length: views that do not start on multiples of four)
    q, k = proj[:, :G * K], proj[:, G * K:2 * G * K]
    v = torch.randn((T, H * V), generator=g).to(v_t)
    decay = torch.rand((T, H * K if per_channel else H), generator=g) ** 0.2
    decay[T // 3] = 0.0                                            # forgets everything, and nothing divides by it
    decay[T // 2, 0] = 1e-30
    vscale, beta, bonus = torch.rand((T, H), generator=g), torch.rand((T, H), generator=g), torch.randn(H * K, generator=g)
    state = torch.randn((n + 1, 1, H * K * V + pad), generator=g)
    slots = torch.randperm(n + 1, generator=g)[:n].int()
    cu = [0]
    for x in lens:
        cu.append(cu[-1] + x)
    starts = [0 if s % 2 == 0 else 40 + s for s in range(n)]
    pos = torch.tensor([starts[s] + i for s in range(n) for i in range(lens[s])], dtype=torch.int32)
    tok_seq = torch.tensor([s for s in range(n) for _ in range(lens[s])], dtype=torch.int32)
    heads = lambda x: x.double().view(T, G, K).repeat_interleave(H // G, dim=1)
    want, S = _scan(form, heads(q), heads(k), v.double().view(T, H, V), (decay.double().view(T, H, -1)).expand(T, H, K),
                    vscale.double() if form == "decay" else torch.ones((T, H), dtype=torch.float64), beta.double(), bonus.double().view(H, K),
                    state[slots.long(), 0, pad:].double().view(n, H, K, V), cu, [p == 0 for p in starts])
    d = lambda x: x.cuda()
    st = d(state)
    before = st.clone()
    seq = SequenceState(st, d(slots), d(tok_seq))
    pd = d(proj)
    got = state_scan(form, pd[:, :G * K], pd[:, G * K:2 * G * K], d(v), d(decay), seq, pad, d(torch.tensor(cu, dtype=torch.int32)), d(pos), H, G, K, V,
                     vscale=d(vscale) if form == "decay" else None, beta=d(beta) if form == "delta" else None, bonus=d(bonus) if form == "bonus" else None)
    _check("out", got, want.reshape(T, H * V))
    _check("state", st[slots.long().cuda(), 0, pad:].view(n, H, K, V), S)
    other = [s for s in range(n + 1) if s not in slots.tolist()]
    assert torch.equal(st[other], before[other]) and torch.equal(st[:, 0, :pad], before[:, 0, :pad])


# What is not a finite number in a token's operands shows from that token on, in its columns, and nowhere before: the tokens are a chunk's
# last, one in its middle and one behind it.
@pytest.mark.parametrize("K, V", [(64, 64), (128, 128), (12, 20)])
@pytest.mark.parametrize("form, per_channel", [("decay", False), ("decay", True), ("delta", False), ("bonus", True)])
@pytest.mark.parametrize("what, value", [("v", float("inf")), ("v", float("nan")), ("k", float("nan")), ("scalar", float("nan"))])
def test_not_finite_numbers_reach_later_tokens_only(K, V, form, per_channel, what, value):
    from hydrainfer_amd._C.kernel.seq_mix import state_scan
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    g = torch.Generator().manual_seed(K + V)
    lens, bad, H = [40, 16, 23], [25, 55, 58], 2
    n, T = len(lens), sum(lens)
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1).reshape(T, H * K)
    q, k, v = unit(torch.randn((T, H, K), generator=g)), unit(torch.randn((T, H, K), generator=g)), torch.randn((T, H * V), generator=g)
    decay = 0.5 + 0.5 * torch.rand((T, H * K if per_channel else H), generator=g)
    vscale, beta, bonus = torch.rand((T, H), generator=g), torch.rand((T, H), generator=g), torch.randn(H * K, generator=g)
    for t in bad:
        if what == "v":
            v[t, V + 3] = value
        elif what == "k":
            k[t, K + 5] = value
        else:
            vscale[t, 1] = beta[t, 1] = value
    cu = [0, 40, 56, 79]
    state = torch.randn((n, 1, H * K * V), generator=g)
    h = lambda x, m: x.double().view(T, H, m)
    want, S = _scan(form, h(q, K), h(k, K), h(v, V), decay.double().view(T, H, -1).expand(T, H, K),
                    vscale.double() if form == "decay" else torch.ones((T, H), dtype=torch.float64), beta.double(), bonus.double().view(H, K),
                    state.double().view(n, H, K, V), cu, [True, False, False])
    d = lambda x: x.cuda()
    pos = torch.tensor([(0 if s == 0 else 9) + i for s in range(n) for i in range(lens[s])], dtype=torch.int32)
    st = d(state)
    seq = SequenceState(st, torch.arange(n, dtype=torch.int32, device="cuda"), d(torch.tensor([s for s in range(n) for _ in range(lens[s])], dtype=torch.int32)))
    got = state_scan(form, d(q), d(k), d(v), d(decay), seq, 0, d(torch.tensor(cu, dtype=torch.int32)), d(pos), H, H, K, V,
                     vscale=d(vscale) if form == "decay" else None, beta=d(beta) if form == "delta" else None, bonus=d(bonus) if form == "bonus" else None)
    for got, want in ((got.double().cpu(), want.reshape(T, H * V)), (st.double().cpu().view(n, H, K, V), S)):
        fine = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), fine)
        _check("finite", got[fine], want[fine])


# Infinities stay infinities of their sign where the arithmetic has one answer: values of a portion's last token (its state is then k times them), keys of
# it, and what the state held before (a decayed sum's stays).  Under the delta rule the last token is a chunk's last: rows past a portion read it.
@pytest.mark.parametrize("form, K, V, types", [("decay", 128, 64, "bf16"), ("decay", 64, 34, "bf16"), ("decay", 128, 128, "f32"), ("decay", 64, 64, "mixed"),
                                               ("delta", 128, 64, "bf16"), ("delta", 100, 130, "f32"), ("delta", 128, 128, "mixed"), ("delta", 64, 64, "mixed")])
@pytest.mark.parametrize("what", ["v", "k", "state"])
def test_infinities_stay_infinities(form, K, V, types, what):
    if form == "delta" and what != "v":
        pytest.skip("the portion's tokens read what is infinite, in sums of both signs")
    from hydrainfer_amd._C.kernel.seq_mix import state_scan
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    g = torch.Generator().manual_seed(K + V)
    lens, H, inf = [60, 17, 55, 96] if form == "decay" else [64, 32, 32, 96], 2, float("inf")
    n, T, cu = len(lens), sum(lens), [sum(lens[:s]) for s in range(len(lens) + 1)]
    qk_t, v_t = (torch.bfloat16 if types == "bf16" else torch.float32), (torch.float32 if types == "f32" else torch.bfloat16)
    unit = lambda: torch.nn.functional.normalize(torch.randn((T, H, K), generator=g), dim=-1).reshape(T, H * K).to(qk_t)
    q, k, v = unit(), unit(), torch.randn((T, H * V), generator=g).to(v_t)
    decay, beta, state = 0.5 + 0.5 * torch.rand((T, H), generator=g), torch.rand((T, H), generator=g), torch.randn((n, 1, H * K * V), generator=g)
    for s in range(n):
        last = cu[s + 1] - 1
        if what == "v":
            v[last, V + 3], v[last, 7] = inf, -inf
        elif what == "k":
            k[last, 5], k[last, K + 9] = inf, -inf
        else:
            state.view(n, H, K, V)[s, 1, 5, 3], state.view(n, H, K, V)[s, 0, 9, 7] = inf, -inf
    h = lambda x, m: x.double().view(T, H, m)
    want, S = _scan(form, h(q, K), h(k, K), h(v, V), decay.double().view(T, H, 1).expand(T, H, K), torch.ones((T, H), dtype=torch.float64), beta.double(), None,
                    state.double().view(n, H, K, V), cu, [False] * n)
    d = lambda x: x.cuda()
    st = d(state)
    seq = SequenceState(st, torch.arange(n, dtype=torch.int32, device="cuda"), d(torch.tensor([s for s in range(n) for _ in range(lens[s])], dtype=torch.int32)))
    got = state_scan(form, d(q), d(k), d(v), d(decay), seq, 0, d(torch.tensor(cu, dtype=torch.int32)), d(torch.tensor([9 + i for m in lens for i in range(m)], dtype=torch.int32)),
                     H, H, K, V, beta=d(beta) if form == "delta" else None)
    for name, got, want in (("out", got.double().cpu(), want.reshape(T, H * V)), ("state", st.double().cpu().view(n, H, K, V), S)):
        fine = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), fine)
        if name == "state":                   # (results are sums over infinities of both signs)
            assert bool(torch.isinf(want).any()) and not bool(torch.isnan(want).any())
            assert torch.equal(got[~fine], want[~fine])
        _check("finite", got[fine], want[fine])


@pytest.mark.parametrize("what", ["v", "k"])
def test_not_finite_numbers_in_the_gated_recurrence(what):
    from hydrainfer_amd._C.kernel.recurrence import gated_recurrence
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    g = torch.Generator().manual_seed(5)
    T, H, K, V, bad = 37, 2, 128, 64, 30
    proj = torch.randn((T, H * (2 * K + V)), generator=g)
    f_bias, low, norm_w = torch.randn(H * K, generator=g), torch.rand(H * K, generator=g), 1 + 0.1 * torch.randn(V, generator=g)

    def run(p):
        seq = SequenceState(torch.zeros((1, 1, H * K * V), device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda"), torch.zeros(T, dtype=torch.int32, device="cuda"))
        p = p.cuda()
        return gated_recurrence(p[:, :H * K], p[:, H * K:2 * H * K], p[:, 2 * H * K:], f_bias.cuda(), low.cuda(), norm_w.cuda(), 1e-5, seq, 0,
                                torch.tensor([0, T], dtype=torch.int32).cuda(), torch.arange(T, dtype=torch.int32).cuda(), H, K, V, max_q_len=T).cpu()
    clean = run(proj)
    proj[bad, H * K + K + 7 if what == "k" else 2 * H * K + V + 3] = float("nan")
    got = run(proj)
    assert torch.isfinite(got[:bad]).all() and torch.equal(got[:, :V], clean[:, :V]) and torch.isnan(got[bad:, V:]).all()
    _check("before", got[:bad], clean[:bad].double(), 2 * TOL)


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("K, V", [(64, 64), (128, 128), (12, 20), (100, 130), (65, 7)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_portions_through_the_gated_recurrence(lens, K, V, dtype):
    _through_the_gated_recurrence(lens, K, V, dtype)


@pytest.mark.parametrize("lens", LONG)
@pytest.mark.parametrize("K, V, dtype", [(64, 64, torch.bfloat16), (100, 130, torch.float32)])
def test_long_portions_through_the_gated_recurrence(lens, K, V, dtype):
    _through_the_gated_recurrence(lens, K, V, dtype)


# the longest portion at which chunks begin: 8 and 16 tokens (24 and 64 where small states fill the chip, 2 where large ones do)
@pytest.mark.parametrize("lens, K, V", [([7, 2], 64, 64), ([8, 2], 64, 64), ([15, 2], 128, 64), ([16, 2], 128, 64), ([23] + [2] * 180, 20, 12), ([24] + [2] * 180, 20, 12),
                                        ([63] + [2] * 180, 16, 16), ([64] + [2] * 180, 16, 16), ([2] * 100, 65, 12)], ids=lambda v: f"{len(v)}x{v[0]}" if isinstance(v, list) else v)
def test_portions_at_the_rule_of_the_gated_recurrence(lens, K, V):
    _through_the_gated_recurrence(lens, K, V, torch.float32)


def _through_the_gated_recurrence(lens, K, V, dtype):
    from hydrainfer_amd._C.kernel.recurrence import gated_recurrence
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    g = torch.Generator().manual_seed(sum(lens) * 1000 + K + V)
    n, T, H, eps = len(lens), sum(lens), 3, 1e-5
    proj = (2 * torch.randn((T, H * (2 * K + V) + 1), generator=g)).to(dtype)
    proj[0, :4] = torch.tensor([300.0, -300.0, 90.0, -90.0])      # where a plain exponential leaves the range of a float
    proj[1 % T, H * K:H * K + 4] = torch.tensor([300.0, -300.0, 90.0, -90.0])
    f_bias, low, norm_w = torch.randn(H * K, generator=g), torch.rand(H * K, generator=g) ** 2, 1 + 0.1 * torch.randn(V, generator=g)
    low[0] = 0.0
    state = torch.randn((n, 2, H * K * V), generator=g)
    cu = [0]
    for x in lens:
        cu.append(cu[-1] + x)
    starts = [0 if s % 2 == 0 else 40 + s for s in range(n)]
    pos = torch.tensor([starts[s] + i for s in range(n) for i in range(lens[s])], dtype=torch.int32)
    tok_seq = torch.tensor([s for s in range(n) for _ in range(lens[s])], dtype=torch.int32)
    x = proj.double()
    f = low.double() + (1 - low.double()) * torch.sigmoid(x[:, H * K:2 * H * K] + f_bias.double())
    q = torch.nn.functional.silu(x[:, :H * K])
    ones = torch.ones((T, H), dtype=torch.float64)
    o, S = _scan("decay", q.view(T, H, K), (1 - f).view(T, H, K), x[:, 2 * H * K:-1].reshape(T, H, V), f.view(T, H, K), ones, ones, None,
                 state[:, 1].double().view(n, H, K, V), cu, [p == 0 for p in starts])
    want = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * norm_w.double()
    st, pd = state.cuda(), proj.cuda()
    seq = SequenceState(st, torch.arange(n, dtype=torch.int32, device="cuda"), tok_seq.cuda())
    got = gated_recurrence(pd[:, :H * K], pd[:, H * K:2 * H * K], pd[:, 2 * H * K:-1], f_bias.cuda(), low.cuda(), norm_w.cuda(), eps, seq, 1,
                           torch.tensor(cu, dtype=torch.int32).cuda(), pos.cuda(), H, K, V, max_q_len=max(lens))
    # (1 - f) is taken from a float f: an absolute 2^-24, the larger part of a small gate
    _check("state", st[:, 1].view(n, H, K, V), S, 2 * TOL)
    _check("out", got, want.reshape(T, H * V), 2 * TOL if dtype == torch.float32 else 2.0 ** -8)
    assert torch.equal(st[:, 0].cpu(), state[:, 0])


@pytest.mark.parametrize("max_q_len", [0, 2])      # (in chunks, and a token at a time)
def test_small_gates_are_as_exact_as_large_ones(max_q_len):
    # without values a state is the product of its gates; two of them, each off by a few units in the last place (2^-23) of its exponential,
    # sum and reciprocal
    from hydrainfer_amd._C.kernel.recurrence import gated_recurrence
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    H, K, V, T = 4, 128, 64, 2
    proj = torch.zeros((T, H * (2 * K + V)))
    proj[:, H * K:2 * H * K] = torch.linspace(-40.0, 100.0, T * H * K).view(T, H * K).flip(1)
    proj[0, H * K], proj[1, H * K], proj[0, H * K + 1], proj[1, H * K + 1] = -80.0, 300.0, math.inf, math.inf
    st = torch.ones((1, 1, H * K * V), device="cuda")
    seq = SequenceState(st, torch.zeros(1, dtype=torch.int32, device="cuda"), torch.zeros(T, dtype=torch.int32, device="cuda"))
    zero, p = torch.zeros(H * K, device="cuda"), proj.cuda()
    gated_recurrence(p[:, :H * K], p[:, H * K:2 * H * K], p[:, 2 * H * K:], zero, zero, torch.ones(V, device="cuda"), 1e-5, seq, 0,
                     torch.tensor([0, T], dtype=torch.int32).cuda(), torch.tensor([5, 6], dtype=torch.int32).cuda(), H, K, V, max_q_len=max_q_len)
    want = torch.sigmoid(proj[:, H * K:2 * H * K].double()).prod(0).view(H, K, 1)
    off = (st.double().cpu().view(H, K, V) - want).abs() / want
    assert float(off.max()) <= 8 * 2.0 ** -23, float(off.max())


# One decay a head in one launch (csrc/chunk_head.hip): portions at the edges of its chunks of 32 tokens and their tiles of 16, channels that fill no
# tile and no vector, q and k in one part (float ones: the test below; here they go sixteen tokens at a time)
@pytest.mark.parametrize("lens", [[13, 16, 17, 31, 32, 0, 33, 48, 49, 64, 65, 97] * 2, [47, 1, 15, 96]], ids=["edges", "few"])
@pytest.mark.parametrize("form, K, V", [("delta", 128, 128), ("delta", 100, 34), ("delta", 65, 68), ("decay", 128, 64), ("decay", 64, 130), ("decay", 100, 7), ("decay", 17, 64)])
@pytest.mark.parametrize("types, pad", [("bf16", 4), ("f32", 4), ("mixed", 3)])
def test_chunks_of_two_tiles(lens, form, K, V, types, pad):
    _through_a_scan(lens, K, V, form, False, types, pad)


# The same of float q and k under the delta rule, which take chunks of 32 where portions fill them in the mean (17 - 32 tokens, 49 - 64, and more than 80)
@pytest.mark.parametrize("lens", [[13, 16, 17, 31, 32, 33, 48, 5], [49, 64, 65, 97, 33, 48, 1], [81, 96, 97]], ids=["short", "two", "three"])
@pytest.mark.parametrize("K, V", [(128, 128), (100, 34), (65, 68)])
@pytest.mark.parametrize("types, pad", [("f32", 4), ("mixed", 3)])
def test_chunks_of_two_tiles_in_three_parts(lens, K, V, types, pad):
    mean = sum(lens) / len(lens)
    assert 1.7 * -(-mean // 32) < -(-mean // 16)
    _through_a_scan(lens, K, V, "delta", False, types, pad)


# rows so far apart that chunks of thirty-two tokens do not address them: in chunks of sixteen all the same
@pytest.mark.parametrize("form", ["decay", "delta"])
def test_rows_far_apart(form):
    from hydrainfer_amd._C.kernel.seq_mix import state_scan
    from hydrainfer_amd._C.kernel.stream_ops import SequenceState
    T, H, K, V, stride = 17, 2, 128, 64, 2 ** 28
    g = torch.Generator(device="cuda").manual_seed(5)
    f = lambda *s: torch.randn(s, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    unit = lambda: torch.nn.functional.normalize(f(T, H, K), dim=-1).reshape(T, H * K).bfloat16()
    near, state, decay, beta = (unit(), unit(), f(T, H * V).bfloat16()), f(1, 1, H * K * V), torch.rand((T, H), generator=g, device="cuda"), torch.rand((T, H), generator=g, device="cuda")
    room = torch.empty((T - 1) * stride + 2048, dtype=torch.bfloat16, device="cuda")      # (9 GB, of which the rows are touched)
    far = [room[512 * n:].as_strided(x.shape, (stride, 1)).copy_(x) for n, x in enumerate(near)]
    got = []
    for q, k, v in (near, far):
        st = state.clone()
        seq = SequenceState(st, i32([0]), i32([0] * T))
        got.append((state_scan(form, q, k, v, decay, seq, 0, i32([0, T]), i32(list(range(9, 9 + T))), H, H, K, V, beta=beta if form == "delta" else None).double(), st.double()))
    # thirty-two tokens in parts and sixteen in float: either is within 2e-7 of 64 bits (2-norm)
    for a, b in zip(*got):
        assert float((a - b).norm() / a.norm()) < 1e-6
