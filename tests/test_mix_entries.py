"""What the entries of libhydra_mix.so refuse on the host, before anything is launched."""
import ctypes

import pytest


@pytest.mark.parametrize("n_tokens", [1, 2, 5, 100])
@pytest.mark.parametrize("mode", [3, -1])
def test_state_scan_refuses_an_unknown_recurrence(mode, n_tokens):
    from hydrainfer_amd import _lib
    buf = ctypes.create_string_buffer(1 << 16)
    at = ctypes.addressof(buf)
    a = _lib.hxm_state_scan_args(out=at, q=at, k=at, v=at, q_stride=64, k_stride=64, v_stride=64, decay=at, state=at, slot_stride=4096, slots=at, q_cu=at,
                                 positions=at, n_tokens=n_tokens, n_seq=1, heads=1, qk_heads=1, dim=64, vdim=64, mode=mode)
    HX_ERR_UNSUPPORTED = -5
    assert _lib.mix_lib().hxm_state_scan(ctypes.byref(a), None) == HX_ERR_UNSUPPORTED


@pytest.mark.parametrize("rows, experts, n, k, tile", [
    (1, 8, 2816, 2048, 32), (256, 8, 2816, 2048, 32), (768, 8, 2816, 2048, 128), (7976, 16, 4096, 2752, 256), (15956, 16, 5504, 4096, 256),
    # the measured best by more than a tenth (us in tiles of 64 / 128 / 256): 61 76 35, 86 104 54, 74 86 51, 48 60 33; 36 28 48; 35 28 48, 36 28 48
    (64 * 140, 64, 1024, 704, 256), (64 * 140, 64, 1024, 1408, 256), (32 * 140, 32, 2048, 1408, 256), (32 * 140, 32, 2048, 704, 256), (8 * 110, 8, 2816, 2048, 128),
    (16 * 80, 16, 1408, 2048, 128), (16 * 110, 16, 1408, 2048, 128),
    # 22 26 47, 43 55 57, 16 20 32
    (8 * 50, 8, 2816, 2048, 64), (16 * 50, 16, 2816, 2048, 64), (8 * 57, 8, 2048, 1408, 64)])
def test_tiles_of_the_grouped_product(rows, experts, n, k, tile):
    from hydrainfer_amd import _lib
    assert _lib.mix_lib().hxm_grouped_linear_tile_rows(rows, experts, n, k) == tile


@pytest.mark.parametrize("n_seq, tokens, heads, dim, vdim, ahead", [
    (1, 1151, 32, 128, 128, True), (4, 4000, 8, 128, 128, True), (4, 4000, 16, 128, 128, True), (4, 4000, 17, 128, 128, False), (4, 4000, 32, 128, 128, False),
    (64, 64000, 32, 128, 128, False), (4, 4000, 8, 65, 32, True), (4, 4000, 8, 64, 128, False), (1, 4000, 1, 64, 64, False), (1, 60, 8, 128, 128, False)])
def test_delta_rule_in_two_launches(n_seq, tokens, heads, dim, vdim, ahead):
    """Only where the keys of a value channel are dealt to four waves: there is no other form for the delta rule behind a launch ahead."""
    from hydrainfer_amd import _lib
    HX_F32 = 0
    a = _lib.hxm_state_scan_args(q_dtype=HX_F32, k_dtype=HX_F32, v_dtype=HX_F32, n_tokens=tokens, n_seq=n_seq, heads=heads, qk_heads=heads, dim=dim, vdim=vdim,
                                 mode=2)
    assert (_lib.mix_lib().hxm_state_scan_workspace(ctypes.byref(a)) > 0) == ahead
    assert not ahead or (dim > 64 and n_seq * heads * ((vdim + 31) // 32) <= 256)


def test_no_call_with_a_launch_ahead_is_taken_for_a_short_one():
    """long_chains, which spares short calls the question, holds wherever the library would have asked for a workspace; and calls of short portions
    and steps are spared it."""
    import random
    from hydrainfer_amd import _lib
    from hydrainfer_amd._C.kernel.stream_ops import long_chains
    lib, rng, HX_F32, asked = _lib.mix_lib(), random.Random(5), 0, 0
    for _ in range(20000):
        n_seq, heads, dim, vdim = rng.choice([1, 2, 3, 4, 7, 16, 40, 100]), rng.randint(1, 64), rng.choice([16, 64, 65, 128]), rng.choice([7, 64, 65, 128, 200])
        longest = int(2 ** rng.uniform(0, 11))
        tokens = rng.randint(longest, longest * n_seq)
        for mode, per_channel in ((0, 0), (0, 1), (1, 1), (2, 0)):
            a = _lib.hxm_state_scan_args(q_dtype=HX_F32, k_dtype=HX_F32, v_dtype=HX_F32, n_tokens=tokens, n_seq=n_seq, heads=heads, qk_heads=heads, dim=dim, vdim=vdim,
                                         mode=mode, decay_per_channel=per_channel)
            if tokens > n_seq and lib.hxm_state_scan_workspace(ctypes.byref(a)) > 0:
                assert long_chains(tokens, n_seq, heads, vdim)
                asked += 1
        for known in (0, longest):
            if lib.hxm_gated_recurrence_batch_workspace(n_seq, tokens, heads, dim, vdim, known, HX_F32) > lib.hxm_gated_recurrence_workspace(tokens, heads, dim, vdim):
                assert long_chains(tokens, n_seq, heads, vdim, known)
                asked += 1
    assert asked > 1000
    assert not long_chains(3, 3, 16, 64, 1) and not long_chains(300, 4, 32, 128) and not long_chains(100, 1, 64, 128, 100) and not long_chains(0, 0, 8, 64)


def _latent_splits(lens, kv, heads, rank, window=0):
    from hydrainfer_amd import _lib
    HX_BF16 = _lib._DTYPE[__import__("torch").bfloat16]
    a = _lib.hxm_latent_attn_args(q_token_stride=heads * rank, q_head_stride=rank, out_token_stride=heads * rank, out_head_stride=rank, cache_block_stride=16 * rank,
                                  cache_row_stride=rank, n_tokens=sum(lens), n_seq=len(lens), n_heads=heads, kv_rank=rank, block_size=16, window=window,
                                  max_q_len=max(lens), scale=1.0, dtype=HX_BF16, max_kv_len=kv)
    n, floats = ctypes.c_int32(), ctypes.c_int64()
    assert _lib.mix_lib().hxm_latent_attention_plan(ctypes.byref(a), ctypes.byref(n), ctypes.byref(floats)) == 0
    assert floats.value == (0 if n.value == 1 else len(lens) * ((max(lens) * heads + 15) // 16) * n.value * 16 * (rank + 2))
    return n.value


@pytest.mark.parametrize("lens, kv, heads, rank, splits", [
    # two groups of waves in the place of two splits, and of three where the keys that a row sees are few: no workspace
    ([302], 302, 16, 320, 1), ([922], 922, 16, 128, 1), ([948], 948, 8, 320, 1), ([100, 64], 500, 16, 256, 1), ([5] * 8, 250, 32, 64, 1),
    # three splits of more keys or wider rows (us in three and by two groups, the second and third: 46.6 58, 31.6 40.7)
    ([28] * 6, 1128, 32, 256, 3), ([3] * 96, 1771, 32, 320, 3), ([1] * 192, 2047, 33, 128, 3), ([25, 9, 11, 20], 694, 40, 64, 3), ([5] * 8, 250, 32, 256, 3),
    # more row tiles than can be there at once (24.7 33.1, 68.2 90, 82 103)
    ([2] * 320, 522, 8, 256, 2), ([1] * 320, 1500, 33, 256, 2), ([116] * 24, 2172, 8, 192, 2)])
def test_splits_of_latent_portions(lens, kv, heads, rank, splits):
    assert _latent_splits(lens, kv, heads, rank) == splits
@pytest.mark.parametrize("tokens, kv, heads, rank, window, splits", [
    # a token's keys shared by the waves of a workgroup: up to 2048 tiles of 64 keys in all, 1365 for more than 16 heads and 64 tokens
    (1, 149, 32, 512, 0, 3), (32, 1747, 32, 512, 512, 5), (64, 2047, 32, 512, 0, 4), (64, 2047, 32, 128, 0, 8), (128, 300, 32, 512, 0, 1), (300, 300, 16, 512, 0, 1),
    # row tiles of 64 rows, as many splits as before there was the other form (us there and in it: 29.6 43.2, 53 69, 44 59, 33.8 37.3, 61 66)
    (192, 2047, 32, 128, 0, 3), (192, 2047, 32, 320, 0, 3), (192, 2047, 8, 320, 0, 3), (128, 2047, 8, 320, 0, 4), (160, 2047, 32, 320, 0, 4), (64, 8000, 32, 128, 0, 8)])
def test_splits_of_single_latent_tokens(tokens, kv, heads, rank, window, splits):
    assert _latent_splits([1] * tokens, kv, heads, rank, window) == splits


@pytest.mark.parametrize("stride", [128 * 128, 2 ** 28 - 1, 2 ** 28, 2 ** 40])
@pytest.mark.parametrize("mode, per_channel", [(0, 0), (0, 1), (1, 1), (2, 0)])
def test_rows_far_apart_still_go_in_chunks(stride, mode, per_channel):
    """The launch ahead is asked for wherever chunks serve; how far apart rows are is no reason not to."""
    from hydrainfer_amd import _lib
    HX_F32 = 0
    a = _lib.hxm_state_scan_args(q_dtype=HX_F32, k_dtype=HX_F32, v_dtype=HX_F32, n_tokens=1151, n_seq=1, heads=32, qk_heads=32, dim=128, vdim=128, mode=mode,
                                 decay_per_channel=per_channel, q_stride=stride, k_stride=stride, v_stride=stride)
    assert _lib.mix_lib().hxm_state_scan_workspace(ctypes.byref(a)) > 0


@pytest.mark.parametrize("n_seq, q, heads, kv_heads, dim, vdim, kv, mask, size, splits", [
    # one row tile a key head: two splits from four tiles of 32 keys on, four from six on, more where they take rounds of four
    (1, 1, 32, 8, 128, 128, 64, 0, 0, 1), (1, 1, 32, 8, 128, 128, 127, 0, 0, 2), (1, 1, 32, 8, 128, 128, 160, 0, 0, 2), (1, 1, 32, 8, 128, 128, 161, 0, 0, 4),
    (1, 1, 32, 8, 128, 128, 512, 0, 0, 4), (1, 1, 32, 8, 128, 128, 513, 0, 0, 8), (1, 1, 32, 8, 128, 128, 576, 0, 0, 12), (1, 1, 32, 8, 128, 128, 20000, 0, 0, 64),
    (7, 1, 32, 8, 128, 128, 700, 0, 0, 12), (2, 16, 32, 8, 128, 128, 1500, 0, 0, 16), (1, 1, 8, 1, 64, 128, 700, 1, 300, 4), (1, 1, 8, 1, 64, 128, 700, 2, 60, 1),
    # 64 row tiles and more of up to 2000 keys: four in the place of up to eleven
    (8, 1, 32, 8, 128, 128, 704, 0, 0, 4), (8, 1, 32, 8, 128, 128, 768, 0, 0, 12), (16, 1, 32, 8, 128, 128, 2000, 0, 0, 4), (16, 1, 32, 8, 128, 128, 2001, 0, 0, 8),
    # more than 128 row tiles behind longer keys: seven, and four where there would be seven
    (17, 1, 32, 8, 128, 128, 2000, 0, 0, 4), (17, 1, 32, 8, 128, 128, 2001, 0, 0, 7), (18, 1, 32, 8, 128, 128, 2100, 0, 0, 7), (19, 1, 32, 8, 128, 128, 2100, 0, 0, 4),
    # 257 - 383 row tiles: as many as there are waves for
    (32, 1, 32, 8, 128, 128, 700, 0, 0, 4), (33, 1, 32, 8, 128, 128, 700, 0, 0, 4), (42, 1, 32, 8, 128, 128, 700, 0, 0, 4), (43, 1, 32, 8, 128, 128, 700, 0, 0, 3),
    (47, 1, 32, 8, 128, 128, 700, 0, 0, 3), (48, 1, 32, 8, 128, 128, 700, 0, 0, 4), (64, 1, 32, 8, 128, 128, 700, 0, 0, 2), (127, 1, 32, 8, 128, 128, 700, 0, 0, 2),
    (128, 1, 32, 8, 128, 128, 700, 0, 0, 1),
    # portions of 64 rows and more: only few of them behind many keys; heads of other sizes: 2048 waves
    (1, 100, 32, 8, 128, 128, 2000, 0, 0, 4), (1, 100, 32, 8, 128, 128, 1000, 0, 0, 1), (1, 1, 32, 8, 96, 96, 2000, 0, 0, 31)])
def test_splits_of_attention(n_seq, q, heads, kv_heads, dim, vdim, kv, mask, size, splits):
    import torch
    from hydrainfer_amd import _lib
    a = _lib.hxm_biased_attn_args(n_tokens=n_seq * q, n_seq=n_seq, n_heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, block_size=16, mask_kind=mask, mask_size=size,
                                  max_q_len=q, dtype=_lib._DTYPE[torch.bfloat16])
    n, floats = ctypes.c_int32(), ctypes.c_int64()
    plan = lambda: _lib.mix_lib().hxm_biased_attention_plan(ctypes.byref(a), kv, ctypes.byref(n), ctypes.byref(floats))
    tiles = n_seq * kv_heads * ((q * (heads // kv_heads) + 15) // 16)
    assert plan() == 0 and n.value == splits
    assert floats.value == (0 if splits == 1 else tiles * splits * 16 * ((vdim + 15) // 16 * 16 + 2))
    # no splits for what the forms with splits do not serve
    for name, value in (("form", 1), ("dtype", 0), ("max_q_len", 0), ("dim", 260), ("vdim", 36)):
        before = getattr(a, name)
        setattr(a, name, value)
        assert plan() == 0 and (n.value, floats.value) == (1, 0)
        setattr(a, name, before)
