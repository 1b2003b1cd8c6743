"""The grouped product of the experts' rows (csrc/moe_mix.hip, the matrix-core form) at the edges of its tiles: one row, a tile
and one row more, columns and k that no tile divides, experts without rows, rows gathered and rows as they come, and inputs
whose rows lie further apart than 32-bit offsets reach."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LIMIT, ALPHA, SHIFT = 7.0, 1.702, 1.0


def _reference(x, w, act):
    """(result, bound of its float sum's error) of one expert's rows in 64 bits"""
    z = x @ w.t()
    dz = w.shape[1] * 2.0 ** -24 * (x.abs() @ w.abs().t())
    if act == "relu2":
        return z.clamp(min=0) ** 2, 2 * (z.abs() + dz) * dz
    if act == "glu":
        n = z.shape[1] // 32
        g, u = z.view(-1, n, 2, 16).unbind(2)
        dg, du = dz.view(-1, n, 2, 16).unbind(2)
        g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
        # |d/dg g sigmoid(alpha g)| < 1.1, and a few units in the last place of the hardware's exponential and reciprocal
        silu = g * torch.sigmoid(ALPHA * g)
        y = silu * (u + SHIFT)
        return y.reshape(-1, 16 * n), (1.1 * dg * (u + SHIFT).abs() + silu.abs() * du + 2.0 ** -19 * y.abs()).reshape(-1, 16 * n)
    return z, dz


@pytest.mark.parametrize("rows", [[1], [0, 33, 0, 31], [129, 0, 127], [128, 200], [256, 257], [1, 511, 128, 130], [0, 700]])
@pytest.mark.parametrize("n, k", [(32, 8), (160, 72), (288, 64), (544, 200)])
@pytest.mark.parametrize("act", ["none", "relu2", "glu"])
def test_grouped_linear_edges(rows, n, k, act):
    _check(rows, n, k, act, False)


# more slices of 64 than a tile has slots for, several turns of them, with a tail and without: tiles of 32 and 64 rows
@pytest.mark.parametrize("rows", [[20, 0, 33], [128, 61], [300, 257]])
@pytest.mark.parametrize("k", [256, 328, 1032])
@pytest.mark.parametrize("act", ["none", "glu"])
def test_grouped_linear_over_many_slices(rows, k, act):
    _check(rows, 288, k, act, False)


# few rows an expert and short and long weight rows (four slots and six), with a tail and without, columns that no tile divides
@pytest.mark.parametrize("rows", [[1], [0, 16, 17], [32, 0, 31], [33, 1, 0, 20]])
@pytest.mark.parametrize("n, k", [(96, 2040), (160, 2048), (32, 2056), (224, 2432)])
@pytest.mark.parametrize("act", ["none", "glu"])
def test_grouped_linear_of_few_rows(rows, n, k, act):
    _check(rows, n, k, act, False)


# more experts than a wave has lanes, with rows on both sides of every 64th
@pytest.mark.parametrize("experts", [63, 64, 65, 130])
@pytest.mark.parametrize("every", [1, 21])
def test_grouped_linear_of_many_experts(experts, every):
    _check([1 + 40 * (e % 5 == 0) if e % every == 0 or e in (63, 64, 128) else 0 for e in range(experts)], 96, 136, "glu", False)


# long weight rows and about a hundred rows an expert
@pytest.mark.parametrize("rows", [[70, 100], [129, 0, 150]])
@pytest.mark.parametrize("k, act", [(2560, "glu"), (2568, "none")])
def test_grouped_linear_of_long_weight_rows(rows, k, act):
    _check(rows, 160, k, act, False)


# enough columns for tiles of 128 rows, and for tiles of 256 of which not every one starts where the walk from tile to tile needs it: up to a tile's
# rows and one more, several turns of the slots, with a tail and without
@pytest.mark.parametrize("rows, n, k, act, tile", [
    ([128, 128], 8352, 1600, "glu", 128), ([129, 99], 8360, 1544, "none", 128), ([65, 127], 8352, 1544, "relu2", 128), ([128, 1, 128], 8352, 1600, "none", 128),
    ([256, 257], 11040, 1096, "glu", 256), ([300, 212], 11044, 1088, "none", 256)])
def test_grouped_linear_in_large_tiles(rows, n, k, act, tile):
    from hydrainfer_amd import _lib
    assert _lib.mix_lib().hxm_grouped_linear_tile_rows(sum(rows), len(rows), n, k) == tile
    _check(rows, n, k, act, False)


# tiles of 64 and of 128 rows by eight waves, 64 columns wide and 128: up to a tile's rows and one more, columns that no tile divides, with a
# tail and without
@pytest.mark.parametrize("rows, n, k, act, tile", [
    ([129, 71], 4136, 264, "none", 128), ([1, 130, 128, 141], 2080, 520, "glu", 128), ([128, 72], 4128, 320, "relu2", 128), ([129, 171], 6184, 136, "none", 128),
    ([172, 128], 6176, 520, "glu", 128), ([65, 1, 127, 87], 8256, 264, "glu", 64), ([63, 337], 8264, 520, "none", 64), ([65, 64, 1, 150], 8256, 320, "none", 64)])
def test_grouped_linear_by_eight_waves(rows, n, k, act, tile):
    from hydrainfer_amd import _lib
    assert _lib.mix_lib().hxm_grouped_linear_tile_rows(sum(rows), len(rows), n, k) == tile
    _check(rows, n, k, act, False)


# tiles of 128 x 192, 192 x 192 and 128 x 256 (the last three): up to a tile's rows and one more, columns that no tile divides, with a tail and without
@pytest.mark.parametrize("rows, n, k, act, tile", [
    ([129, 1, 128, 142], 8264, 520, "none", 128), ([100, 127, 173, 0], 8256, 520, "glu", 128), ([64, 192, 0, 144], 8264, 1096, "relu2", 128),
    ([192, 193, 1, 126], 8264, 264, "none", 192), ([191, 321, 0, 0], 8256, 1096, "glu", 192), ([128, 129, 1, 127, 115], 11040, 520, "glu", 128),
    ([255, 257, 128, 360], 6184, 520, "none", 128), ([385, 127, 0, 488], 6184, 320, "relu2", 128)])
def test_grouped_linear_in_tiles_for_full_rounds(rows, n, k, act, tile):
    from hydrainfer_amd import _lib
    assert _lib.mix_lib().hxm_grouped_linear_tile_rows(sum(rows), len(rows), n, k) == tile
    _check(rows, n, k, act, False)


# enough tiles for those of 256 x 256: from tile to tile with two slices and with more, columns in 8s and whole turns, the last ones in
# part; and k and n that take the form before it
@pytest.mark.parametrize("rows", [[300, 257], [700, 0, 129], [1, 513]])
@pytest.mark.parametrize("n, k, act", [(11040, 128, "glu"), (11048, 128, "none"), (11048, 192, "relu2"), (33088, 192, "glu"), (11040, 1088, "glu"),
                                       (11044, 128, "none"), (11040, 200, "glu")])
def test_grouped_linear_from_tile_to_tile(rows, n, k, act):
    _check(rows, n, k, act, False)


# the same with rows enough that tiles of 256 are chosen for two slices too: the walk starts and ends in the first turn of its slots
@pytest.mark.parametrize("rows", [[500, 520], [1000, 20], [1, 1023]])
@pytest.mark.parametrize("n, k, act", [(11040, 128, "glu"), (11048, 128, "none"), (11048, 192, "relu2"), (33088, 192, "glu")])
def test_grouped_linear_from_tile_to_tile_with_few_slices(rows, n, k, act):
    from hydrainfer_amd import _lib
    assert _lib.mix_lib().hxm_grouped_linear_tile_rows(sum(rows), len(rows), n, k) == 256
    _check(rows, n, k, act, False)


# the same with more experts than a wave has lanes, some of them without rows
def test_grouped_linear_from_tile_to_tile_of_many_experts():
    from hydrainfer_amd import _lib
    rows = [0 if e in (0, 5, 64) else 257 if e % 2 else 240 for e in range(67)]
    assert _lib.mix_lib().hxm_grouped_linear_tile_rows(sum(rows), len(rows), 512, 256) == 256
    _check(rows, 512, 256, "none", False)


@pytest.mark.parametrize("rows", [[1, 30], [129, 0, 127], [256, 257]])
def test_grouped_linear_of_rows_far_apart(rows):
    _check(rows, 160, 200, "none", True)


@pytest.mark.parametrize("rows", [[3, 0, 5], [60, 70], [300, 1]])
def test_grouped_linear_of_few_rows_out_of_a_long_input(rows):
    # rows on both sides of 4 GiB, where an offset of 32 bits would start again at x: there lie other numbers
    from hydrainfer_amd._C.kernel.moe_mix import grouped_linear
    E, total, n, k, stride = len(rows), sum(rows), 160, 328, 2 ** 20
    g = torch.Generator().manual_seed(total)
    x = torch.empty((2600, stride), dtype=torch.bfloat16, device="cuda")
    src = torch.randperm(2600, generator=g)[:total].int()
    src[:2] = torch.tensor([2599, 2599 - 2048])
    x[:, :k] = torch.randn((2600, k), generator=g).bfloat16().cuda()
    w = (torch.randn((E, n, k), generator=g) * k ** -0.5).bfloat16()
    seg = [0]
    for r in rows:
        seg.append(seg[-1] + r)
    got = grouped_linear(x[:, :k], w.cuda(), torch.tensor(seg, dtype=torch.int32, device="cuda"), total, src=src.cuda()).double().cpu()
    xs = x[:, :k].cpu().double()[src.long()]
    for e in range(E):
        want, bound = _reference(xs[seg[e]:seg[e + 1]], w[e].double(), "none")
        off = (got[seg[e]:seg[e + 1]] - want).abs()
        assert bool((off <= 2.0 ** -8 * want.abs() + 1.01 * bound + 1e-30).all()), (e, float(off.max()))      # one rounding to bfloat16


def _check(rows, n, k, act, far):
    from hydrainfer_amd._C.kernel.moe_mix import grouped_linear
    g = torch.Generator().manual_seed(len(rows) * 1000 + sum(rows) + n + k)
    E, total = len(rows), sum(rows)
    x = torch.randn((total, k), generator=g).bfloat16()
    w = (torch.randn((E, n, k), generator=g) * k ** -0.5).bfloat16()
    src = torch.randperm(total, generator=g).int()
    seg = [0]
    for r in rows:
        seg.append(seg[-1] + r)
    xd = x.cuda()
    if far:                      # the same rows, (2^30 / rows) elements apart and more
        stride = (2 ** 30 // total + 8) // 8 * 8 + 8
        wide = torch.empty(total * stride, dtype=torch.bfloat16, device="cuda").view(total, stride)
        wide[:, :k] = xd
        xd = wide[:, :k]
    segd = torch.tensor(seg, dtype=torch.int32, device="cuda")
    for gather in (None, src):
        got = grouped_linear(xd, w.cuda(), segd, total, src=None if gather is None else gather.cuda(), act=act, limit=LIMIT, alpha=ALPHA,
                             up_shift=SHIFT).double().cpu()
        xs = x.double() if gather is None else x.double()[gather.long()]
        for e in range(E):
            want, bound = _reference(xs[seg[e]:seg[e + 1]], w[e].double(), act)
            off = (got[seg[e]:seg[e + 1]] - want).abs()
            assert bool((off <= 2.0 ** -8 * want.abs() + 1.01 * bound + 1e-30).all()), (e, float(off.max()))      # one rounding to bfloat16
