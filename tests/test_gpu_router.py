"""The router's two forms (csrc/moe_mix.hip: a workgroup a token, sixteen tokens a workgroup) on both sides of the rule between them,
with rows that end inside a wave's piece, against logits in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [4, 260, 1020, 1028, 2052])
@pytest.mark.parametrize("E, T", [(16, 1), (16, 256), (16, 257), (16, 512), (16, 513), (33, 256), (33, 257), (128, 256), (128, 300)])
@pytest.mark.parametrize("biased", [True, False])
def test_router_forms(K, E, T, biased):
    from hydrainfer_amd._C.kernel.moe_mix import router_topk
    g = torch.Generator().manual_seed(K + E + T)
    top = 5
    x, w, b = torch.randn(T, K + 4, generator=g), torch.randn(E, K, generator=g), torch.randn(E, generator=g)
    weights, experts = (t.cpu() for t in router_topk(x.cuda()[:, 4:], w.cuda(), b.cuda() if biased else None, top))
    z = x[:, 4:].double() @ w.double().t() + (b.double() if biased else 0.0)
    # a sum of K products in float, in any order: each rounding is 2^-24 of a partial sum, none larger than the sum of magnitudes
    eps = (K + 2) * 2.0 ** -24 * (x[:, 4:].abs().double() @ w.abs().double().t() + 1.0).max(dim=1, keepdim=True).values
    e = experts.long()
    assert all(len(set(row)) == top for row in e.tolist())
    chosen = z.gather(1, e)
    best = z.topk(top, dim=1).values
    assert bool(((chosen - best).abs() <= 2 * eps).all())
    want = torch.softmax(chosen, dim=1)
    # a logit off by eps moves a weight by at most 2 eps of itself; 1e-6 for the exponentials and the quotient
    assert bool(((weights.double() - want).abs() <= want * (2 * torch.expm1(2 * eps) + 1e-6) + 1e-30).all())


# four tokens a workgroup: its groups of experts, ends of rows inside a wave's piece and inside a round of waves, and the lines at 128, 256, 1024 and 3072 tokens
@pytest.mark.parametrize("K", [4, 516, 1028, 2052, 4100])
@pytest.mark.parametrize("E, T", [(5, 1), (8, 1024), (8, 1027), (9, 130), (16, 1025), (16, 3071), (16, 3073), (17, 258), (32, 1024), (32, 1025)])
def test_four_tokens_a_workgroup(K, E, T):
    test_router_forms(K, E, T, True)


# the combine (csrc/moe_mix.hip): rows in pieces of eight, four and single elements, on both sides of the 256 tokens up to which pieces are of four
@pytest.mark.parametrize("W", [8, 1028, 2048, 2056, 4099])
@pytest.mark.parametrize("T", [1, 256, 257])
@pytest.mark.parametrize("top, shared, missing", [(1, False, False), (3, True, False), (5, True, True)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_combine_pieces(W, T, top, shared, missing, dt):
    from hydrainfer_amd._C.kernel.moe_mix import moe_combine
    g = torch.Generator().manual_seed(W + T + top)
    y, sh, same = (torch.randn(n, W, generator=g).to(dt) for n in (T * top, T, T))
    row_of = torch.randperm(T * top, generator=g).int().view(T, top)
    if missing:
        row_of[::3, 1] = -1
    w = torch.rand(T, top, generator=g)
    got = moe_combine(y.cuda(), row_of.cuda(), w.cuda(), sh.cuda() if shared else None, identity=same.cuda() if missing else None).cpu()
    parts = [torch.where(row_of[:, k:k + 1] >= 0, y[row_of[:, k].clamp(min=0).long()].double(), same.double() if missing else torch.zeros(())) * w[:, k:k + 1].double()
             for k in range(top)]
    parts += [sh.double()] if shared else []
    want, size = sum(parts), sum(p.abs() for p in parts)
    # at most seven sums in float and one rounding to the result's type
    unit = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -23
    assert bool(((got.double() - want).abs() <= unit * want.abs() + 8 * 2.0 ** -24 * size + 1e-30).all())
