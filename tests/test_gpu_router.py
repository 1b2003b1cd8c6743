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
