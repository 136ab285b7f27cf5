"""mm_readout2 (energy and gradient of the hidden-layer readout) at hidden widths around its 16- and 32-column forms and
node counts around its 16-node workgroups, against fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 17, 333])
@pytest.mark.parametrize("H", [1, 16, 17, 32])
def test_readout2(n, H):
    from mace_onegpu import _lib
    g = torch.Generator().manual_seed(n + H)
    h = torch.randn(n, 132, generator=g)
    W1, w2 = torch.randn(128, H, generator=g) / 128 ** 0.5, torch.randn(H, generator=g)
    eat0 = torch.randn(n, generator=g, dtype=torch.float64)
    cst, scale = 1.6, 0.7
    eat, gh = eat0.cuda(), torch.full((n + 1, 136), float("nan"), device="cuda")
    _lib.K.mm_readout2(n, h.cuda(), 132, W1.cuda(), w2.cuda(), H, cst, scale, eat, gh, 136, _lib.stream())
    x = h[:, :128].double().requires_grad_(True)
    z = x @ W1.double()
    y = scale * cst * (z * torch.sigmoid(z)) @ w2.double()
    y.sum().backward()
    # 128 products per unit, then H terms: fp32 roundings of sums of that many terms
    mag = scale * cst * (x.detach().abs() @ W1.abs().double()) @ w2.abs().double()
    assert bool(((eat.cpu() - eat0 - y.detach()).abs() <= 2 ** -24 * 24 * mag + 1e-7).all())
    gmag = scale * cst * 1.1 * (w2.abs()[None] * W1.abs()).double().sum(1)
    # |d2 silu| <= 0.5: the error of z enters the gradient through it
    zerr = 2 ** -24 * 24 * (x.detach().abs() @ W1.abs().double()).max()
    assert bool(((gh[:n, :128].cpu().double() - x.grad).abs() <= gmag * (2 ** -24 * (16 + H) + zerr)).all())
    assert bool(gh[n:].isnan().all()) and bool(gh[:, 128:].isnan().all())
