"""Weight gradient of the projections in single precision (ss2d_linear_dw_f32) against float64.

An output is a sum of M products in fp32: rounding leaves it within M * 2^-24 of the sum of the products' magnitudes (the bound
for any order of the sum)."""
import pytest
import torch
import torch.nn as nn

from vmamba_amd.linear import LinearDw, linear_dw_hip, linear_dw_pays

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,N,K", [
    (1, 4, 4),               # one position: every other one masked
    (129, 64, 64),           # two shares, the second one position long
    (127, 68, 60),           # tiles one column group over and under
    (515, 100, 40),
    (4096, 384, 384),
    (5001, 96, 192),
    (131, 2052, 2048),       # more tiles than workgroups are resident: one share
])
def test_linear_dw(M, N, K):
    print("CASE linear_dw", M, N, K, flush=True)
    g = torch.Generator().manual_seed(M)
    x, dy = torch.randn(M, K, generator=g), torch.randn(M, N, generator=g)
    got = linear_dw_hip(x.to(DEV), dy.to(DEV)).cpu().double()
    want, size = dy.double().t() @ x.double(), dy.double().abs().t() @ x.double().abs()
    assert bool(((got - want).abs() <= M * 2.0 ** -24 * size + 1e-30).all())


@pytest.mark.parametrize("with_residual", [False, True])
def test_linear_dw_autograd(with_residual):
    print("CASE linear_dw autograd", with_residual, flush=True)
    torch.manual_seed(0)
    layer = nn.Linear(48, 64, bias=False).to(DEV)
    x = torch.randn(8, 32, 16, 48, device=DEV, requires_grad=True)
    res = torch.randn(8, 32, 16, 64, device=DEV, requires_grad=True) if with_residual else None
    dy = torch.randn(8, 32, 16, 64, device=DEV)
    assert linear_dw_pays(layer, x)
    wanted = [x, layer.weight] + ([res] if with_residual else [])
    y = LinearDw.apply(x, layer.weight, res)
    y_ref = layer(x) if res is None else res + layer(x)
    got, want = torch.autograd.grad(y, wanted, dy), torch.autograd.grad(y_ref, wanted, dy)
    # y and dx are the layer's own products in another call: 48 and 64 of them, n * 2^-24 of the sum of their magnitudes each,
    # and one more rounding where the residual is added
    assert torch.allclose(y, y_ref, rtol=0, atol=1e-5)
    w, dy2, x2 = layer.weight.detach().double(), dy.double().reshape(-1, 64), x.detach().double().reshape(-1, 48)
    dx, dw = got[0].double().reshape(-1, 48), got[1].double()
    assert bool(((dx - dy2 @ w).abs() <= 64 * 2.0 ** -24 * (dy2.abs() @ w.abs())).all())
    assert bool(((dw - dy2.t() @ x2).abs() <= 4096 * 2.0 ** -24 * (dy2.abs().t() @ x2.abs())).all())
    assert all(torch.equal(a, b) for a, b in zip(got[2:], want[2:]))                     # the residual's is dy
    # second order: through the library's products
    y = LinearDw.apply(x, layer.weight, res)
    (dw,) = torch.autograd.grad((y * y).sum(), layer.weight, create_graph=True)
    assert torch.autograd.grad(dw.sum(), x)[0].shape == x.shape


def test_linear_dw_of_views_between_16_byte_boundaries():
    """x and dy as contiguous views one element into their storage, as slices and the backward of a concatenation give them:
    the gradients are the layer's own (4096 products of unit size: M * 2^-24 of their magnitudes' sum)."""
    print("CASE linear_dw unaligned", flush=True)
    torch.manual_seed(1)
    layer = nn.Linear(48, 64, bias=False).to(DEV)
    aligned = [torch.randn(4096, n, device=DEV) for n in (48, 64)]
    shifted = []
    for t in aligned:
        shifted.append(torch.empty(t.numel() + 1, device=DEV)[1:].view(t.shape).copy_(t))
        assert shifted[-1].is_contiguous() and shifted[-1].data_ptr() % 16 == 4
    want, size = aligned[1].double().t() @ aligned[0].double(), aligned[1].double().abs().t() @ aligned[0].double().abs()
    for x, dy in ((shifted[0], aligned[1]), (aligned[0], shifted[1]), shifted):
        x = x.detach().requires_grad_()
        assert linear_dw_pays(layer, x)
        dx, dw = torch.autograd.grad(LinearDw.apply(x, layer.weight, None), [x, layer.weight], dy)
        assert bool(((dw.double() - want).abs() <= 4096 * 2.0 ** -24 * size).all())
        assert torch.equal(dx, torch.autograd.grad(layer(x), x, dy)[0])


def test_linear_dw_rule():
    layer, x = nn.Linear(48, 64, bias=False).to(DEV), torch.zeros(4096, 48, device=DEV)
    assert linear_dw_pays(layer, x) and not linear_dw_pays(layer, x[:4095]) and not linear_dw_pays(layer, x.half())
    with torch.no_grad():
        assert not linear_dw_pays(layer, x)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not linear_dw_pays(layer, x)
    assert not linear_dw_pays(nn.Linear(48, 64).to(DEV), x) and not linear_dw_pays(nn.Linear(48, 66, bias=False).to(DEV), x)
    layer.register_forward_hook(lambda *a: None)
    assert not linear_dw_pays(layer, x)
