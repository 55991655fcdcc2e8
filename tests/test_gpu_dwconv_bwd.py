"""ss2d_dwconv3x3_silu_bwd against float64 autograd of silu(conv2d(x)) on the same values.

Every result is a sum of n products (9 for dx, B H W for the weights and the bias), each factor carrying a few fp32
roundings: off by at most (n + 16) * 2^-23 of the sum of their magnitudes, bounded here by running the same sums on absolute
values (|silu'| <= 1.1), plus the rounding to the result's type."""
import pytest
import torch
import torch.nn.functional as F

from vmamba_amd.conv import DwConv3x3SiLU, dwconv3x3_silu_bwd_hip, dwconv_silu_trainable

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def check(got, want, size, n, dtype):
    bound = (n + 16) * 2.0 ** -23 * size + 2 * EPS[dtype] * want.abs() + (2.0 ** -24 if dtype == torch.float16 else 1e-37)
    assert bool(((got.cpu().double() - want).abs() <= bound).all()), ((got.cpu().double() - want).abs() - bound).max()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,H,W", [(9, 6, 14, 14),         # several planes a round and a short last one
                                     (3, 5, 7, 9), (1, 3, 1, 1), (2, 2, 1, 40), (70, 1, 3, 5),
                                     (2, 3, 56, 56),         # one whole plane
                                     (2, 2, 100, 96),        # rows of a plane with a halo, even parts
                                     (1, 2, 131, 300)])      # many parts, the last one short
def test_gradients(B, D, H, W, dtype):
    print("CASE dwconv bwd", B, D, H, W, dtype, flush=True)
    g = torch.Generator().manual_seed(H * W)
    x, dy = torch.randn(B, D, H, W, generator=g).to(dtype), torch.randn(B, D, H, W, generator=g).to(dtype)
    w, b = (torch.randn(D, 1, 3, 3, generator=g) * 0.4).to(dtype), torch.randn(D, generator=g).to(dtype)
    ref = [t.double().requires_grad_() for t in (x, w, b)]
    want = torch.autograd.grad(F.silu(F.conv2d(*ref, padding=1, groups=D)), ref, dy.double())
    ab = [t.double().abs().requires_grad_() for t in (x, w)]
    size = torch.autograd.grad(F.conv2d(*ab, padding=1, groups=D), ab, 1.1 * dy.double().abs())
    # the error of z moves silu' by at most half of it: 9 products and the bias
    z_size = F.conv2d(ab[0], ab[1], padding=1, groups=D).detach() + b.double().abs().view(1, D, 1, 1)
    wide = torch.autograd.grad(F.conv2d(*ab, padding=1, groups=D), ab, dy.double().abs() * z_size)
    got = dwconv3x3_silu_bwd_hip(*(t.to(DEV) for t in (x, w, b, dy)))
    check(got[0], want[0], size[0] + wide[0], 9, dtype)
    check(got[1], want[1], size[1] + wide[1], B * H * W, dtype)
    check(got[2], want[2], (dy.double().abs() * (1.1 + z_size)).sum((0, 2, 3)), B * H * W, dtype)
    if dtype == torch.float32:              # the forward: one rounding of z and a few of the SiLU
        y = DwConv3x3SiLU.apply(*(t.to(DEV) for t in (x, w, b)), False).cpu().double()
        z = F.conv2d(*(t.double() for t in (x, w, b)), padding=1, groups=D)
        assert bool(((y - F.silu(z)).abs() <= 6 * 2.0 ** -24 * (F.silu(z).abs() + z.abs()) + 1e-37).all())
    again = dwconv3x3_silu_bwd_hip(*(t.to(DEV) for t in (x, w, b, dy)))
    assert all(torch.equal(p, q) for p, q in zip(got, again))


@pytest.mark.parametrize("channel_last", [False, True])
@pytest.mark.parametrize("has_bias", [False, True])
def test_function_in_both_layouts(channel_last, has_bias):
    conv = torch.nn.Conv2d(8, 8, 3, padding=1, groups=8, bias=has_bias).to(DEV)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, 8, 10, 12, generator=g).to(DEV)
    dy = torch.randn(2, 8, 10, 12, generator=g).to(DEV)
    xin = (x.permute(0, 2, 3, 1).contiguous() if channel_last else x).requires_grad_()
    assert dwconv_silu_trainable(conv, xin, channel_last)
    params = [xin] + list(conv.parameters())
    got = torch.autograd.grad(DwConv3x3SiLU.apply(xin, conv.weight, conv.bias, channel_last), params, dy.permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2))
    want = torch.autograd.grad(F.silu(conv(xin.permute(0, 3, 1, 2) if channel_last else xin)), params, dy)
    for p, q in zip(got, want):
        assert p.shape == q.shape and torch.allclose(p, q, rtol=1e-4, atol=1e-4)     # 240 products of magnitude about 1


def test_what_stays_on_the_operators():
    x = torch.zeros(1, 8, 6, 6, device=DEV)
    plain = torch.nn.Conv2d(8, 8, 3, padding=1, groups=8).to(DEV)
    assert dwconv_silu_trainable(plain, x, False) and not dwconv_silu_trainable(plain, x.half(), False)
    for other in (torch.nn.Conv2d(8, 8, 3, padding=1), torch.nn.Conv2d(8, 8, 3, padding=1, groups=8, padding_mode="circular"),
                  torch.nn.Conv2d(8, 8, 3, padding=1, dilation=2, groups=8)):
        assert not dwconv_silu_trainable(other.to(DEV), x, False)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not dwconv_silu_trainable(plain, x, False)
    plain.register_forward_hook(lambda m, i, o: o)
    assert not dwconv_silu_trainable(plain, x, False)
    assert not dwconv_silu_trainable(torch.nn.Conv2d(1, 1, 3, padding=1).to(DEV), torch.zeros(1, 1, 2, 5000, device=DEV), False)
