"""The channel-last depthwise convolution of few images: tiles of 8 channels up to the line, 64 or 32 beyond it, the same bits."""
import pytest
import torch
import torch.nn.functional as F

from vmamba_amd.conv import dwconv3x3_silu_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("silu,with_bias", [(True, False), (False, True)])
@pytest.mark.parametrize("C,H,W", [(96, 56, 56), (384, 14, 14), (768, 7, 7), (64, 1, 1), (64, 3, 2), (32, 5, 4), (32, 28, 12), (64, 9, 120), (96, 40, 116), (64, 11, 19)])
def test_few_images(C, H, W, silu, with_bias, dtype):
    print("CASE dwconv_few", C, H, W, silu, with_bias, dtype, flush=True)
    g = torch.Generator().manual_seed(C + H + W)
    x = torch.randn(1, H, W, C, generator=g).to(dtype)
    w = (torch.randn(C, 1, 3, 3, generator=g) / 3).to(dtype)
    b = torch.randn(C, generator=g).to(dtype) if with_bias else None
    run = lambda t: dwconv3x3_silu_hip(t.cuda(), w.cuda(), None if b is None else b.cuda(), in_channel_last=True, apply_silu=silu)
    got = run(x)
    many = run(x.expand(128, H, W, C).contiguous())          # 128 workgroups or more: the standard split
    assert torch.equal(many, got.expand_as(many))
    want = F.conv2d(x.double().permute(0, 3, 1, 2), w.double(), None if b is None else b.double(), padding=1, groups=C)
    # nine products summed in fp32, rounded to the 16-bit type once, and once more behind the SiLU (slope at most 1.1)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = u * want.abs() * (1.1 if silu else 1.0) + 16 * 2.0 ** -24 * 9 * x.abs().max().double() * w.abs().max().double()
    if silu:
        want = F.silu(want)
        bound = bound + u * want.abs() + 2.0 ** -20
    # 2^-24: the spacing of fp16's subnormals, half of it at each of the two roundings
    assert ((got.cpu().double() - want).abs() <= 1.02 * bound + 2.0 ** -24).all()
