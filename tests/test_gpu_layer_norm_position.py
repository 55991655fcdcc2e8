"""Channel-first LayerNorm of few short images of an odd length (a wavefront per position) against float64.

The mean and the variance are fp32 sums of C <= 1024 values of unit size: (C + 4) * 2^-24 of their magnitude each, so that a result
of at most 6 is off by 6 * 3 * 1028 * 2^-24 < 1.2e-3 at the very worst; 16-bit results add half an ulp."""
import pytest
import torch

from vmamba_amd.norm import layer_norm_cf_hip

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("channel_last", [True, False])
@pytest.mark.parametrize("B,C,H,W", [
    (1, 1, 1, 1),             # one value: the variance is 0
    (1, 768, 7, 7), (3, 63, 3, 3), (2, 65, 5, 7),      # a channel under and over a wavefront
    (1, 1024, 13, 13), (1, 1032, 13, 13),              # the most channels, and beyond them
    (16, 48, 7, 7), (17, 48, 7, 7),                    # the most positions, and beyond them
])
def test_few_positions(B, C, H, W, channel_last):
    print("CASE layer_norm positions", B, C, H, W, channel_last, flush=True)
    g = torch.Generator().manual_seed(C)
    x, w, b = torch.randn(B, C, H, W, generator=g), torch.randn(C, generator=g), torch.randn(C, generator=g)
    want = torch.nn.functional.layer_norm(x.double().permute(0, 2, 3, 1), (C,), w.double(), b.double(), 1e-5)
    for dtype, ulp in ((torch.float32, 0.0), (torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)):
        wd, bd = w.to(dtype), b.to(dtype)
        ref = want if dtype == torch.float32 else torch.nn.functional.layer_norm(
            x.double().permute(0, 2, 3, 1), (C,), wd.double(), bd.double(), 1e-5)
        got = layer_norm_cf_hip(x.to(DEV), wd.to(DEV), bd.to(DEV), 1e-5, out_channel_last=channel_last, out_dtype=dtype).cpu().double()
        got = got.reshape(B, H, W, C) if channel_last else got.reshape(B, C, H, W).permute(0, 2, 3, 1)
        assert bool(((got - ref).abs() <= ulp * ref.abs() + 1.2e-3 * w.double().abs().clamp(min=1)).all())
