"""ss2d_linear_tiles and ss2d_conv3x3s2_cl against float64 at the edges of their tiles, and who takes them.

The sums are fp32 of exact 16-bit products; a result is the float64 one rounded to 16 bits once (GELU's argument too), up to the sums'
K 2^-24 of their terms' magnitudes: half a unit of the result's last place (2^-8 or 2^-11 of it) and a little."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from vmamba_amd import _lib, vssm
from vmamba_amd.linear import linear_tiles_fusable, linear_tiles_hip, linear_tiles_pays
from vmamba_amd.stem import conv_tiles_fusable, conv_tiles_hip, conv_tiles_pays
from vmamba_amd.vssm import Mlp, VSSBlock, vmamba_tiny_s1l8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def near(got, want, terms, dtype):
    """|got - want| within a rounding to dtype of either and the sum's own error."""
    return bool(((got.double() - want).abs() <= ULP[dtype] * want.abs() + terms + 1e-7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [(1, 32, 8), (128, 32, 192), (127, 64, 184), (129, 96, 200), (300, 160, 40), (515, 384, 392)])
def test_linear(M, K, N, dtype):
    print("CASE linear_tiles", M, K, N, dtype, flush=True)
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, K, generator=g).to(dtype).to(DEV), (torch.randn(N, K, generator=g) / K ** 0.5).to(dtype).to(DEV)
    b, r = torch.randn(N, generator=g).to(dtype).to(DEV), torch.randn(M, N, generator=g).to(dtype).to(DEV)
    z = x.double() @ w.double().t()
    terms = (K + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs() + r.double().abs())
    assert near(linear_tiles_hip(x, w), z, terms, dtype)
    assert near(linear_tiles_hip(x, w, b, r), z + b.double() + r.double(), terms, dtype)
    got, pre = linear_tiles_hip(x, w, b, gelu=True), linear_tiles_hip(x, w, b)
    assert near(pre, z + b.double(), terms, dtype)
    assert near(got, F.gelu(pre.double()), 2e-7, dtype)               # GELU of what the product alone leaves


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [(128 * 1024, 32, 8), (128 * 1024 + 1, 32, 8), (128 * 1024 + 127, 64, 16), (128 * 512 + 5, 96, 200), (43 * 128 - 3, 160, 192 * 24 - 8)])
def test_linear_of_many_tiles(M, K, N, dtype):
    """The GELU on both sides of 1024 workgroups, from where on the ring has two buffers: one step and several, edges in both directions."""
    print("CASE linear_tiles many", M, K, N, dtype, flush=True)
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = torch.randn(M, K, generator=g, device=DEV).to(dtype), (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).to(dtype)
    b = torch.randn(N, generator=g, device=DEV).to(dtype)
    z = x.double() @ w.double().t() + b.double()
    terms = (K + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs())
    pre = linear_tiles_hip(x, w, b)
    assert near(pre, z, terms, dtype)
    assert near(linear_tiles_hip(x, w, b, gelu=True), F.gelu(pre.double()), 2e-7, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,W,C,N", [(1, 1, 1, 32, 8), (2, 2, 3, 32, 192), (3, 7, 9, 64, 200), (1, 16, 15, 96, 192), (2, 23, 1, 32, 40), (5, 14, 14, 192, 384)])
def test_convolution(B, H, W, C, N, dtype):
    print("CASE conv_tiles", B, H, W, C, N, dtype, flush=True)
    g = torch.Generator().manual_seed(H)
    x, w = torch.randn(B, H, W, C, generator=g).to(dtype).to(DEV), (torch.randn(N, C, 3, 3, generator=g) / (9 * C) ** 0.5).to(dtype).to(DEV)
    b = torch.randn(N, generator=g).to(dtype).to(DEV)
    conv = lambda x, w, b: F.conv2d(x.cpu().double().permute(0, 3, 1, 2), w.cpu().double(), b.cpu().double(), stride=2, padding=1).permute(0, 2, 3, 1).to(DEV)
    want, size = conv(x, w, b), conv(x.abs(), w.abs(), b.abs())
    for weight in (w, w.to(memory_format=torch.channels_last)):
        assert near(conv_tiles_hip(x, weight, b), want, (9 * C + 2) * 2.0 ** -24 * size, dtype)


def test_refused():
    x, w = torch.zeros(8, 48, device=DEV, dtype=torch.float16), torch.zeros(8, 48, device=DEV, dtype=torch.float16)
    for args in ((x, w), (x[:, :32].contiguous(), torch.zeros(6, 32, device=DEV, dtype=torch.float16)),
                 (torch.zeros(257, device=DEV, dtype=torch.float16)[1:].view(8, 32), w[:, :32].contiguous())):
        with pytest.raises(_lib.Ss2dError):
            linear_tiles_hip(*args)
    with pytest.raises(_lib.Ss2dError):
        linear_tiles_hip(x[:, :32].contiguous(), w[:, :32].contiguous(), None, torch.zeros(8, 8, device=DEV, dtype=torch.float16), gelu=True)
    with pytest.raises(_lib.Ss2dError):
        conv_tiles_hip(torch.zeros(1, 4, 4, 48, device=DEV, dtype=torch.float16), torch.zeros(8, 48, 3, 3, device=DEV, dtype=torch.float16))


def test_who_takes_them():
    mlp = Mlp(384, 1536, channel_first=False).to(DEV).bfloat16().eval()
    x = torch.randn(3136, 384, device=DEV).bfloat16()
    conv = nn.Conv2d(192, 384, 3, stride=2, padding=1).to(DEV).bfloat16()
    m = torch.randn(16, 28, 28, 192, device=DEV).bfloat16().permute(0, 3, 1, 2)
    takes = lambda t=x: linear_tiles_fusable(t, mlp.fc1, mlp.act)
    convolves = lambda t=m: conv_tiles_fusable(t, conv)
    assert not takes()                                               # autograd
    with torch.no_grad():
        assert takes() and not takes(x[:3135]) and not takes(x.float()) and not takes(x.t().contiguous().t())
        assert convolves() and not convolves(m[:15]) and not convolves(m.contiguous()) and not convolves(m.float())
        for layer in (mlp.fc1, mlp.act):
            handle = layer.register_forward_hook(lambda *a: None)
            assert not takes()
            handle.remove()
        with torch.autocast("cuda", torch.float16):
            assert not takes() and not convolves()
        with torch.overrides.BaseTorchFunctionMode():
            assert not takes() and not convolves()
        conv._conv_forward = conv._conv_forward
        assert not convolves()
        mlp.act.approximate = "tanh"
        assert not takes()
    # both sides of the lines
    assert linear_tiles_pays(12544, 2048, 512, True) and not linear_tiles_pays(6272, 2048, 512, True) and not linear_tiles_pays(25088, 3072, 768, True)
    assert linear_tiles_pays(25088, 384, 384, False) and not linear_tiles_pays(12544, 384, 384, False) and not linear_tiles_pays(50176, 256, 256, False)
    assert conv_tiles_pays(3136, 192) and not conv_tiles_pays(3135, 192) and conv_tiles_pays(6272, 96) and not conv_tiles_pays(6271, 96)


def test_model_no_further_from_float64(monkeypatch):
    """Through the kernels and through the library's operators: logits as far from the same model in float32."""
    torch.manual_seed(0)
    model = vmamba_tiny_s1l8(channel_first=False).to(DEV).eval()
    x = torch.randn(32, 3, 224, 224, device=DEV).bfloat16()
    with torch.no_grad():
        half = vmamba_tiny_s1l8(channel_first=False).to(DEV).bfloat16().eval()
        half.load_state_dict(model.state_dict())
        model.load_state_dict(half.state_dict())
        taken = []
        monkeypatch.setattr(vssm, "conv_tiles_hip", lambda *a: taken.append(0) or conv_tiles_hip(*a))
        monkeypatch.setattr(vssm, "linear_tiles_hip", lambda *a, **k: taken.append(1) or linear_tiles_hip(*a, **k))
        got, want = half(x).double(), model(x.float()).double()
        assert taken.count(0) == 2 and taken.count(1) == 8
        monkeypatch.setattr(vssm, "conv_tiles_fusable", lambda *a: False)
        monkeypatch.setattr(vssm, "linear_tiles_fusable", lambda *a: False)
        before = half(x).double()
    error = lambda y: ((y - want).norm() / want.norm()).item()
    assert error(got) <= 1.1 * error(before)


@pytest.mark.parametrize("lo,hi", [(-8, -4), (-4, -3), (-3, -2), (-2, -1), (-1, 0), (0, 1), (1, 2), (2, 4), (4, 65504)])
def test_fp16_gelu_rounds_no_worse_than_erff(lo, hi):
    """Every fp16 argument in (lo, hi], as a bias behind a product of zeros: no more results than the library's erff form gives are another
    neighbour than the exact value's -- one of the 15 360 on either side of 0, where x = 0.0013 has an exact value 4.2e-8 of itself from the middle of two
    neighbours, less than a rounding in fp32 --, and none is further off than its furthest or 0.502 of a unit."""
    from vmamba_amd.linear import linear_rows_hip
    every = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.float16)
    every = every[every.isfinite() & (every > lo) & (every <= hi)]
    n = every.numel() // 8 * 8
    x = every[:n].to(DEV)
    exact = F.gelu(x.double())
    nearest = exact.to(torch.float16)
    unit = (torch.nextafter(nearest.abs(), torch.full_like(nearest, float("inf"))) - nearest.abs()).double()
    zero, weight = torch.zeros(8, 32, device=DEV, dtype=torch.float16), torch.zeros(n, 32, device=DEV, dtype=torch.float16)
    lib = F.gelu(x)
    off = lambda y: ((y.double() - exact).abs() / unit).max().item()
    for kernel in (linear_tiles_hip, linear_rows_hip):
        got = kernel(zero, weight, x, gelu=True)[0]
        print("fp16 gelu", lo, hi, n, "other neighbours %d / %d, furthest %.3f / %.3f" % ((got != nearest).sum(), (lib != nearest).sum(), off(got), off(lib)), flush=True)
        assert (got != nearest).sum() <= (lib != nearest).sum() + (n > 15000 and abs(lo + hi) == 1) and off(got) <= max(off(lib), 0.502)
