"""ss2d_layer_norm_bwd_f32 and ss2d_column_sums_f32 against float64: rows in every lane group, rows and shares that end early.

dx is a handful of fp32 operations on values of unit size behind sums of C terms, dw and db are sums over the rows: (C + 16) 2^-24 and
(rows + C + 16) 2^-24 of their terms' magnitudes bound them whatever the order."""
import pytest
import torch
import torch.nn.functional as F
from torch.utils._python_dispatch import TorchDispatchMode

from vmamba_amd.linear import LinearDw
from vmamba_amd.norm import LayerNorm, LayerNormF32, column_sums, layer_norm_trains
from vmamba_amd.ss2d import SS2D
from vmamba_amd.vssm import Mlp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("affine", [True, False])
@pytest.mark.parametrize("rows,C", [(1, 4), (33, 64), (1000, 60), (257, 68), (5000, 96), (2049, 128), (515, 132), (4100, 256), (300, 260), (12544, 384), (700, 516),
                                    (129, 768), (31, 1024)])
def test_backward(rows, C, affine):
    print("CASE ln_bwd", rows, C, affine, flush=True)
    g = torch.Generator().manual_seed(C)
    x, dy = (torch.randn(rows, C, generator=g) * 2 + 0.5).to(DEV), torch.randn(rows, C, generator=g).to(DEV)
    w, b = (torch.randn(C, generator=g).to(DEV), torch.randn(C, generator=g).to(DEV)) if affine else (None, None)
    wanted = [t.requires_grad_() for t in (x, w, b) if t is not None]
    y = LayerNormF32.apply(x, w, b, 1e-5)
    got = torch.autograd.grad(y, wanted, dy)
    exact = [t.detach().double().requires_grad_() for t in wanted]
    yd = F.layer_norm(exact[0], (C,), *(exact[1:] if affine else (None, None)), 1e-5)
    want = torch.autograd.grad(yd, exact, dy.double(), create_graph=True)
    assert torch.allclose(y.double(), yd, rtol=1e-5, atol=1e-4)
    xd = exact[0].detach()
    rstd = (xd.var(-1, unbiased=False, keepdim=True) + 1e-5).rsqrt()
    size = rstd * 8 * (dy.double() * (exact[1].detach() if affine else 1)).abs().amax(-1, keepdim=True) * (1 + ((xd - xd.mean(-1, keepdim=True)) * rstd).abs())
    assert bool(((got[0].double() - want[0]).abs() <= (C + 16) * 2.0 ** -24 * size + 1e-12).all())
    for q, terms in ((1, (dy.double() * (1 + ((xd - xd.mean(-1, keepdim=True)) * rstd).abs())).abs()), (2, dy.double().abs())):
        if affine:
            assert bool(((got[q].double() - want[q]).abs() <= (rows + C + 16) * 2.0 ** -24 * terms.sum(0) * 2 + 1e-12).all())
            assert ((got[q].double() - want[q]).norm() / want[q].norm().clamp(min=1e-30)).item() < 1e-5 or rows * C < 100
    # a second backward, through the torch operators
    if rows <= 1000 and C > 4:
        first = torch.autograd.grad(LayerNormF32.apply(x, w, b, 1e-5), x, dy, create_graph=True)[0]
        second = torch.autograd.grad(first.square().sum(), x)[0]
        ref = torch.autograd.grad(want[0].square().sum(), exact[0])[0]
        assert ((second.double() - ref).norm() / ref.norm()).item() < 1e-4


@pytest.mark.parametrize("rows,N", [(1, 4), (7, 260), (1000, 1536), (50000, 48), (12544, 384)])
def test_column_sums(rows, N):
    x = torch.randn(rows, N, device=DEV)
    with torch.no_grad():
        got = column_sums(x)
    assert bool(((got.double() - x.double().sum(0)).abs() <= rows * 2.0 ** -24 * x.double().abs().sum(0)).all())


def test_who_takes_it():
    norm, x = LayerNorm(96).to(DEV), torch.randn(22000, 96, device=DEV, requires_grad=True)
    takes = lambda t=x, n=norm: layer_norm_trains(t, n.normalized_shape, n.weight, n.bias)
    assert takes() and not takes(x.half()) and not takes(x[:21000]) and not takes(x[:, :48]) and norm(x).grad_fn.name().startswith("LayerNormF32")
    assert not takes(n=LayerNorm(96).to(DEV).half()) and not takes(torch.randn(2100, 1028, device=DEV), LayerNorm(1028).to(DEV))
    with torch.autocast("cuda", torch.bfloat16):
        assert not takes()
    with torch.autograd.forward_ad.dual_level():
        assert not takes()
    assert torch.func.grad(lambda t: norm(t).square().sum())(x).shape == x.shape
    # a non-contiguous gradient and views between 16-byte boundaries
    off = lambda: torch.randn(22000 * 96 + 1, device=DEV)[1:].view(22000, 96)
    shifted = off().requires_grad_()
    for t, dy in ((x, torch.randn(96, 22000, device=DEV).t()), (shifted, off())):
        got, want = (torch.autograd.grad(f(t), t, dy)[0] for f in (norm, lambda t: F.layer_norm(t, (96,), norm.weight, norm.bias)))
        assert torch.allclose(got, want, rtol=1e-4, atol=1e-5)


def test_out_norm_of_a_map():
    """out_norm in training: the map transposed by the package's kernel, both ways."""
    torch.manual_seed(0)
    op = SS2D(d_model=64, channel_first=False).to(DEV)
    with torch.no_grad():
        op.out_norm.weight.uniform_(0.5, 1.5)
    y = torch.randn(600, 64, 9, 7, device=DEV, requires_grad=True)
    dy = torch.randn(600, 9, 7, 64, device=DEV)
    got = op.finish_core(y.view(600, 64, 63), 600, 64, 9, 7, torch.float32)
    assert got.grad_fn.name().startswith("LayerNormF32")
    want = F.layer_norm(y.permute(0, 2, 3, 1), (64,), op.out_norm.weight, op.out_norm.bias)
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-5)
    for a, b in zip(torch.autograd.grad(got, [y, op.out_norm.weight], dy), torch.autograd.grad(want, [y, op.out_norm.weight], dy)):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-5 * max(1.0, b.abs().max().item()))


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.calls = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.calls.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("what", ["norm", "out_norm", "mlp", "linear"])
def test_gradients_whose_memory_is_not_theirs(what):
    """A batch of gradients (is_grads_batched, a vectorised jacobian) and a mode around the backward alone: both go through torch's operators,
    as they do where those stand in the forward, and give the gradients of the separate calls (sums of up to 35 000 terms in fp32)."""
    torch.manual_seed(0)
    if what == "out_norm":
        op = SS2D(d_model=64, channel_first=False).to(DEV)
        x = torch.randn(600, 64, 9, 7, device=DEV, requires_grad=True)
        y, wanted = op.finish_core(x.view(600, 64, 63), 600, 64, 9, 7, torch.float32), [x, op.out_norm.weight, op.out_norm.bias]
    else:
        x = torch.randn(22000, 96, device=DEV, requires_grad=True)
        if what == "linear":
            layer = torch.nn.Linear(96, 96, bias=False).to(DEV)
            y, wanted = LinearDw.apply(x, layer.weight, None), [x, layer.weight]
        else:
            layer = LayerNorm(96).to(DEV) if what == "norm" else Mlp(96, 384, channel_first=False).to(DEV)
            y, wanted = layer(x), [x] + list(layer.parameters())
    assert y.grad_fn.name().split("Backward")[0] in ("LayerNormF32", "MlpF32", "LinearDw")
    dys = torch.randn(3, *y.shape, device=DEV)
    singly = [torch.autograd.grad(y, wanted, dy, retain_graph=True) for dy in dys]
    near = lambda a, b: ((a - b).norm() / b.norm()).item() < 1e-5
    batched = torch.autograd.grad(y, wanted, dys, is_grads_batched=True, retain_graph=True)
    assert all(near(many, torch.stack(few)) for many, few in zip(batched, zip(*singly)))
    with Seen() as mode:
        seen = torch.autograd.grad(y, wanted, dys[0])
    assert all(near(a, b) for a, b in zip(seen, singly[0]))
    assert any(("mm" if what in ("mlp", "linear") else "rsqrt") in call for call in mode.calls)
