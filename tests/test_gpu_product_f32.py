"""ss2d_product_f32 against float64: the edges of its tiles, steps and shares, both ways either operand may be stored, and what stands
behind the sum; MlpF32 and its derivatives.

An output is a sum of six products a term, added in fp32: it stays within 6 K 2^-24 of the sum of the terms' magnitudes whatever the order
(the terms left out and the rest of a value behind its third part are below 2^-25 of a term)."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from vmamba_amd import _lib
from vmamba_amd.linear import PRODUCT_GELU, PRODUCT_GELU_GRAD, LinearDw, MlpF32, mlp_f32_pays, product_f32_hip, product_pays
from vmamba_amd.vssm import Mlp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def make(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    a, b = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    return (a * torch.exp2(torch.randint(-20, 20, (M, 1), generator=g).float())).to(DEV), b.to(DEV)


def stored(t, by_columns):
    return t.t().contiguous() if by_columns else t


@pytest.mark.parametrize("a_cols,b_cols", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(4, 4, 4), (128, 64, 32), (124, 68, 36), (132, 132, 60), (260, 60, 512), (64, 192, 4100), (1000, 1028, 100), (12544, 128, 96)])
def test_product(M, N, K, a_cols, b_cols):
    print("CASE product_f32", M, N, K, a_cols, b_cols, flush=True)
    a, b = make(M, N, K, M + K)
    got = product_f32_hip(stored(a, a_cols), stored(b, b_cols), a_cols, b_cols).double()
    want, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    assert bool(((got - want).abs() <= 6 * K * 2.0 ** -24 * size).all())
    lib = (a @ b.t()).double()
    scale = want.norm(dim=1, keepdim=True)
    assert ((got - want) / scale).norm().item() <= 1.1 * ((lib - want) / scale).norm().item() + 1e-7


@pytest.mark.parametrize("M,N,K", [(300, 132, 64), (200, 68, 2048)])       # one share, and several added by the second kernel
def test_what_stands_behind_the_sum(M, N, K):
    print("CASE product_f32 epilogue", M, N, K, flush=True)
    assert (_lib.lib().ss2d_product_f32_workspace_bytes(M, N, K, 0, 0) > 0) == (K > 1000)
    g = torch.Generator().manual_seed(K)
    a, b = torch.randn(M, K, generator=g).to(DEV), torch.randn(N, K, generator=g).to(DEV) / K ** 0.5
    bias, other = torch.randn(N, generator=g).to(DEV), torch.randn(M, N, generator=g).to(DEV)
    z = a.double() @ b.double().t()
    close = lambda got, want: torch.allclose(got.double(), want, rtol=1e-5, atol=1e-5)        # sums of unit size, 2^-24 a rounding
    assert close(product_f32_hip(a, b, bias=bias, other=other), z + bias.double() + other.double())
    pre, act = product_f32_hip(a, b, bias=bias, mode=PRODUCT_GELU)
    assert close(pre, z + bias.double()) and close(act, F.gelu(z + bias.double()))
    x = other.double().requires_grad_()
    slope = torch.autograd.grad(F.gelu(x).sum(), x)[0]
    assert close(product_f32_hip(a, b, other=other, mode=PRODUCT_GELU_GRAD), z * slope)


@pytest.mark.parametrize("a_cols,b_cols", [(False, False), (True, True)])
def test_infinities_and_nan(a_cols, b_cols):
    """The same outputs are infinite and NaN as in the library's product, and values near fp32's largest, which round beyond bf16's, count."""
    a, b = make(300, 132, 384, 3)
    a, b = a / a.abs().amax(1, keepdim=True), b * 0.01
    a[5, 7], a[9, 3], a[200, 1], a[201, 1], b[77, 11] = float("inf"), float("nan"), 3.4e38, -3.402e38, -float("inf")
    got, want = product_f32_hip(stored(a, a_cols), stored(b, b_cols), a_cols, b_cols), a @ b.t()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())
    ok = want.isfinite()
    assert torch.allclose(got[ok], want[ok], rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("a_cols,b_cols", [(False, False), (False, True), (True, True)])
@pytest.mark.parametrize("down,M,N,K", [((100, 0), 132, 68, 96), ((116, 0), 132, 68, 96), ((0, 116), 132, 68, 96), ((58, 58), 132, 68, 96), ((120, -100), 64, 64, 4096)])
def test_small_operands_lose_nothing(down, M, N, K, a_cols, b_cols):
    """Operands times powers of two give the same digits, as long as the results are fp32 normals (a share's of a long sum too)."""
    print("CASE product_f32 small", down, M, N, K, a_cols, b_cols, flush=True)
    g = torch.Generator().manual_seed(K)
    a, b = torch.randn(M, K, generator=g).to(DEV) * 2.0 ** -down[0], torch.randn(N, K, generator=g).to(DEV) * 2.0 ** -down[1]      # (some subnormal)
    small = product_f32_hip(stored(a, a_cols), stored(b, b_cols), a_cols, b_cols)
    one = product_f32_hip(stored(a * 2.0 ** down[0], a_cols), stored(b * 2.0 ** down[1], b_cols), a_cols, b_cols)
    normal = one.abs() * 2.0 ** -sum(down) > 2.0 ** -125
    assert normal.float().mean() > 0.99 and torch.equal((small * 2.0 ** sum(down))[normal], one[normal])


def test_subnormal_operands():
    """Subnormal fp32 values, exact as integers of 2^-149, against float64: an error of a product in fp32."""
    g = torch.Generator().manual_seed(0)
    a = (torch.randint(-2 ** 23, 2 ** 23, (132, 64), generator=g).double() * 2.0 ** -149).float().to(DEV)
    b = torch.randn(68, 64, generator=g).to(DEV) * 2.0 ** 60
    got, want = product_f32_hip(a, b).double(), a.double() @ b.double().t()
    assert bool((a.abs() < 2.0 ** -126).all()) and ((got - want).norm() / want.norm()).item() < 2.0 ** -22


def test_refused():
    a = torch.zeros(8, 8, device=DEV)
    with pytest.raises(ValueError):
        product_f32_hip(a, a[:, :4])
    with pytest.raises(ValueError):
        product_f32_hip(a, a.half())
    for args in ((torch.zeros(8, 6, device=DEV), torch.zeros(8, 6, device=DEV)), (a, torch.zeros(6, 8, device=DEV)),
                 (torch.zeros(65, device=DEV)[1:].view(8, 8), a)):
        with pytest.raises(_lib.Ss2dError):
            product_f32_hip(*args)


@pytest.mark.parametrize("bias", [True, False])
def test_mlp_autograd(bias):
    """Both derivatives against float64: relative errors of a few hundred roundings of 2^-24."""
    torch.manual_seed(0)
    mlp = Mlp(96, 384, channel_first=False).to(DEV)
    if not bias:
        mlp.fc1.bias = mlp.fc2.bias = None
    x = torch.randn(7, 56, 56, 96, device=DEV, requires_grad=True)
    dy = torch.randn_like(x)
    assert mlp_f32_pays(x, mlp.fc1, mlp.act, mlp.fc2)
    params = [x] + list(mlp.parameters())
    exact = [t.detach().double().requires_grad_() for t in params]
    e = iter(exact[1:])
    xd = exact[0]
    w1, b1, w2, b2 = next(e), next(e) if bias else None, next(e), next(e) if bias else None
    y, want_y = mlp(x), F.linear(F.gelu(F.linear(xd, w1, b1)), w2, b2)
    assert y.grad_fn.name().startswith("MlpF32")
    got, want = torch.autograd.grad(y, params, dy), torch.autograd.grad(want_y, exact, dy.double(), create_graph=True)
    for g, w in zip((y,) + got, (want_y,) + want):
        assert ((g.double() - w).norm() / w.norm()).item() < 2e-6
    # a second backward, through the torch operators
    dx = torch.autograd.grad(mlp(x), x, dy, create_graph=True)[0]
    got, want = torch.autograd.grad(dx.square().sum(), params[:2]), torch.autograd.grad(want[0].square().sum(), exact[:2])
    for g, w in zip(got, want):
        assert ((g.double() - w).norm() / w.norm()).item() < 1e-5


def test_who_is_left_to_the_operators():
    mlp = Mlp(96, 384, channel_first=False).to(DEV)
    x = torch.randn(22000, 96, device=DEV)
    takes = lambda t=x: mlp_f32_pays(t, mlp.fc1, mlp.act, mlp.fc2)
    assert takes() and not takes(x[:21000]) and not takes(x.half())
    with torch.no_grad():
        assert not takes()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not takes()
    seen = []
    handle = mlp.act.register_forward_hook(lambda *a: seen.append(1))
    mlp(x)
    assert seen and not takes()
    handle.remove()
    with torch.autograd.forward_ad.dual_level():
        assert not takes()
    assert torch.func.grad(lambda t: mlp(t).sum())(x).shape == x.shape
    mlp.act.approximate = "tanh"
    assert not takes()
    mlp.act.approximate = "none"
    mlp.fc1.weight = nn.Parameter(torch.randn(96, 384, device=DEV).t())
    assert not takes()
    # both sides of the line
    assert product_pays(12544, 1536, 384) and not product_pays(784, 1536, 384) and product_pays(1536, 384, 4096, True) and not product_pays(1536, 384, 4095, True)


def test_projection_with_residual():
    layer = nn.Linear(768, 512, bias=False).to(DEV)
    x, r = torch.randn(7000, 768, device=DEV, requires_grad=True), torch.randn(7000, 512, device=DEV)
    dy = torch.randn(7000, 512, device=DEV)
    y = LinearDw.apply(x, layer.weight, r)
    got = (y,) + torch.autograd.grad(y, (x, layer.weight), dy)
    w, xd = layer.weight.double(), x.double()
    for g, want in zip(got, (r.double() + xd @ w.t(), dy.double() @ w, dy.double().t() @ xd)):
        assert ((g.double() - want).norm() / want.norm()).item() < 2e-6


def test_projections_of_the_core_in_training():
    """x_proj and dt_proj of forward_core on the kernels, their gradients against the operators they stand for (sums of 96 and 21 952 terms)."""
    from vmamba_amd import ss2d
    torch.manual_seed(0)
    op = ss2d.SS2D(d_model=96, channel_first=False).to(DEV)
    x = torch.randn(28, 96, 28, 28, device=DEV, requires_grad=True)
    dy = torch.randn(28, 28, 28, 96, device=DEV)
    wanted = [x] + [p for n, p in op.named_parameters() if n.split(".")[0] in ("x_proj_weight", "dt_projs_weight", "A_logs", "Ds", "dt_projs_bias")]
    def run():
        y = op.forward_core(x)
        return (y.detach(),) + torch.autograd.grad(y, wanted, dy)
    calls, apply = [], ss2d.XProjF32.apply
    ss2d.XProjF32.apply = lambda *a: calls.append(1) or apply(*a)
    try:
        got = run()
    finally:
        ss2d.XProjF32.apply = apply
    assert calls
    takes, ss2d.projections_train = ss2d.projections_train, lambda *a: False
    try:
        want = run()
    finally:
        ss2d.projections_train = takes
    for g, w in zip(got, want):
        assert ((g - w).norm() / w.norm()).item() < 1e-5


def routes(x):
    """(B, D, H, W) -> (B, 4, D, L) in the directions' scan orders."""
    rows, cols = x.flatten(2), x.transpose(2, 3).flatten(2)
    return torch.stack([rows, cols, rows.flip(-1), cols.flip(-1)], 1)


@pytest.mark.parametrize("what", ["x_proj", "dt_proj", "transpose"])
def test_second_derivatives_of_the_projections(what):
    """Both derivatives of the cubes' sum, every input, against the same expression in float64: sums of up to 1000 terms in fp32."""
    from vmamba_amd.core import DtProjF32, XProjF32
    from vmamba_amd.csm import TransposeBCL
    g = torch.Generator().manual_seed(3)
    make = lambda *s: torch.randn(*s, generator=g).to(DEV).requires_grad_()
    if what == "x_proj":
        wanted = [make(2, 32, 6, 9), make(4, 5, 32)]
        call, exact = XProjF32.apply, lambda x, w: torch.matmul(w, routes(x))
    elif what == "dt_proj":
        wanted = [make(4, 6, 200), make(4, 24, 6)]
        call, exact = DtProjF32.apply, lambda rows, w: torch.matmul(w, rows)
    else:
        wanted = [make(3, 20, 33)]
        call, exact = TransposeBCL.apply, lambda x: x.transpose(1, 2)

    def derivatives(f, inputs):
        y = f(*inputs)
        first = torch.autograd.grad((y ** 3).sum(), inputs, create_graph=True)
        return [y.detach()] + [t.detach() for t in first] + list(torch.autograd.grad(sum((t ** 2).sum() for t in first), inputs))
    for got, want in zip(derivatives(call, wanted), derivatives(exact, [t.detach().double().requires_grad_() for t in wanted])):
        assert got.shape == want.shape and ((got.double() - want).norm() / want.norm()).item() < 1e-5


GELU_RANGES = [(-0.01, 0.01), (-0.5, 0.0), (0.0, 0.5), (-1.0, -0.5), (0.5, 1.0), (-1.5, -1.0), (1.0, 1.5), (-2.0, -1.5), (1.5, 2.0), (-3.0, -2.0), (2.0, 3.0),
               (-4.0, -3.0), (3.0, 5.0), (-8.0, -4.0)]


@pytest.mark.parametrize("lo,hi", GELU_RANGES + [(None, None)])
def test_gelu_and_its_derivative_are_no_further_from_float64_than_erff(lo, hi):
    """GELU and GELU' behind a product that leaves x as it is, against the library's erff form by range (None: a normal x).  Either is a rounding
    or two of Phi and of the result; 200 000 samples give the rms to half a per cent, their largest error to the last of a few units in the last place."""
    g = torch.Generator().manual_seed(7)
    x = torch.randn(800 * 256, generator=g) if lo is None else torch.rand(800 * 256, generator=g) * (hi - lo) + lo
    x = x.to(DEV)
    zero = torch.zeros(4, 4, device=DEV)
    pre, act = product_f32_hip(zero, torch.zeros(x.numel(), 4, device=DEV), bias=x, mode=PRODUCT_GELU)
    one = torch.zeros(800, 4, device=DEV)
    one[:, 0] = 1.0
    slope = product_f32_hip(one, one[:256].contiguous(), other=x.view(800, 256), mode=PRODUCT_GELU_GRAD)
    assert torch.equal(pre[0], x)
    xd = x.double().requires_grad_()
    y = F.gelu(xd)
    dy = torch.autograd.grad(y.sum(), xd)[0]
    lib = torch.ops.aten.gelu_backward(torch.ones_like(x), x)
    for what, got, erff, want in (("gelu", act[0], F.gelu(x), y.detach()), ("slope", slope.view(-1), lib, dy)):
        err, ref = (got.double() - want).abs(), (erff.double() - want).abs()
        print(what, lo, hi, "rms %.2e / %.2e, largest %.2e / %.2e" % (err.square().mean().sqrt(), ref.square().mean().sqrt(), err.max(), ref.max()), flush=True)
        assert err.square().mean().sqrt() <= 1.02 * ref.square().mean().sqrt() and err.max() <= 1.1 * ref.max()
