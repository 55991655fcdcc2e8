"""A block of few positions as one call (ss2d_block_fwd): the bits of the separate calls, and who is left to them."""
import pytest
import torch
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from vmamba_amd import vssm
from vmamba_amd.block import vss_block_hip
from vmamba_amd.conv import dwconv3x3_silu_hip
from vmamba_amd.linear import linear_cf_ln_hip, linear_cl_hip, linear_rows_hip
from vmamba_amd.norm import LayerNorm, add_layer_norm_hip
from vmamba_amd.vssm import Mlp, VSSBlock, VSSM

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def unlike_norms(block, biases=True):
    """Norms that cannot stand in for one another, nor be applied twice: weights, biases and eps of their own."""
    with torch.no_grad():
        for norm, eps in ((block.norm, 1e-5), (block.norm2, 3e-2), (block.op.out_norm, 4e-1)):
            norm.eps = eps
            norm.weight.uniform_(0.5, 1.5)
            norm.bias.uniform_(-0.5, 0.5)
            if not biases:
                norm.bias = None
    return block


def make(dim, B, H, W, dtype, norm_biases=True, **kwargs):
    torch.manual_seed(dim + H)
    block = VSSBlock(dim, channel_first=False, **kwargs).to(DEV, dtype).eval()
    return unlike_norms(block, norm_biases), torch.randn(B, H, W, dim, device=DEV, dtype=dtype)


def one_by_one(block, x, residual=None):
    """What the call gives without the MLP -- x + op(norm(x)), or residual + op(x) with x normalised already -- from its kernels."""
    op, norm = block.op, block.norm
    ln = (norm.weight, norm.bias, norm.eps) if residual is None else ()
    narrow, M = x.shape[-1] == op.d_inner == 96, x.numel() // x.shape[-1]
    h = (linear_cl_hip if narrow and M > 24576 else linear_rows_hip)(x, op.in_proj.weight, op.in_proj.bias, None, *ln)
    h = dwconv3x3_silu_hip(h, op.conv2d.weight, op.conv2d.bias, in_channel_last=True, apply_silu=True)
    add, out = x if residual is None else residual, op.out_proj
    if narrow and x.shape[1] * x.shape[2] % 32 == 0:
        y = op._forward_core_native(h, False)
        return linear_cf_ln_hip(y, op.out_norm.weight, op.out_norm.bias, op.out_norm.eps, out.weight, out.bias, add).view(x.shape)
    return linear_rows_hip(op.forward_core(h), out.weight, out.bias, add)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("dim,B,H,W,kwargs", [
    (96, 1, 56, 56, {}), (96, 1, 14, 14, {}), (192, 2, 28, 28, {}), (384, 1, 14, 14, {}), (384, 2, 10, 12, {}), (768, 1, 7, 7, {}), (48, 3, 8, 8, {}),
    (384, 8, 14, 14, {}), (768, 8, 7, 7, {}), (96, 8, 56, 56, {}), (192, 8, 28, 28, {}), (192, 1, 12, 12, dict(ssm_ratio=2.0, mlp_ratio=2.0)), (96, 1, 16, 16, dict(bias=True, conv_bias=True)),
    (96, 1, 14, 14, dict(norm_biases=False)), (384, 1, 14, 14, dict(norm_biases=False)), (384, 8, 14, 14, dict(bias=True, norm_biases=False))])
def test_same_bits(dim, B, H, W, kwargs, dtype, monkeypatch):
    print("CASE vss_block", dim, B, H, W, kwargs, dtype, flush=True)
    block, x = make(dim, B, H, W, dtype, **kwargs)
    kept = x.clone()
    with torch.no_grad():
        assert vss_block_hip(block, Mlp, x) is not None
        got = block(x)
        monkeypatch.setattr(vssm, "vss_block_hip", lambda *a: None)
        want = block(x)
        native, whole = vss_block_hip(block, Mlp, x)
        if not whole:
            assert torch.equal(native, one_by_one(block, x))
        normalised, stream = torch.randn_like(x), torch.randn_like(x)
        beside = vss_block_hip(block, Mlp, normalised, stream)
        if not whole:
            assert torch.equal(beside[0], one_by_one(block, normalised, stream))
        else:
            s = one_by_one(block, normalised, stream)
            assert torch.equal(beside[0], block.mlp(s, residual=s, pre_norm=block.norm2))
    assert torch.equal(x, kept) and got.isfinite().all()
    if whole or dim <= 192:
        assert torch.equal(got, want)
    else:                      # out_proj's sum and the MLP are the library's on the other side: 16 u, as any two such blocks
        u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= 16 * u


@pytest.mark.parametrize("B", [6, 8, 12])
def test_projections_of_many_positions(B):
    """22 320, 29 760 and 44 640 positions of width 96, their maps no multiple of 32: either side of in_proj's line, out_proj's kernel."""
    block, x = make(96, B, 60, 62, torch.bfloat16)
    with torch.no_grad():
        got, whole = vss_block_hip(block, Mlp, x)
        assert not whole and torch.equal(got, one_by_one(block, x))


@pytest.mark.parametrize("dim,B,side", [(384, 8, 14), (768, 6, 7)])
def test_blocks_with_the_mlp_left_to_the_library(dim, B, side, monkeypatch):
    """The first block leaves its MLP's sum to the second's LayerNorm, whose result the call takes beside the residual stream: the
    bits of the kernels and the library's MLPs one by one."""
    torch.manual_seed(dim)
    stage = vssm.BlockSequence(*[VSSBlock(dim, channel_first=False) for _ in range(3)]).to(DEV, torch.bfloat16).eval()
    for block in stage:
        unlike_norms(block)
    x = torch.randn(B, side, side, dim, device=DEV, dtype=torch.bfloat16)
    calls = []
    with torch.no_grad():
        monkeypatch.setattr(vssm, "vss_block_hip", lambda *a: calls.append(vss_block_hip(*a)) or calls[-1])
        got = stage(x)
        assert len(calls) == 3 and all(c is not None and not c[1] for c in calls)
        stream, term = x, None
        for block in stage:
            if term is None:
                stream = one_by_one(block, stream)
            else:
                total, h = add_layer_norm_hip(term, stream, block.norm.weight, block.norm.bias, block.norm.eps)
                stream = one_by_one(block, h, total)
            term = block.mlp(block.norm2(stream))
    assert torch.equal(got, stream + term)


def test_who_is_left_to_the_modules():
    block, x = make(384, 1, 14, 14, torch.bfloat16)
    takes = lambda b=block, t=x: vss_block_hip(b, Mlp, t) is not None
    assert not takes()                                               # autograd
    with torch.no_grad():
        assert takes() and not takes(t=x.permute(0, 2, 1, 3)) and not takes(t=x.float()) and not takes(t=x[:, :10, :13].contiguous())
        assert not takes(t=x.expand(64, 14, 14, 384).contiguous())   # many positions
        for module in (block.op, block.op.conv2d, block.op.out_norm, block.mlp, block.mlp.fc2, block.norm):
            handle = module.register_forward_hook(lambda *a: None)
            assert not takes()
            handle.remove()
        block.op.finish_core = lambda *a: None
        assert not takes()
        del block.op.finish_core
        block.mlp.act.approximate = "tanh"
        assert not takes()
        block.mlp.act.approximate = "none"
        with torch.autocast("cuda", torch.bfloat16):
            assert not takes()
        assert takes()
        gated, _ = make(384, 1, 14, 14, torch.bfloat16, disable_z=False)
        assert not takes(gated)


@pytest.mark.parametrize("part", ["stages 1-3", "stage 4"])
def test_model_replayed_from_a_graph(part):
    """Three replays with the program's own work between them, each against the eager call.  Without the library's convolution between
    the last two stages: from 384 to 768 channels on 14 x 14 it differs from call to call, and asked for a deterministic one it also
    leaves that choice -- 6 ms a convolution -- in its database for every later program."""
    torch.manual_seed(1)
    if part == "stage 4":
        model = vssm.BlockSequence(*[VSSBlock(768, channel_first=False) for _ in range(2)])
        shape = 1, 7, 7, 768
    else:
        model, shape = VSSM(depths=(1, 1, 1), dims=(96, 192, 384), channel_first=False, num_classes=16), (1, 3, 224, 224)
    model = model.to(DEV, torch.bfloat16).eval()
    x = torch.randn(shape, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        for _ in range(2):
            model(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = model(x)
        for i in range(3):
            x.copy_(torch.randn(shape, device=DEV))
            want = model(x)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), i


class Seen(torch.Tensor):
    """A weight that sees the operators it is in, as quantised and sharded ones do."""
    functions = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.functions.append(getattr(func, "__name__", ""))
        with torch._C.DisableTorchFunctionSubclass():
            return func(*args, **(kwargs or {}))


def test_weights_of_other_kinds_are_left_to_torch():
    block, x = make(384, 1, 14, 14, torch.bfloat16)
    with torch.no_grad():
        want = block(x)
        own = block.op.in_proj._parameters
        own["weight"] = own["weight"].detach().as_subclass(Seen)
        assert vss_block_hip(block, Mlp, x) is None
        got = block(x)
        assert "linear" in Seen.functions
        # in_proj's sum is the library's on one side: 16 u, as in test_same_bits
        assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= 16 * 2.0 ** -8


@pytest.mark.parametrize("layer", ["fc1", "fc2"])
def test_bias_that_torch_broadcasts(layer):
    """One element in the place of a row: the kernels read a row."""
    block, x = make(384, 1, 14, 14, torch.bfloat16)
    mod = getattr(block.mlp, layer)
    with torch.no_grad():
        mod.bias = torch.nn.Parameter(torch.full((mod.out_features,), 0.5, device=DEV, dtype=torch.bfloat16))
        want = block(x)
        mod.bias = torch.nn.Parameter(torch.full((1,), 0.5, device=DEV, dtype=torch.bfloat16))
        assert vss_block_hip(block, Mlp, x) is None
        got = block(x)
    assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= 16 * 2.0 ** -8


class Functions(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(getattr(func, "__name__", ""))
        return func(*args, **(kwargs or {}))


class Operators(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(func.overloadpacket.__name__)
        return func(*args, **(kwargs or {}))


def test_modes_see_the_products_of_few_positions():
    """Flop counters and loggers see the library's calls at widths whose layers are plain torch ones; the mode behind torch.device does
    not look at them and changes nothing."""
    block, x = make(384, 1, 14, 14, torch.bfloat16)
    with torch.no_grad():
        want = block(x)
        with Functions() as functions:
            got = block(x)
        assert functions.names.count("linear") == 4 and "gelu" in functions.names
        with Operators() as operators:
            again = block(x)
        assert sum(name in ("mm", "addmm", "linear") for name in operators.names) >= 4 and "gelu" in operators.names
        assert torch.equal(got, again)
        with torch.device(DEV):
            assert vss_block_hip(block, Mlp, x) is not None and torch.equal(block(x), want)
    # in_proj, out_proj and the MLP are the library's on one side: 16 u, as in test_same_bits
    assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= 16 * 2.0 ** -8


@pytest.mark.parametrize("cls", [torch.nn.Linear, torch.nn.GELU, LayerNorm])
def test_forward_replaced_on_a_class(cls, monkeypatch):
    block, x = make(384, 1, 14, 14, torch.bfloat16)
    calls, forward = [], cls.forward
    monkeypatch.setattr(cls, "forward", lambda self, *a: calls.append(self) or forward(self, *a))
    with torch.no_grad():
        block(x)
    layers = {torch.nn.Linear: (block.op.in_proj, block.mlp.fc1, block.mlp.fc2), torch.nn.GELU: (block.mlp.act,),
              LayerNorm: (block.norm,)}[cls]                 # (norm2 is in the add's kernel, as at every number of positions)
    assert all(any(call is layer for call in calls) for layer in layers)


def test_forward_mode_derivatives_of_the_mlp():
    """A tangent of fc2's weight goes through torch's product."""
    mlp = Mlp(384, 1536, channel_first=False).to(DEV, torch.bfloat16).eval()
    norm = LayerNorm(384).to(DEV, torch.bfloat16)
    x = torch.randn(1, 14, 14, 384, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad(), forward_ad.dual_level():
        own = mlp.fc2._parameters
        own["weight"] = forward_ad.make_dual(own["weight"].detach(), torch.ones_like(own["weight"]))
        tangent = forward_ad.unpack_dual(mlp(x, pre_norm=norm)).tangent
    assert tangent is not None and tangent.isfinite().all() and tangent.any()


class FormerMlp(Mlp):
    """Knows neither a norm to ask for nor one to take."""

    def takes_norm(self, x):
        return False

    def forward(self, x):
        self.seen = x
        return super().forward(x)


def test_mlp_of_another_kind_is_called_with_the_normalised_rows():
    block, x = make(384, 1, 14, 14, torch.bfloat16)
    torch.nn.init.zeros_(block.norm2.bias)
    torch.nn.init.ones_(block.norm2.weight)
    with torch.no_grad():
        want = block(x)
        former = FormerMlp(384, 1536, channel_first=False).to(DEV, torch.bfloat16).eval()
        former.load_state_dict(block.mlp.state_dict())
        block.mlp = former
        got = block(x)
    # norm2's result: centred rows
    assert former.seen.shape == x.shape and former.seen.float().mean(-1).abs().max() < 1e-2
    assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= 16 * 2.0 ** -8          # as in test_same_bits


@pytest.mark.parametrize("how", ["hook", "class"])
def test_calls_of_the_mlp_are_the_same_with_few_positions(how, monkeypatch):
    """What sees or replaces the MLP's calls gets norm2's result and nothing else, as it does with many positions."""
    block, x = make(384, 1, 14, 14, torch.bfloat16)
    torch.nn.init.zeros_(block.norm2.bias)
    torch.nn.init.ones_(block.norm2.weight)
    seen, forward = [], Mlp.forward
    if how == "hook":
        block.mlp.register_forward_pre_hook(lambda module, args, kwargs: seen.append((args, kwargs)), with_kwargs=True)
    else:
        monkeypatch.setattr(Mlp, "forward", lambda self, *a, **k: seen.append((a, k)) or forward(self, *a, **k))
    with torch.no_grad():
        block(x)
        block(x.expand(32, 14, 14, 384).contiguous())
    assert [(len(args), list(kwargs)) for args, kwargs in seen] == [(1, []), (1, [])]
    assert all(args[0].float().mean(-1).abs().max() < 1e-2 for args, _ in seen)


def test_hooks_of_op_get_what_they_get_with_many_positions():
    block, x = make(384, 1, 14, 14, torch.bfloat16)
    seen = []
    block.op.register_forward_hook(lambda module, args, out: seen.append(type(out)))
    with torch.no_grad():
        block(x)
        block(x.expand(32, 14, 14, 384).contiguous())
    assert seen == [tuple, tuple]


def test_residual_of_another_kind_is_added_by_torch():
    block, x = make(384, 1, 14, 14, torch.bfloat16)
    Seen.functions.clear()
    with torch.no_grad():
        want, got = block.op(x, residual=x), block.op(x, residual=x.as_subclass(Seen))
    assert "reshape" in Seen.functions                               # into torch's addmm
    # two orders of one projection's sum, each rounded once
    assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= 2 * 2.0 ** -8


def block_f64(block, x):
    """The block in float64 from its 16-bit parameters and input (classification/models/vmamba.py:603-663, 1225-1229)."""
    op, mlp = block.op, block.mlp
    d = lambda t: None if t is None else t.double()
    ln = lambda n, t: F.layer_norm(t, n.normalized_shape, d(n.weight), d(n.bias), n.eps)
    x = x.double()
    B, H, W, _ = x.shape
    h = F.linear(ln(block.norm, x), d(op.in_proj.weight), d(op.in_proj.bias)).permute(0, 3, 1, 2)
    h = F.silu(F.conv2d(h, d(op.conv2d.weight), d(op.conv2d.bias), padding=1, groups=h.shape[1]))
    D, L, R = h.shape[1], H * W, op.dt_rank
    rows, cols = h.flatten(2), h.transpose(2, 3).flatten(2)
    u = torch.stack([rows, cols, rows.flip(-1), cols.flip(-1)])                              # (4, B, D, L)
    proj = torch.einsum("kcd,kbdl->kbcl", d(op.x_proj_weight), u)
    step = F.softplus(torch.einsum("kdr,kbrl->kbdl", d(op.dt_projs_weight), proj[:, :, :R]) + d(op.dt_projs_bias).view(4, 1, D, 1))
    decay, state = torch.exp(-step * d(op.A_logs).exp().view(4, 1, D, 1)), step * u * proj[:, :, R, None]
    for j in range(1, L):
        state[..., j] += decay[..., j] * state[..., j - 1]
    y = state * proj[:, :, R + 1, None] + d(op.Ds).view(4, 1, D, 1) * u
    down = (y[1] + y[3].flip(-1)).view(B, D, W, H).transpose(2, 3).flatten(2)
    y = (y[0] + y[2].flip(-1) + down).view(B, D, H, W).permute(0, 2, 3, 1)
    x = x + F.linear(ln(op.out_norm, y), d(op.out_proj.weight), d(op.out_proj.bias))
    return x + F.linear(F.gelu(F.linear(ln(block.norm2, x), d(mlp.fc1.weight), d(mlp.fc1.bias))), d(mlp.fc2.weight), d(mlp.fc2.bias))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("dim,B,H,W", [(96, 1, 28, 28), (192, 1, 28, 20), (384, 1, 14, 14), (384, 8, 14, 14), (768, 1, 7, 7)])
def test_no_further_from_float64_than_the_modules(dim, B, H, W, dtype):
    """The call rounds where the modules do, but for out_proj's and fc2's sums, which are rounded once with the residual instead of
    before and behind it: its error's 2-norm over the result is the modules' or less.  Both are sums over 37 632 independent roundings or
    more, whose ratio strays by about 1 / sqrt(37 632); 2 % is four times that."""
    print("CASE vss_block f64", dim, B, H, W, dtype, flush=True)
    block, x = make(dim, B, H, W, dtype)
    with torch.no_grad():
        assert vss_block_hip(block, Mlp, x) is not None
        got = block(x)
        with Functions():                       # products and GELU are the library's
            modules = block(x)
        want = block_f64(block, x)
    off = lambda t: ((t.double() - want).norm() / want.norm()).item()
    print("  off float64 by", off(got), "modules", off(modules), flush=True)
    assert off(got) <= 1.02 * off(modules)
