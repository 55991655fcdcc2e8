"""GPU parity of the projection of few positions (ss2d_linear_rows: LayerNorm -> Linear -> GELU -> + residual in one kernel)
against float64 math on operands rounded where the separate operators round, and of a block that takes it against the same block
on the separate operators.

Bounds: a result rounded once to 16 bits is off by u = 2^-8 (bf16) or 2^-11 (fp16) of itself at most; the LayerNorm's and the
GELU's own roundings can each fall the other way at a tie of the fp32 value, which moves one operand by 2 u of itself, and the fp32
sums of K products add K 2^-24 of their absolute values.  Compared in the 2-norm against the result's, 2 u covers all of it."""
import pytest
import torch
import torch.nn.functional as F

from vmamba_amd import _lib
from vmamba_amd.linear import linear_rows_fusable, linear_rows_hip
from vmamba_amd.norm import LayerNorm
from vmamba_amd.vssm import VSSBlock

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def make(M, K, N, dtype):
    g = torch.Generator().manual_seed(M * 7919 + K * 31 + N)
    r = lambda *s, scale=1.0, shift=0.0: (torch.randn(*s, generator=g) * scale + shift).to(dtype).to(DEV)
    return (r(M, K, scale=1.5, shift=0.3), r(N, K, scale=K ** -0.5), r(N, scale=0.5), r(M, N), r(K, scale=0.2, shift=1.0), r(K, scale=0.2))


def exact(x, w, b, res, gamma, beta, gelu):
    h = x.double()
    if gamma is not None:
        h = F.layer_norm(h, (h.shape[-1],), gamma.double(), None if beta is None else beta.double()).to(x.dtype).double()
    h = h @ w.double().t() + (0.0 if b is None else b.double())
    if gelu:
        h = F.gelu(h.to(x.dtype).double()).to(x.dtype).double()
    return h + (0.0 if res is None else res.double())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("M,K,N", [(1, 16, 8), (31, 48, 32), (32, 64, 40), (33, 192, 104), (49, 112, 96), (64, 208, 96), (49, 400, 72),
                                   (196, 384, 1536), (49, 768, 3072), (65, 784, 32), (33, 1536, 384), (34, 1552, 40), (49, 3072, 768)])
def test_linear_rows_matches_float64(M, K, N, dtype):
    print("CASE linear_rows", M, K, N, dtype, flush=True)
    x, w, b, res, gamma, beta = make(M, K, N, dtype)
    forms = [(b, None, None, None, False), (None, res, None, None, False), (b, res, None, None, True)]
    if K <= 768:
        forms += [(None, None, gamma, beta, False), (b, None, gamma, beta, True), (b, res, gamma, None, True)]
    for bias, add, g, bt, gelu in forms:
        got = linear_rows_hip(x, w, bias, add, g, bt, 1e-5, gelu)
        want = exact(x, w, bias, add, g, bt, gelu)
        assert got.dtype == dtype and got.shape == (M, N)
        rel = ((got.double() - want).norm() / want.norm()).item()
        assert rel <= 2 * U[dtype], (rel, gelu, g is not None)


def test_linear_rows_keeps_rows_apart():
    """An infinite row, or one of NaN, reaches its own results only; rows past the last position are not written."""
    x, w, b, res, gamma, beta = make(40, 384, 96, torch.bfloat16)
    clean = linear_rows_hip(x, w, b, res, gamma, beta)
    x[3, 5], x[37, 100] = float("inf"), float("nan")
    got = linear_rows_hip(x, w, b, res, gamma, beta)
    rest = [i for i in range(40) if i not in (3, 37)]
    assert torch.equal(got[rest], clean[rest]) and not got[[3, 37]].isfinite().any()
    room = torch.full((48, 96), 7.0, device=DEV, dtype=torch.bfloat16)
    rc = _lib.launch(x, _lib.lib().ss2d_linear_rows, x.data_ptr(), None, None, 1e-5, w.data_ptr(), None, None, room.data_ptr(), 40, 384, 96,
                     0, _lib.SS2D_BF16)
    assert rc == _lib.SS2D_OK and (room[40:] == 7.0).all()


def test_linear_rows_rejections():
    x, w, b, res, gamma, beta = make(8, 96, 96, torch.bfloat16)
    layer, norm = torch.nn.Linear(96, 96).to(DEV, torch.bfloat16), LayerNorm(96).to(DEV, torch.bfloat16)
    with torch.no_grad():
        assert linear_rows_fusable(x, layer, norm)
        assert not linear_rows_fusable(x.float(), layer, norm) and not linear_rows_fusable(x.cpu(), layer)
        assert not linear_rows_fusable(x.view(-1)[8:].view(-1)[:4 * 96 + 1][1:].view(4, 96), layer)      # two bytes off a boundary
        with torch.autocast("cuda", torch.float16):
            assert not linear_rows_fusable(x, layer)
        handle = layer.register_forward_hook(lambda *a: None)
        assert not linear_rows_fusable(x, layer)
        handle.remove()
        assert not linear_rows_fusable(x, layer, norm.float())
    assert not linear_rows_fusable(x, layer)                         # under autograd
    with pytest.raises(ValueError):
        linear_rows_hip(x, w[:, :16])
    with pytest.raises(ValueError):
        linear_rows_hip(x, w, residual=res[:4])
    call = lambda K, N, dt, ln=None: _lib.lib().ss2d_linear_rows(x.data_ptr(), ln, None, 1e-5, w.data_ptr(), None, None, x.data_ptr(), 8, K, N, 0, dt, None)
    for args in ((24, 96, _lib.SS2D_BF16), (96, 4, _lib.SS2D_BF16), (3088, 96, _lib.SS2D_BF16), (96, 96, _lib.SS2D_F32),
                 (784, 96, _lib.SS2D_BF16, gamma.data_ptr())):
        assert call(*args) == _lib.SS2D_ENOTSUP
    assert call(0, 96, _lib.SS2D_BF16) == _lib.SS2D_EINVAL


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("dim,side", [(96, 14), (192, 9), (384, 14), (768, 7)])
def test_block_of_few_positions(dim, side, dtype):
    """A block by linear_rows against the same block whose layers are called (hooks see them), each against the other's rounding:
    four products, two norms and a GELU rounded to 16 bits on either side, 16 u in all."""
    torch.manual_seed(dim)
    block = VSSBlock(dim, channel_first=False).to(DEV, dtype).eval()
    x = torch.randn(1, side, side, dim, device=DEV, dtype=dtype)
    seen = []
    with torch.no_grad():
        got = block(x)
        layers = (block.op.in_proj, block.op.out_proj, block.mlp.act)
        handles = [m.register_forward_hook(lambda m, i, o: seen.append(m)) for m in layers]
        want = block(x)
        for h in handles:
            h.remove()
    assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= 16 * U[dtype]
    if dim > 192:
        assert block.op.in_proj in seen and block.mlp.act in seen


def test_block_of_few_positions_under_capture():
    torch.manual_seed(5)
    block = VSSBlock(384, channel_first=False).to(DEV, torch.bfloat16).eval()
    x = torch.randn(1, 14, 14, 384, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        block(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = block(x)
        for i in range(3):
            x.copy_(torch.randn(1, 14, 14, 384, device=DEV))
            want = block(x)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), i


@pytest.mark.parametrize("layer", ["fc1", "act", "fc2"])
def test_layers_of_another_kind(layer):
    """A layer wrapped in a module that has nothing of nn.Linear's is called: the block gives what the layers give."""
    torch.manual_seed(11)
    block = VSSBlock(384, channel_first=False).to(DEV, torch.bfloat16).eval()
    x = torch.randn(1, 14, 14, 384, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        want = block(x)
        setattr(block.mlp, layer, torch.nn.Sequential(getattr(block.mlp, layer), torch.nn.Dropout(0.5).eval()))
        got = block(x)
    # the layers are the library's on one side: 16 u, as in test_block_of_few_positions
    assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= 16 * U[torch.bfloat16]
