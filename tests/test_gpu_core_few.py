"""ss2d_x_proj_few and ss2d_core_few against float64: the sizes where a lane's share, a wavefront's channels or a rank piece ends."""
import pytest
import torch

from vmamba_amd import _lib
from vmamba_amd.core import core_few_hip, few_applies
from vmamba_amd.ss2d import SS2D

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def routes(x):
    """(B, D, H, W) -> (4, B, D, L) in the directions' scan orders."""
    rows, cols = x.flatten(2), x.transpose(2, 3).flatten(2)
    return torch.stack([rows, cols, rows.flip(-1), cols.flip(-1)])


def core_f64(op, x):
    B, D, H, W = x.shape
    R = op.dt_rank
    u = routes(x.double())
    rows = torch.einsum("kcd,kbdl->kbcl", op.x_proj_weight.double(), u).to(x.dtype).double()
    step = torch.einsum("kdr,kbrl->kbdl", op.dt_projs_weight.double(), rows[:, :, :R])
    step = torch.nn.functional.softplus(step + op.dt_projs_bias.double().view(4, 1, D, 1))
    A, skip = -op.A_logs.double().exp().view(4, 1, D), op.Ds.double().view(4, 1, D, 1)
    decay, drive = torch.exp(step * A[..., None]), step * u * rows[:, :, R, None]
    h, hs = torch.zeros_like(drive[..., 0]), torch.empty_like(drive)
    for j in range(H * W):
        h = decay[..., j] * h + drive[..., j]
        hs[..., j] = h
    y = hs * rows[:, :, R + 1, None] + skip * u
    return y[0] + y[2].flip(-1) + (y[1] + y[3].flip(-1)).view(B, D, W, H).transpose(2, 3).flatten(2)


def make(D, rank, dtype, seed):
    torch.manual_seed(seed)
    op = SS2D(d_model=D, dt_rank=rank, channel_first=False).to(DEV).to(dtype).eval()
    with torch.no_grad():
        op.A_logs.add_(torch.randn_like(op.A_logs) * 0.5)
        op.Ds.add_(torch.randn_like(op.Ds))
    return op


def run(op, x):
    c = op._inference_constants(0)
    return core_few_hip(x, op.x_proj_weight, op.dt_projs_weight, c["As"].view(-1), c["Ds"], c["dt_bias"])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,D,H,W,R", [(1, 768, 7, 7, 48), (2, 8, 2, 2, 1), (1, 40, 1, 5, 3), (3, 384, 14, 14, 24), (2, 192, 16, 16, 12),
                                       (1, 320, 9, 11, 20), (2, 104, 15, 13, 7), (1, 24, 3, 70, 2), (2, 48, 8, 8, 16), (1, 16, 255, 1, 8),
                                       (1, 600, 5, 13, 38), (1, 760, 8, 8, 47), (2, 136, 13, 5, 9), (1, 256, 10, 6, 23)])
def test_against_float64(B, D, H, W, R, dtype):
    """From the same rounded ranks on both compute the same sums, in fp32 here: some hundred roundings of 2^-24.  A rank whose fp32 and
    float64 sums round to different 16-bit neighbours moves one of R terms of one position's step by 2^-8; 1e-4 of the norm allows for a
    few of those in the smallest maps."""
    print("CASE core_few", B, D, H, W, R, dtype, flush=True)
    if dtype == torch.float32 and R > 24:
        assert _lib.lib().ss2d_few_rows_bytes(B, D, R, H, W, _lib.SS2D_F32) == _lib.SS2D_ENOTSUP
        return
    op = make(D, R, dtype, H)
    x = torch.nn.functional.silu(torch.randn(B * D * H * W + 1, device=DEV)).to(dtype)[1:].view(B, D, H, W)      # (off the 16-byte grid)
    with torch.no_grad():
        got, want = run(op, x), core_f64(op, x)
    assert ((got.double() - want).norm() / want.norm()).item() < (1e-6 if dtype == torch.float32 else 1e-4)
    assert ((got.double() - want).abs().max() / want.square().mean().sqrt()).item() < (1e-5 if dtype == torch.float32 else 2e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,W", [(7, 7), (9, 12)])
def test_nan_stays_where_it_is(H, W, dtype):
    op = make(64, 5, dtype, 1)
    x = torch.randn(3, 64, H, W, device=DEV).to(dtype)
    with torch.no_grad():
        clean = run(op, x)
        x[1, 3, H // 2, 2] = float("nan")
        got, want = run(op, x), core_f64(op, x)
    assert torch.equal(got[[0, 2]], clean[[0, 2]]) and torch.equal(got.isnan(), want.isnan())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("names", [("Ds",), ("dt_projs_bias",), ("A_logs",), ("x_proj_weight", "dt_projs_weight"), ("Ds", "dt_projs_bias", "A_logs", "x_proj_weight", "dt_projs_weight")])
def test_strided_parameters(names, dtype):
    """Parameters that are every other element of a larger tensor: forward_core's bits of the same values side by side."""
    op, x = make(64, 5, dtype, 3), torch.randn(2, 64, 7, 9, device=DEV).to(dtype)
    assert few_applies(2, 64, 7, 9, 5, dtype)
    with torch.no_grad():
        want = op.forward_core(x)
        for name in names:
            p = getattr(op, name)
            wide = torch.empty(p.shape + (2,), device=DEV, dtype=p.dtype)
            wide[..., 0].copy_(p)
            setattr(op, name, torch.nn.Parameter(wide[..., 0]))
            assert not getattr(op, name).is_contiguous()
        assert torch.equal(op.forward_core(x), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,W", [(7, 7), (8, 8), (9, 12)])
@pytest.mark.parametrize("bad", range(4))
def test_directions_and_channels_keep_to_themselves(H, W, dtype, bad):
    """One direction's state of one channel overflows on the way, through a step of that direction alone (2^126, no decay): the merged map is
    infinite nowhere but from there on in that direction's order, and the other channels have the bits they had."""
    op, x = make(64, 5, dtype, 4), torch.rand(2, 64, H, W, device=DEV).add(0.5).to(dtype)
    with torch.no_grad():
        op.x_proj_weight.abs_()
        op.x_proj_weight[:, 5:].div_(16)                             # B and C positive, below 1
        c = op._inference_constants(0)
        c = {"As": c["As"].view(-1).clone(), "Ds": c["Ds"].clone(), "dt_bias": c["dt_bias"].clone()}
        call = lambda: core_few_hip(x, op.x_proj_weight, op.dt_projs_weight, c["As"], c["Ds"], c["dt_bias"])
        clean = call()
        c["As"][bad * 64 + 3], c["dt_bias"][bad * 64 + 3] = 0.0, 2.0 ** 126
        got = call()
        others = [d for d in range(64) if d != 3]
        assert torch.equal(got[:, others], clean[:, others])
        # the state in units of the step, which swallows its ranks; where the sum of two lanes' shares would overflow their outputs may still not
        rows = torch.einsum("cd,bdl->bcl", op.x_proj_weight[bad].double(), routes(x.double())[bad]).to(dtype).double()
        state = torch.cumsum(routes(x.double())[bad][:, 3] * rows[:, 5], -1)
        value = torch.stack([state, 2.0 ** 126 * state * rows[:, 6]])
        value = value.flip(-1) if bad >= 2 else value
        state, value = value.view(2, 2, W, H).transpose(2, 3).flatten(2) if bad % 2 else value
    over, near = state > 3.99, torch.isclose(got[:, 3].double(), value, rtol=1e-4 if dtype == torch.float32 else 2.0 ** -7)
    assert 0 < over.sum() < over.numel() and bool((near | over & got[:, 3].isposinf()).all()) and bool(got[:, 3].isposinf().any())


def test_rule():
    """Both sides of the line in one map's sizes, and what has no variant."""
    assert few_applies(1, 768, 7, 7, 48, torch.bfloat16) and few_applies(27, 768, 7, 7, 48, torch.bfloat16)
    assert not few_applies(28, 768, 7, 7, 48, torch.bfloat16) and few_applies(28, 768, 7, 7, 24, torch.float32)
    assert not few_applies(1, 768, 17, 16, 48, torch.bfloat16) and not few_applies(1, 770, 7, 7, 48, torch.bfloat16)
    op = make(64, 5, torch.bfloat16, 2)
    for shape in ((1, 64, 1, 3), (1, 64, 17, 16)):
        with pytest.raises(_lib.Ss2dError):
            run(op, torch.zeros(shape, device=DEV, dtype=torch.bfloat16))
