"""forward_core with dt_proj folded into the core: against float64 from the same 16-bit projections, and what it does with ranks that
are infinite or NaN, which its matrix product would carry to other positions."""
import pytest
import torch

from vmamba_amd.core import padded_map_size, x_proj_hip
from vmamba_amd.ss2d import SS2D

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def make(D, dtype, seed):
    torch.manual_seed(seed)
    return SS2D(d_model=D, channel_first=False).to(DEV).to(dtype).eval()


def routes(x):
    """(B, D, H, W) -> (4, B, D, L) in the directions' scan orders."""
    rows, cols = x.flatten(2), x.transpose(2, 3).flatten(2)
    return torch.stack([rows, cols, rows.flip(-1), cols.flip(-1)])


def core_f64(op, x):
    B, D, H, W = x.shape
    R, L = op.dt_rank, H * W
    rows = x.new_empty(B, 4, R + 2, L)
    x_proj_hip(x, op.x_proj_weight, rows)
    rows = rows.double().permute(1, 0, 2, 3)                                                # (4, B, R + 2, L)
    step = torch.einsum("kdr,kbrl->kbdl", op.dt_projs_weight.double(), rows[:, :, :R])      # einsum over float64: no batched bf16 product
    step = torch.nn.functional.softplus(step + op.dt_projs_bias.double().view(4, 1, D, 1))
    A, skip = -op.A_logs.double().exp().view(4, 1, D), op.Ds.double().view(4, 1, D, 1)
    u = routes(x.double())
    decay, drive = torch.exp(step * A[..., None]), step * u * rows[:, :, R, None]
    h, hs = torch.zeros_like(drive[..., 0]), torch.empty_like(drive)
    for j in range(L):
        h = decay[..., j] * h + drive[..., j]
        hs[..., j] = h
    y = hs * rows[:, :, R + 1, None] + skip * u
    down = (y[1] + y[3].flip(-1)).view(B, D, W, H).transpose(2, 3).flatten(2)
    return y[0] + y[2].flip(-1) + down


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,H,W", [(4, 96, 48, 48), (3, 48, 64, 60),       # 16 positions per lane, three and two pairs of ranks, last pass of 256 / 768
                                     (2, 96, 56, 56),                        # ... and a short one of 64
                                     (6, 112, 28, 28), (11, 80, 32, 24), (10, 128, 20, 24), (58, 128, 8, 9),   # 8, several images per workgroup, even and odd ranks
                                     (2, 64, 80, 80), (1, 48, 112, 108),     # several wavefronts per direction
                                     (2, 96, 57, 58), (3, 80, 57, 58), (9, 48, 33, 35)])     # maps with added rows and columns
def test_against_float64(B, D, H, W, dtype):
    """The ranks are 16-bit numbers in both; from there on the kernel computes in fp32: sums of at most eight products, a step, and a
    state that forgets within some hundred positions, a few hundred roundings of 2^-24.  A delta rounded to bf16 would be 1e-4 off."""
    print("CASE dt_fold", B, D, H, W, dtype, flush=True)
    assert B * D * H * W >= 1 << 19 or padded_map_size(H, W, dtype)
    op = make(D, dtype, H)
    x = torch.nn.functional.silu(torch.randn(B, D, H, W, device=DEV)).to(dtype)
    with torch.no_grad():
        got, want = op._forward_core_native(x, False), core_f64(op, x)
    assert ((got.double() - want).norm() / want.norm()).item() < 1e-5
    assert ((got.double() - want).abs().max() / want.square().mean().sqrt()).item() < 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,H,W", [(16, 96, 28, 28), (4, 96, 56, 56), (4, 96, 57, 58), (2, 64, 80, 80)])
@pytest.mark.parametrize("what", ["inf", "nan", "rank"])
def test_non_finite_ranks_stay_where_they_are(B, D, H, W, dtype, what, monkeypatch):
    """One position of one image is infinite, NaN, or has a rank beyond fp16: the same outputs stay finite as with the kernels one by
    one, whose projections keep to their positions, and those agree to the rounding of delta."""
    print("CASE dt_fold non-finite", B, D, H, W, dtype, what, flush=True)
    op = make(D, dtype, W)
    x = torch.nn.functional.silu(torch.randn(B, D, H, W, device=DEV)).to(dtype)
    with torch.no_grad():
        if what == "rank":
            op.x_proj_weight[1, 2] = 20.0                          # one rank of one direction: 20 * 60000 there, ordinary elsewhere
            x[1, :, H // 2, W // 3] = 60000.0 / D
        else:
            x[1, 3, H // 2, W // 3] = float(what)
        got = op.forward_core(x).float()
        monkeypatch.setattr(SS2D, "_forward_core_native", lambda self, x, normalise: None)
        want = op.forward_core(x).float()
    assert torch.equal(got.isfinite(), want.isfinite())
    if what != "rank" or dtype == torch.float16:
        assert not got[1].isfinite().all()
    ok = want.isfinite()
    assert ((got - want)[ok].norm() / want[ok].norm()).item() < (2e-2 if dtype == torch.bfloat16 else 2.5e-3)
