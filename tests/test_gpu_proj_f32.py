"""ss2d_x_proj_f32 and ss2d_dt_proj_f32 against the float64 products: n products summed in fp32 are off by at
most n * 2^-24 of the sum of their magnitudes, in whatever order (and half as much again where a product is rounded first)."""
import pytest
import torch

from vmamba_amd.core import dt_proj_f32_hip, x_proj_f32_hip

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B,D,C,H,W", [(2, 192, 14, 28, 28),          # 56 of 64 rows
                                       (3, 96, 8, 9, 7),              # two row tiles; positions of several images per wavefront
                                       (1, 50, 17, 5, 13),            # a second chunk of four rows; channels no multiple of four
                                       (2, 3, 1, 1, 1),               # one row tile, fewer channels than a step
                                       (1, 16, 50, 8, 64)])           # four chunks
def test_x_proj_f32(B, D, C, H, W):
    print("CASE x_proj_f32", B, D, C, H, W, flush=True)
    g = torch.Generator().manual_seed(D)
    x, w = torch.randn(B, D, H, W, generator=g), torch.randn(4, C, D, generator=g)
    out = torch.full((4, C, B + 1, H * W), 7.0, device=DEV)            # direction-major, batch-innermost, one spare image
    x_proj_f32_hip(x.to(DEV), w.to(DEV), out[:, :, :B].permute(2, 0, 1, 3))
    assert bool((out[:, :, B] == 7.0).all())
    rows, cols = x.flatten(2).double(), x.transpose(2, 3).flatten(2).double()
    xs = torch.stack([rows, cols, rows.flip(-1), cols.flip(-1)], 1)
    want, size = torch.matmul(w.double(), xs), torch.matmul(w.double().abs(), xs.abs())
    got = out[:, :, :B].permute(2, 0, 1, 3).cpu().double()
    assert bool(((got - want).abs() <= 1.5 * (D + 4) * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("K,D,R,N", [(4, 192, 12, 2048), (4, 70, 6, 1028), (3, 9, 1, 4), (4, 33, 13, 260), (4, 96, 24, 516),
                                     (4, 40, 22, 1022), (2, 8, 24, 77), (1, 5, 3, 1)])      # the last three: single elements
def test_dt_proj_f32(K, D, R, N):
    print("CASE dt_proj_f32", K, D, R, N, flush=True)
    g = torch.Generator().manual_seed(R)
    x_dbl, w = torch.randn(K, R + 2, N, generator=g), torch.randn(K, D, R, generator=g)
    x = x_dbl.to(DEV)[:, :R]                                           # rows of a larger tensor
    want, size = torch.bmm(w.double(), x_dbl[:, :R].double()), torch.bmm(w.double().abs(), x_dbl[:, :R].double().abs())
    got = dt_proj_f32_hip(x, w.to(DEV)).cpu().double()
    assert bool(((got - want).abs() <= 1.5 * (R + 1) * 2.0 ** -24 * size).all())


def test_wide_ranks_are_refused():
    with pytest.raises(RuntimeError):
        dt_proj_f32_hip(torch.zeros(1, 25, 8, device=DEV), torch.zeros(1, 8, 25, device=DEV))
