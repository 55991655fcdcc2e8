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


@pytest.mark.parametrize("d_state, B, D, H, W, kernel", [(2, 1, 416, 71, 71, True), (2, 1, 416, 73, 71, False), (2, 5, 416, 64, 64, False),
                                                         (1, 1, 416, 71, 71, True), (1, 1, 416, 73, 71, False), (2, 1, 96, 151, 151, True)])
def test_projection_on_either_side_of_the_rule(d_state, B, D, H, W, kernel, monkeypatch):
    """forward_core takes ss2d_x_proj_f32 where x_proj_f32_pays says so and the library's product elsewhere, with one result: the
    projections differ by D * 2^-24 of their products' magnitudes, some 1e-6 of the output after the scan and the norm."""
    from vmamba_amd import ss2d
    torch.manual_seed(D + H)
    op = ss2d.SS2D(d_model=D, d_state=d_state).cuda().eval()
    x = torch.nn.functional.silu(torch.randn(B, D, H, W)).cuda()
    ran, kept = [], ss2d.x_proj_f32_hip
    monkeypatch.setattr(ss2d, "x_proj_f32_hip", lambda *a: (ran.append(1), kept(*a))[1])
    with torch.no_grad():
        got = op.forward_core(x)
        assert bool(ran) == kernel
        monkeypatch.setattr(ss2d, "x_proj_f32_pays", lambda *a: not kernel)
        other = op.forward_core(x)
        assert len(ran) == 1
    assert ((got - other).double().norm() / other.double().norm()).item() < 1e-5
