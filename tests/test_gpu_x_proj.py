"""x_proj in scan order (ss2d_x_proj) against the float64 product on the four scan-ordered copies of the map.

The sums are fp32 over D <= 768 products of 16-bit values and are rounded once: half an ulp of the result (at most 2^-8 of
its value in bf16, with 7 mantissa bits stored, and 2^-11 in fp16, with 10) plus D * 2^-24 of the sum of the products' magnitudes."""
import pytest
import torch

from vmamba_amd import _lib
from vmamba_amd.core import x_proj_hip

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def scan_orders(m, H, W):
    """(B, C, H, W) -> (B, 4, C, L)"""
    rows, cols = m.flatten(2), m.transpose(2, 3).flatten(2)
    return torch.stack([rows, cols, rows.flip(-1), cols.flip(-1)], 1)


CASES = [
    # B, D, C, H, W, padded, mask row
    (2, 96, 8, 56, 56, None, -1),          # two bands of rows
    (3, 192, 14, 28, 28, None, -1),        # whole maps, two wide stores per position group
    (2, 384, 26, 14, 14, None, -1),        # L % 8 = 4
    (5, 768, 50, 7, 7, None, -1),          # odd maps: channels split over the wavefronts, element stores
    (1, 40, 5, 3, 3, None, -1),            # 9 positions, channels no multiple of 32
    (1, 8, 1, 1, 8, None, -1),             # one row
    (2, 48, 38, 10, 12, None, -1),         # two position groups: channels split in two
    (1, 64, 70, 24, 16, None, -1),         # more than 64 output rows
    (1, 96, 8, 256, 200, None, -1),        # large map: tiles in both directions, the last column tile narrower
    (1, 32, 4, 100, 98, None, -1),         # wide map whose width is no multiple of 4: full rows
    (1, 40, 5, 18, 18, None, -1),          # last tile (9 rows) ends inside a group of four positions, the map does not
    (2, 48, 26, 66, 66, None, -1),         # the same with two directions a workgroup
    (24, 64, 12, 58, 58, None, -1),        # five-row tiles, all directions in one workgroup
    (1, 40, 3, 65, 1, None, -1),           # one column: the tile before the last ends inside the map's last four positions
    (1, 32, 8, 137, 1, None, -1),
    (1, 8, 8, 256, 1931, None, -1),        # a row that fits LDS with two directions, not with four
    (1, 336, 23, 45, 45, None, -1),        # one odd map: tiles of two rows, channels split in two
    (1, 768, 50, 28, 28, None, -1),        # one even map: tiles of four rows
    (2, 64, 10, 56, 56, None, -1),         # from eight rows to four
    (1, 96, 8, 113, 113, None, -1),        # one row per tile
    (1, 32, 7, 9, 200, None, -1),          # tiles of half the rows in two columns of tiles
    (1, 24, 6, 131, 2, None, -1),          # two columns: tiles of 33 rows
    (2, 96, 8, 57, 58, (60, 60), 6),       # padded map with a mask row
    (1, 384, 26, 19, 19, (20, 20), -1),    # padded map without one
    (3, 16, 3, 5, 7, (8, 8), 3),           # mask row behind the last row
]

# Plans by rounds of workgroups: four, two and one direction, tiles of 4, 8 and 12 rows, a last tile of 4 of 8 rows, pieces of a row, a padded map, 90 output rows.
ROUNDS = [(12, 128, 10, 84, 84, None, -1), (15, 176, 13, 48, 48, None, -1), (3, 528, 45, 56, 56, None, -1), (5, 320, 22, 60, 28, None, -1), (2, 144, 29, 152, 152, None, -1),
          (10, 136, 43, 52, 40, None, -1), (9, 208, 15, 92, 94, (92, 96), 14)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", ROUNDS, ids=lambda c: "x".join(map(str, c[:5])))
def test_x_proj_plans_by_rounds(case, dtype):
    test_x_proj(case, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])))
def test_x_proj(case, dtype):
    B, D, C, H, W, padded, mask_row = case
    print("CASE x_proj", case, dtype, flush=True)
    g = torch.Generator().manual_seed(D + H)
    x = torch.randn(B, D, H, W, generator=g).to(dtype)
    w = (torch.randn(4, C, D, generator=g) * 0.1).to(dtype)
    Hp, Wp = padded or (H, W)
    L, rows = Hp * Wp, C + (mask_row >= 0)
    out = torch.full((4, rows, B + 1, L), 7.0, dtype=dtype, device=DEV)         # direction-major, batch-innermost, one spare image
    x_proj_hip(x.to(DEV), w.to(DEV), out[:, :, :B].permute(2, 0, 1, 3), padded, mask_row)
    got = out.cpu()
    assert bool((got[:, :, B] == 7.0).all())                                    # nothing beyond the last image
    got = got[:, :, :B].permute(2, 0, 1, 3).double()
    xp = torch.zeros(B, D, Hp, Wp, dtype=torch.float64)
    xp[:, :, :H, :W] = x.double()
    xs = scan_orders(xp, Hp, Wp)
    want, size = torch.matmul(w.double(), xs), torch.matmul(w.double().abs(), xs.abs())
    if mask_row >= 0:
        m = torch.ones(B, 1, Hp, Wp, dtype=torch.float64)
        m[:, :, :H, :W] = 0
        m = scan_orders(m, Hp, Wp)
        want = torch.cat([want[:, :, :mask_row], m, want[:, :, mask_row:]], 2)
        size = torch.cat([size[:, :, :mask_row], m, size[:, :, mask_row:]], 2)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    tiny = 2.0 ** -24                                                           # fp16's smallest step
    assert bool(((got - want).abs() <= eps * want.abs() * (1 + eps) + D * 2.0 ** -24 * size + tiny).all())


def test_x_proj_strides_and_offsets():
    """Rows that start on 2-byte boundaries only, and the reference's (B, 4, C, L) layout."""
    B, D, C, H, W = 2, 32, 6, 12, 10
    g = torch.Generator().manual_seed(1)
    x, w = torch.randn(B, D, H, W, generator=g).bfloat16(), torch.randn(4, C, D, generator=g).bfloat16()
    plain = x_proj_hip(x.to(DEV), w.to(DEV), torch.empty(B, 4, C, H * W, dtype=torch.bfloat16, device=DEV))
    store = torch.zeros(B * 4 * C * (H * W + 3) + 1, dtype=torch.bfloat16, device=DEV)
    shifted = store[1:].view(B, 4, C, H * W + 3)[..., :H * W]
    x_shifted = torch.empty(x.numel() + 1, dtype=torch.bfloat16, device=DEV)[1:].view(B, D, H, W)
    x_shifted.copy_(x)
    x_proj_hip(x_shifted, w.to(DEV), shifted)
    assert torch.equal(plain, shifted)
    want = torch.matmul(w.double(), scan_orders(x.double(), H, W))
    assert torch.allclose(plain.cpu().double(), want, rtol=2 ** -8, atol=1e-3)


def test_x_proj_refuses():
    x = torch.zeros(1, 12, 4, 4, dtype=torch.bfloat16, device=DEV)
    out = torch.zeros(1, 4, 3, 16, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(_lib.Ss2dError):
        x_proj_hip(x, torch.zeros(4, 3, 12, dtype=torch.bfloat16, device=DEV), out)            # D not a multiple of 8
    with pytest.raises(RuntimeError):
        x_proj_hip(x, torch.zeros(4, 3, 12, dtype=torch.float16, device=DEV), out)


@pytest.mark.parametrize("D, N, B, side, kernel", [(64, 16, 2, 14, True), (384, 16, 1, 14, True), (768, 16, 1, 7, True), (768, 16, 8, 19, False),
                                                   (384, 2, 2, 73, False), (384, 2, 1, 73, True),
                                                   (384, 2, 26, 15, True)])
def test_projections_of_several_states(D, N, B, side, kernel, monkeypatch):
    """project_from_map on either side of x_proj_pays: the kernel runs where it is the faster one and not beyond, and B and C are
    the float64 product's on both (bounds as above)."""
    from vmamba_amd import ss2d
    torch.manual_seed(D + side)
    op = ss2d.SS2D(d_model=D, d_state=N).to(DEV, torch.bfloat16).eval()
    x = torch.randn(B, D, side, side).bfloat16()
    ran = []
    monkeypatch.setattr(ss2d, "x_proj_hip", lambda *a: (ran.append(1), x_proj_hip(*a))[1])
    with torch.no_grad():
        _, Bs, Cs = op.project_from_map(x.to(DEV), op._inference_constants(B))
    assert bool(ran) == kernel
    w, xs = op.x_proj_weight.detach().cpu().double()[:, op.dt_rank:], scan_orders(x.double(), side, side)
    want, size = torch.matmul(w, xs), torch.matmul(w.abs(), xs.abs())
    got = torch.cat([Bs, Cs], 2).cpu().double()
    assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() * (1 + 2.0 ** -8) + D * 2.0 ** -24 * size).all())
