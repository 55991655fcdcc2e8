"""Fused SS2D core operator: CrossScan -> selective scan -> CrossMerge in one HIP kernel (d_state = 1).

Stands in for the three operator calls of SS2Dv2.forward_corev2 (classification/models/vmamba.py:604,
625-633, 638) when the model has one state per channel; the projections between them remain the caller's.
"""
import math

import torch

from . import _lib
from .csm import cross_merge_fn
from .norm import TENSOR_KINDS, TRAIN_FROM, calls_unseen

_DTYPE_CODE = {torch.float32: _lib.SS2D_F32, torch.bfloat16: _lib.SS2D_BF16, torch.float16: _lib.SS2D_F16}


def _check(cond, msg):
    if not cond:
        raise RuntimeError(msg)


def _lds_extent(n, es):
    """Elements an LDS array of n logical elements takes: one spare 4-byte word per 32 words, rounded to 8 elements."""
    idx = n + (n >> 5) if es == 4 else n + ((n >> 6) << 1)
    return (idx + 8) & ~7


def core_fits(H, W, dtype):
    """True when the fused core takes an H x W image of this dtype: at least 8 positions, and either the LDS arrays
    of one image (two fp32 merge planes, two copies of the x map plus a block of 8 zeros each) within the 160 KiB of a CU --
    the single kernel, maps of up to ~13 000 positions -- or 16-bit maps whose sides are multiples of 8, which the tiled two-pass kernels take at any size."""
    if dtype not in _DTYPE_CODE:
        return False
    L = H * W
    es = 4 if dtype == torch.float32 else 2
    if _fits_single_kernel(L, es):
        return True
    return es == 2 and ((H % 8 == 0 and W % 8 == 0) or padded_map_size(H, W, dtype) is not None)


def _fits_single_kernel(L, es):
    maps = _lds_extent(((L + 7) & ~7) + 8, es)
    return L >= 8 and 2 * _lds_extent(L, 4) * 4 + 2 * maps * es <= 160 * 1024 - 256


def padded_map_size(H, W, dtype):
    """(H', W') >= (H, W) in which a caller should embed an H x W map for the fused core, or None when the map is fine
    as it is (or padding would not pay).  16-bit maps only.  The core's vector paths want a number of positions that is
    a multiple of 8 and, for the 4 x 4 tiles of its staging and merge, sides that are multiples of 4 (so: multiples of
    4, whose product is a multiple of 16); maps beyond the single kernel's LDS arrays go to the tiled kernels, which want
    multiples of 8.  Without them the core walks the map element by element at a third to a quarter of the rate, which a
    padded area of up to 1.5 times the map's beats."""
    if dtype not in (torch.bfloat16, torch.float16):
        return None
    L = H * W
    if H == W == 7:                      # has a kernel of its own (one map row per lane)
        return None
    if _fits_single_kernel(L, 2):
        if math.gcd(L, 8) >= 4:
            return None
        H4, W4 = (H + 3) & ~3, (W + 3) & ~3
        if _fits_single_kernel(H4 * W4, 2):
            return (H4, W4) if H4 * W4 <= 1.5 * L else None
    if H % 8 == 0 and W % 8 == 0:
        return None
    H8, W8 = (H + 7) & ~7, (W + 7) & ~7
    return (H8, W8) if H8 * W8 <= 1.5 * L else None


def core_mask_pads_hip(delta, H, W, Hp, Wp):
    """delta (4, D, B, Hp*Wp) view of the padded map's steps: -inf at the scan positions that fall on the rows >= H and the
    columns >= W, in every direction's order (ss2d_core_mask_pads).  In place."""
    _check(delta.is_cuda and delta.dim() == 4 and delta.shape[0] == 4 and delta.shape[3] == Hp * Wp, "delta must be (4, D, B, Hp*Wp) on the GPU")
    _check(delta.dtype in _DTYPE_CODE and (delta.stride(3) == 1 or delta.shape[3] == 1), "delta must be contiguous along the map")
    rc = _lib.launch(delta, _lib.lib().ss2d_core_mask_pads, delta.data_ptr(), delta.shape[2], delta.shape[1], H, W, Hp, Wp,
                     delta.stride(0), delta.stride(1), delta.stride(2), _DTYPE_CODE[delta.dtype])
    _lib.check(rc, "ss2d_core_mask_pads")
    return delta


def embed_maps_hip(src, dst_rows, dst_cols):
    """src (n_maps, rows, cols), contiguous, 2- or 4-byte elements -> (n_maps, dst_rows, dst_cols): the maps zero-padded at
    the bottom / right or cropped there, in one pass (ss2d_core_embed_maps)."""
    _check(src.is_cuda and src.dim() == 3 and src.is_contiguous(), "embed_maps: a contiguous (n_maps, rows, cols) GPU tensor")
    _check(src.element_size() in (2, 4), "embed_maps: 2- or 4-byte elements")
    n, rows, cols = src.shape
    dst = src.new_empty((n, dst_rows, dst_cols))
    if dst.numel() == 0:
        return dst
    if src.numel() == 0:
        return dst.zero_()
    rc = _lib.launch(src, _lib.lib().ss2d_core_embed_maps, src.data_ptr(), dst.data_ptr(), n, rows, cols, dst_rows, dst_cols,
                     src.element_size())
    _lib.check(rc, "ss2d_core_embed_maps")
    return dst


def ss2d_core_hip(x, delta, Bs, Cs, As, Ds=None, delta_bias=None, delta_softplus=True, out=None):
    """x (B,D,H,W); delta (4,D,B,L) view; Bs, Cs (4,B,L) views (last stride 1), all of x.dtype and already in the
    scan order of their direction; As, Ds, delta_bias (4*D) fp32.  Returns the merged y (B,D,L) fp32 (written into
    ``out`` when given: a contiguous fp32 tensor of that shape).

    Raises Ss2dError with status SS2D_ENOTSUP when the shape has no fused kernel (an image too large for the LDS
    planes that the tiled kernels do not take either: fp32, sides not multiples of 8, unaligned rows): callers fall
    back to the three separate operators.
    """
    _check(x.is_cuda, "ss2d_core: vmamba_amd runs on the GPU only")
    _check(x.dim() == 4, "x must be (B, D, H, W)")
    _check(x.dtype in _DTYPE_CODE, f"ss2d_core not implemented for input type '{x.dtype}'")
    B, D, H, W = x.shape
    L = H * W
    for name, t in (("delta", delta), ("B", Bs), ("C", Cs)):
        _check(t.is_cuda and t.dtype == x.dtype, f"{name} must be a GPU tensor of x's dtype")
        _check(t.stride(-1) == 1 or t.size(-1) == 1, f"{name} must be contiguous in its last dimension")
    _check(tuple(delta.shape) == (4, D, B, L), "delta must have shape (4, dim, batch, L)")
    _check(tuple(Bs.shape) == (4, B, L) and tuple(Cs.shape) == (4, B, L), "B and C must have shape (4, batch, L)")
    _check(As.dtype == torch.float32 and As.is_cuda and As.numel() == 4 * D, "A must be (4*dim) float32 (one state)")
    As = As.contiguous()
    if Ds is not None:
        _check(Ds.dtype == torch.float32 and Ds.is_cuda and tuple(Ds.shape) == (4 * D,), "D must be (4*dim) float32")
        Ds = Ds.contiguous()
    if delta_bias is not None:
        _check(delta_bias.dtype == torch.float32 and delta_bias.is_cuda and tuple(delta_bias.shape) == (4 * D,),
               "delta_bias must be (4*dim) float32")
        delta_bias = delta_bias.contiguous()
    x = x.contiguous()
    if out is None:
        y = torch.empty((B, D, L), device=x.device, dtype=torch.float32)
    else:
        _check(out.is_cuda and out.dtype == torch.float32 and tuple(out.shape) == (B, D, L) and out.is_contiguous(),
               "out must be a contiguous float32 GPU tensor of shape (batch, dim, L)")
        y = out
    p = _lib.CoreParams()
    p.batch, p.dim, p.height, p.width = B, D, H, W
    p.in_dtype = _DTYPE_CODE[x.dtype]
    p.delta_softplus = 1 if delta_softplus else 0
    p.x, p.delta, p.A, p.B, p.C = x.data_ptr(), delta.data_ptr(), As.data_ptr(), Bs.data_ptr(), Cs.data_ptr()
    p.D = Ds.data_ptr() if Ds is not None else None
    p.delta_bias = delta_bias.data_ptr() if delta_bias is not None else None
    p.y = y.data_ptr()
    p.delta_dir_stride, p.delta_dim_stride, p.delta_batch_stride = delta.stride(0), delta.stride(1), delta.stride(2)
    p.B_dir_stride, p.B_batch_stride = Bs.stride(0), Bs.stride(1)
    p.C_dir_stride, p.C_batch_stride = Cs.stride(0), Cs.stride(1)
    # maps too large for the single kernel are walked in tiles, twice, through scratch memory of the size the library asks for
    need = _lib.lib().ss2d_core_workspace_bytes(p)
    _lib.check(min(need, 0), "ss2d_core_workspace_bytes")
    if need > 0:
        workspace = torch.empty(need, dtype=torch.uint8, device=x.device)
        rc = _lib.launch(x, _lib.lib().ss2d_core_fwd_ws, p, workspace.data_ptr(), need)
    else:
        rc = _lib.launch(x, _lib.lib().ss2d_core_fwd, p)
    _lib.check(rc, "ss2d_core_fwd")
    return y


def forward_core_hip(x, x_proj_weight, dt_proj_weight, As, Ds, dt_bias, norm=None, out_channel_last=False, pad_mask=None):
    """x_proj, dt_proj, the fused core and -- with ``norm`` -- out_norm in one call (ss2d_forward_core): x (B,D,H,W),
    x_proj_weight (4,R+2,D), dt_proj_weight (4,D,R) of one dtype; As, Ds, dt_bias (4*D) fp32; norm a LayerNorm over D.  Returns
    (B,H,W,D) if ``out_channel_last`` else (B,D,H,W) in x.dtype, the merged map (B,D,L) in fp32 without ``norm``, or None
    where the kernels have no variant for the call and the separate ones have to be tried.  Maps that padded_map_size embeds in
    larger ones need pad_mask(H, W, padded H, padded W, B, device): the mask dt_proj_hip takes."""
    _check(x.is_cuda, "forward_core: vmamba_amd runs on the GPU only")
    B, D, H, W = x.shape
    R = dt_proj_weight.shape[2]
    dtype = x.dtype
    padded = None if few_applies(B, D, H, W, R, dtype) and x_proj_weight.data_ptr() % 16 == 0 else padded_map_size(H, W, dtype)
    mask = None
    if padded is not None:
        if pad_mask is None or R > DT_PROJ_MAX_RANK or dtype not in _DTYPE_CODE or x.numel() == 0:
            return None
        mask = pad_mask(H, W, *padded, B, x.device)
        _check(mask.get_device() == x.get_device() and mask.dtype == torch.int16 and mask.is_contiguous()
               and tuple(mask.shape) == (4, B * padded[0] * padded[1]), "pad_mask: (4, B * L) int16")
        H, W = padded
    weight, bias, eps = (None, None, 0.0) if norm is None else (norm.weight, norm.bias, norm.eps)
    out = _lib.host().forward_core(x, x_proj_weight, dt_proj_weight, As, Ds, dt_bias, weight, bias, eps, norm is not None, out_channel_last, H, W, mask)
    if type(out) is int:
        _lib.check(out, "ss2d_forward_core")
    return out


def few_applies(B, D, H, W, rank, dtype):
    """True when the two kernels for a few short maps (B, D, H, W) are the faster way from the map to its merged map, one state per
    channel and ``rank`` ranks per direction (ss2d_few_applies)."""
    code = _DTYPE_CODE.get(dtype)
    return (code is not None and H * W <= FEW_MOST_POSITIONS
            and _lib.lib().ss2d_few_applies(B, D, rank, H, W, code) == _lib.SS2D_OK)


FEW_MOST_POSITIONS = 256             # of a map; a first look that costs nothing


def core_few_hip(x, x_proj_weight, dt_proj_weight, As, Ds, dt_bias):
    """x (B, D, H, W), x_proj_weight (4, R + 2, D), dt_proj_weight (4, D, R) of one dtype, As, Ds, dt_bias (4 * D) fp32: the merged
    map (B, D, L) in fp32 of a few short maps (ss2d_x_proj_few, ss2d_core_few)."""
    _check(x.is_cuda and x.dim() == 4 and x.dtype in _DTYPE_CODE, "core_few: a (B, D, H, W) map on the GPU")
    B, D, H, W = x.shape
    R = dt_proj_weight.shape[2]
    _check(tuple(x_proj_weight.shape) == (4, R + 2, D) and tuple(dt_proj_weight.shape) == (4, D, R), "core_few: weights (4, R + 2, D) and (4, D, R)")
    for t in (x_proj_weight, dt_proj_weight):
        _check(t.dtype == x.dtype and t.device == x.device, "core_few: weights of x's dtype on its device")
    for t in (As, Ds, dt_bias):
        _check(t.dtype == torch.float32 and t.device == x.device and t.numel() == 4 * D, "core_few: A, D and the bias (4 * D) float32")
    x, x_proj_weight, dt_proj_weight, As, Ds, dt_bias = (t.contiguous() for t in (x, x_proj_weight, dt_proj_weight, As, Ds, dt_bias))
    code, L = _DTYPE_CODE[x.dtype], _lib.lib()
    need = L.ss2d_few_rows_bytes(B, D, R, H, W, code)
    _lib.check(min(need, 0), "ss2d_few_rows_bytes")
    rows = torch.empty(need, dtype=torch.uint8, device=x.device)
    y = torch.empty((B, D, H * W), device=x.device, dtype=torch.float32)
    _lib.check(_lib.launch(x, L.ss2d_x_proj_few, x.data_ptr(), x_proj_weight.data_ptr(), rows.data_ptr(), B, D, R, H, W, code), "ss2d_x_proj_few")
    _lib.check(_lib.launch(x, L.ss2d_core_few, x.data_ptr(), rows.data_ptr(), dt_proj_weight.data_ptr(), As.data_ptr(), Ds.data_ptr(),
                           dt_bias.data_ptr(), y.data_ptr(), B, D, R, H, W, code), "ss2d_core_few")
    return y


def x_proj_fits(x, weight):
    """True when ss2d_x_proj takes this map (B, D, H, W) and these weights (4, C, D)."""
    return (x.is_cuda and weight.device == x.device and x.dtype in (torch.bfloat16, torch.float16) and weight.dtype == x.dtype
            and weight.is_contiguous() and weight.data_ptr() % 16 == 0
            and _lib.lib().ss2d_x_proj_applies(x.shape[0], x.shape[1], weight.shape[1], x.shape[2], x.shape[3], _DTYPE_CODE[x.dtype]) == _lib.SS2D_OK)


def x_proj_pays(x, weight):
    """False where the library's batched product with the one-by-one CrossScan behind it is the faster way to what ss2d_x_proj
    gives for a map (B, D, H, W) and weights (4, C, D).  Many channels on large maps, where the library's product fills the chip
    and the kernel's four readings of the map add up (48 images of 768 x 28 x 28, C = 56: 60 us against 49); earlier on odd maps,
    whose stores are single elements (48 images of 576 x 31 x 31, C = 44: 70 against 47; of 192 x 56 x 56, C = 44, the kernel 62
    against 77), and beyond C = 64, where a workgroup has six accumulator tiles of one direction (48 images of 768 x 28 x 28, C = 80:
    82 against 68).  On small maps the kernel may be the slower one too (one image of 768 x 14 x 14, C = 80: 15 against 10) but is a
    launch fewer, and a call that short waits for the host: forward_core there 121 us with the kernel, 153 with the library.  Many
    images of few positions are the kernel's at any size, the library's product of one image being too narrow (128 of 768 x 7 x 7,
    C = 50: 19 against 25; 64 of 768 x 15 x 15: 28 against 46)."""
    B, D, H, W = x.shape
    many = weight.shape[1] > 64
    return H * W < 256 or B * D * H * W < (2 << 20 if many or H * W % 2 else 16 << 20) or (D < 384 and not many)


def x_proj_hip(x, weight, out, padded=None, mask_row=-1):
    """weight (4, C, D) applied to the map x (B, D, H, W), each direction's rows in its scan order, written into ``out``: a
    (B, 4, C', L') view with contiguous rows (any batch / direction / row strides), L' = H' * W' of the ``padded`` size
    (default: H, W), C' = C, or C + 1 with a row at index ``mask_row`` that is 1 at the added positions (ss2d_x_proj)."""
    _check(x.is_cuda and x.dim() == 4 and weight.dim() == 3 and weight.shape[0] == 4 and weight.shape[2] == x.shape[1],
           "x_proj expects x (B, D, H, W) and weight (4, C, D)")
    _check(x.dtype == weight.dtype == out.dtype and x.dtype in _DTYPE_CODE, "x_proj: one 16-bit dtype")
    _check(weight.device == out.device == x.device, "x_proj: tensors on one device")
    B, D, H, W = x.shape
    Hp, Wp = padded or (H, W)
    C = weight.shape[1]
    _check(tuple(out.shape) == (B, 4, C + (mask_row >= 0), Hp * Wp) and (out.stride(3) == 1 or out.shape[3] == 1),
           "x_proj: out must be a (B, 4, rows, L) view with contiguous rows")
    x, weight = x.contiguous(), weight.contiguous()
    rc = _lib.launch(x, _lib.lib().ss2d_x_proj, x.data_ptr(), weight.data_ptr(), out.data_ptr(), B, D, C, H, W, Hp, Wp,
                     mask_row, out.stride(1), out.stride(2), out.stride(0), _DTYPE_CODE[x.dtype])
    _lib.check(rc, "ss2d_x_proj")
    return out


DT_PROJ_MAX_RANK = 48


def dt_proj_hip(x, weight, mask=None, fill=0.0):
    """delta[k] = weight[k] @ x[k]: x (K, R, N) with contiguous rows (any direction / rank strides), weight (K, D, R),
    both bf16 or fp16 -> (K, D, N) of the same dtype, on the matrix cores (ss2d_dt_proj).  With ``mask`` -- (K, N) int16,
    0 or -1 -- every channel's delta at the positions marked -1 is ``fill`` instead (ss2d_dt_proj_masked)."""
    _check(x.is_cuda and weight.is_cuda, "dt_proj: vmamba_amd runs on the GPU only")
    _check(x.dim() == 3 and weight.dim() == 3 and x.shape[0] == weight.shape[0] and x.shape[1] == weight.shape[2],
           "dt_proj expects x (K, R, N) and weight (K, D, R)")
    _check(x.dtype == weight.dtype and x.dtype in (torch.bfloat16, torch.float16), "dt_proj: bf16 or fp16 tensors")
    _check(x.stride(2) == 1 or x.size(2) == 1, "x must be contiguous in its last dimension")
    K, R, N = x.shape
    D = weight.shape[1]
    if mask is not None:
        _check(mask.is_cuda and mask.device == x.device and mask.dtype == torch.int16 and tuple(mask.shape) == (K, N)
               and mask.is_contiguous(), "dt_proj: mask must be a contiguous (K, N) int16 tensor on x's device")
    weight = weight.contiguous()
    out = torch.empty((K, D, N), device=x.device, dtype=x.dtype)
    rc = _lib.launch(x, _lib.lib().ss2d_dt_proj_masked, x.data_ptr(), weight.data_ptr(),
                     None if mask is None else mask.data_ptr(), float(fill), out.data_ptr(), K, D, R, N, x.stride(0),
                     x.stride(1), _DTYPE_CODE[x.dtype])
    _lib.check(rc, "ss2d_dt_proj")
    return out


def x_proj_f32_fits(x, weight):
    """True when ss2d_x_proj_f32 takes this map (B, D, H, W) and these weights (4, C, D)."""
    return (x.is_cuda and x.dtype == weight.dtype == torch.float32 and weight.device == x.device and x.numel() > 0
            and x.numel() // x.shape[1] < 2 ** 31)


def x_proj_f32_pays(x, weight):
    """x_proj_pays in single precision.  Few wavefronts share many channels there and load them step by step, single floats on
    maps of no whole 16-byte pieces: with 384 channels or more the library is ahead from 2 Mi elements on for those (48 images of
    576 x 17 x 17, one state: forward_core 396 us, with the kernel 413) and from 8 Mi on for the others (16 of 768 x 28 x 28,
    four states: 341 against 356).  Below, the library's time jumps between neighbouring shapes -- 48 images of 576 x 7 x 7 take it
    four times the kernel's -- and the call waits for the host; many images of few positions are the kernel's at any size (64 of
    768 x 14 x 14, C = 50: 72 against 196)."""
    B, D, H, W = x.shape
    return D < 384 or H * W < 256 or B * D * H * W < (2 << 20 if H * W % 4 else 8 << 20)


def x_proj_f32_hip(x, weight, out):
    """x_proj_hip in single precision: weight (4, C, D) applied to the map x (B, D, H, W), each direction's rows in its scan
    order, into ``out``: a (B, 4, C, L) view with contiguous rows (ss2d_x_proj_f32)."""
    _check(x.is_cuda and x.dim() == 4 and weight.dim() == 3 and weight.shape[0] == 4 and weight.shape[2] == x.shape[1],
           "x_proj_f32 expects x (B, D, H, W) and weight (4, C, D)")
    _check(x.dtype == weight.dtype == out.dtype == torch.float32 and weight.device == out.device == x.device,
           "x_proj_f32: float32 tensors on one device")
    B, D, H, W = x.shape
    C = weight.shape[1]
    _check(tuple(out.shape) == (B, 4, C, H * W) and (out.stride(3) == 1 or out.shape[3] == 1),
           "x_proj_f32: out must be a (B, 4, rows, L) view with contiguous rows")
    x, weight = x.contiguous(), weight.contiguous()
    rc = _lib.launch(x, _lib.lib().ss2d_x_proj_f32, x.data_ptr(), weight.data_ptr(), out.data_ptr(), B, D, C, H, W,
                     out.stride(1), out.stride(2), out.stride(0))
    _lib.check(rc, "ss2d_x_proj_f32")
    return out


DT_PROJ_F32_MAX_RANK = 24


def dt_proj_f32_hip(x, weight):
    """dt_proj_hip in single precision: x (K, R, N) with contiguous rows, weight (K, D, R) -> (K, D, N) (ss2d_dt_proj_f32)."""
    _check(x.is_cuda and x.dim() == 3 and weight.dim() == 3 and x.shape[0] == weight.shape[0] and x.shape[1] == weight.shape[2],
           "dt_proj_f32 expects x (K, R, N) and weight (K, D, R)")
    _check(x.dtype == weight.dtype == torch.float32 and x.device == weight.device, "dt_proj_f32: float32 tensors on one device")
    _check(x.stride(2) == 1 or x.size(2) == 1, "x must be contiguous in its last dimension")
    K, R, N = x.shape
    D = weight.shape[1]
    weight = weight.contiguous()
    out = torch.empty((K, D, N), device=x.device, dtype=x.dtype)
    rc = _lib.launch(x, _lib.lib().ss2d_dt_proj_f32, x.data_ptr(), weight.data_ptr(), out.data_ptr(), K, D, R, N, x.stride(0),
                     x.stride(1))
    _lib.check(rc, "ss2d_dt_proj_f32")
    return out


def projections_train(x, x_proj_weight, dt_proj_weight):
    """True when XProjF32 and DtProjF32 stand for the two projections of the map x (B, D, H, W) in training: TRAIN_FROM elements of plain
    float32 tensors that the kernels take, and operators that nothing sees.  64 maps of 384 x 14 x 14: x_proj 60 -> 16 us, with the one-by-one CrossScan 5 more before; dt_proj 51 -> 16."""
    return (x.numel() >= TRAIN_FROM and all(type(t) in TENSOR_KINDS and t.dtype == torch.float32 for t in (x, x_proj_weight, dt_proj_weight)) and dt_proj_weight.shape[2] > 0
            and dt_proj_weight.shape[2] <= DT_PROJ_F32_MAX_RANK and x.is_contiguous() and x_proj_f32_fits(x, x_proj_weight)
            and x_proj_f32_pays(x, x_proj_weight) and dt_proj_weight.device == x.device and calls_unseen())


class XProjF32(torch.autograd.Function):
    """x_proj_f32_hip of the map x (B, D, H, W) with weight (4, C, D) -> (B, 4, C, L) in each direction's scan order."""

    @staticmethod
    def forward(ctx, x, weight):
        ctx.save_for_backward(x, weight)
        B, D, H, W = x.shape
        return x_proj_f32_hip(x, weight, x.new_empty((B, 4, weight.shape[1], H * W)))

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        B, D, H, W = x.shape
        K, C = weight.shape[:2]
        # the adjoint of the one-by-one CrossScan, back in the map's order, and the products' own gradients
        d = cross_merge_fn(dy.reshape(B, K, C, H, W), in_channel_first=True, out_channel_first=True, one_by_one=True, scans=0).reshape(B, K * C, H * W)
        dx = torch.bmm(weight.reshape(1, K * C, D).expand(B, -1, -1).transpose(1, 2), d).view(x.shape) if ctx.needs_input_grad[0] else None
        dw = torch.bmm(d, x.reshape(B, D, H * W).transpose(1, 2)).sum(0).view(weight.shape) if ctx.needs_input_grad[1] else None
        return dx, dw


class DtProjF32(torch.autograd.Function):
    """dt_proj_f32_hip: rows (K, R, N) with weight (K, D, R) -> (K, D, N)."""

    @staticmethod
    def forward(ctx, rows, weight):
        ctx.save_for_backward(rows, weight)
        return dt_proj_f32_hip(rows, weight)

    @staticmethod
    def backward(ctx, dy):
        rows, weight = ctx.saved_tensors
        drows = torch.bmm(weight.transpose(1, 2), dy) if ctx.needs_input_grad[0] else None
        return drows, torch.bmm(dy, rows.transpose(1, 2)) if ctx.needs_input_grad[1] else None
