"""Depthwise 3x3 convolution + SiLU in front of the SS2D core, on the HIP kernel ss2d_dwconv3x3_silu.

Mirrors the three lines of SS2Dv2.forwardv2 (classification/models/vmamba.py:654-658): bring the in_proj
output to channel-first, depthwise conv2d, SiLU -- as one kernel that reads either layout and always writes
(B, D, H, W) -- and, for training, the same pair as an autograd function on ss2d_dwconv3x3_silu_bwd.  GPU tensors only.
"""
import torch

from . import _lib
from .csm import transpose_bcl_hip
from .norm import observed

_DTYPE_CODE = {torch.float32: _lib.SS2D_F32, torch.bfloat16: _lib.SS2D_BF16, torch.float16: _lib.SS2D_F16}


def dwconv3x3_silu_hip(x, weight, bias=None, in_channel_last=False, apply_silu=True):
    """x (B,H,W,D) if in_channel_last else (B,D,H,W); weight (D,1,3,3); returns (B,D,H,W)."""
    if not x.is_cuda:
        raise NotImplementedError("dwconv3x3_silu_hip: vmamba_amd runs on the GPU only")
    if x.dim() != 4 or weight.dim() != 4 or tuple(weight.shape[1:]) != (1, 3, 3):
        raise ValueError(f"dwconv3x3_silu_hip: expected a 4-D input and a (D,1,3,3) weight, got {tuple(x.shape)}, {tuple(weight.shape)}")
    if x.dtype not in _DTYPE_CODE:
        raise TypeError(f"dwconv3x3_silu_hip: unsupported dtype {x.dtype}")
    x = x.contiguous()
    if in_channel_last:
        B, H, W, D = x.shape
    else:
        B, D, H, W = x.shape
    if weight.shape[0] != D:
        raise ValueError("dwconv3x3_silu_hip: weight channels do not match the input")
    weight = weight.to(x.dtype).contiguous()
    bias = bias.to(x.dtype).contiguous() if bias is not None else None
    y = torch.empty((B, D, H, W), device=x.device, dtype=x.dtype)
    rc = _lib.launch(x, _lib.lib().ss2d_dwconv3x3_silu, x.data_ptr(), weight.data_ptr(),
                     bias.data_ptr() if bias is not None else None, y.data_ptr(), B, D, H, W, _DTYPE_CODE[x.dtype],
                     int(bool(in_channel_last)), int(bool(apply_silu)))
    _lib.check(rc, "ss2d_dwconv3x3_silu")
    return y


def dwconv3x3_silu_bwd_hip(x, weight, bias, dy):
    """Gradients (dx, dweight, dbias or None) of dwconv3x3_silu_hip on the channel-first x (B,D,H,W) for dy (B,D,H,W)."""
    if not x.is_cuda:
        raise NotImplementedError("dwconv3x3_silu_bwd_hip: vmamba_amd runs on the GPU only")
    B, D, H, W = x.shape
    if tuple(weight.shape) != (D, 1, 3, 3) or dy.shape != x.shape or (bias is not None and tuple(bias.shape) != (D,)):
        raise ValueError("dwconv3x3_silu_bwd_hip: expected weight (D,1,3,3), bias (D) and dy of x's shape")
    if x.dtype not in _DTYPE_CODE or any(t is not None and (t.dtype != x.dtype or t.device != x.device) for t in (weight, bias, dy)):
        raise TypeError("dwconv3x3_silu_bwd_hip: one floating dtype and one device")
    dx, dweight = torch.empty_like(x, memory_format=torch.contiguous_format), torch.empty((D, 1, 3, 3), device=x.device, dtype=x.dtype)
    dbias = torch.empty_like(bias, memory_format=torch.contiguous_format) if bias is not None else None
    if x.numel() == 0:
        return dx, dweight.zero_(), dbias.zero_() if dbias is not None else None
    x, weight, dy = x.contiguous(), weight.contiguous(), dy.contiguous()
    bias = bias.contiguous() if bias is not None else None
    need = _lib.lib().ss2d_dwconv3x3_silu_bwd_workspace_bytes(B, D, H, W)
    _lib.check(min(need, 0), "ss2d_dwconv3x3_silu_bwd_workspace_bytes")
    workspace = torch.empty(need, dtype=torch.uint8, device=x.device)
    rc = _lib.launch(x, _lib.lib().ss2d_dwconv3x3_silu_bwd, x.data_ptr(), weight.data_ptr(),
                     bias.data_ptr() if bias is not None else None, dy.data_ptr(), dx.data_ptr(), dweight.data_ptr(),
                     dbias.data_ptr() if dbias is not None else None, B, D, H, W, _DTYPE_CODE[x.dtype], workspace.data_ptr(),
                     need)
    _lib.check(rc, "ss2d_dwconv3x3_silu_bwd")
    return dx, dweight, dbias


class DwConv3x3SiLU(torch.autograd.Function):
    """dwconv3x3_silu_hip with a gradient: x (B,H,W,D) if ``channel_last`` else (B,D,H,W) -> silu(conv(x)) (B,D,H,W).  First
    order only, as the selective scan behind it is."""

    @staticmethod
    def forward(ctx, x, weight, bias, channel_last):
        if not x.is_cuda:
            raise NotImplementedError("DwConv3x3SiLU: vmamba_amd runs on the GPU only")
        D = x.shape[3 if channel_last else 1]
        if tuple(weight.shape) != (D, 1, 3, 3) or (bias is not None and tuple(bias.shape) != (D,)):
            raise ValueError("DwConv3x3SiLU: expected weight (D,1,3,3) and bias (D)")
        if x.dtype not in _DTYPE_CODE or any(t is not None and (t.dtype != x.dtype or t.device != x.device) for t in (weight, bias)):
            raise TypeError("DwConv3x3SiLU: one floating dtype and one device")
        ctx.channel_last = channel_last
        x = x.contiguous()
        if channel_last:
            B, H, W, D = x.shape
            x = transpose_bcl_hip(x.view(B, H * W, D)).view(B, D, H, W)
        ctx.save_for_backward(x, weight, bias)
        if x.dtype != torch.float32:
            return dwconv3x3_silu_hip(x, weight, bias, in_channel_last=False, apply_silu=True)
        weight, bias = weight.contiguous(), bias.contiguous() if bias is not None else None
        y = torch.empty_like(x)
        rc = _lib.launch(x, _lib.lib().ss2d_dwconv3x3_silu_f32, x.data_ptr(), weight.data_ptr(),
                         bias.data_ptr() if bias is not None else None, y.data_ptr(), *x.shape)
        _lib.check(rc, "ss2d_dwconv3x3_silu_f32")
        return y

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dy):
        x, weight, bias = ctx.saved_tensors
        dx, dweight, dbias = dwconv3x3_silu_bwd_hip(x, weight, bias, dy)
        if ctx.channel_last:
            B, D, H, W = x.shape
            dx = transpose_bcl_hip(dx.view(B, D, H * W)).view(B, H, W, D)
        return dx, dweight, dbias, None


def dwconv_silu_trainable(conv2d, x, channel_last):
    """True when DwConv3x3SiLU stands for silu(conv2d(x)) in training: a plain depthwise 3 x 3 nn.Conv2d (stride 1, zero
    padding 1) called without hooks or autocast on a GPU tensor of its own dtype, on maps the backward kernel takes."""
    if not (type(conv2d) is torch.nn.Conv2d and x.is_cuda and x.dim() == 4 and x.numel() > 0 and x.dtype in _DTYPE_CODE):
        return False
    D, H, W = (x.shape[3], x.shape[1], x.shape[2]) if channel_last else x.shape[1:]
    return (conv2d.kernel_size == (3, 3) and conv2d.padding == (1, 1) and conv2d.stride == (1, 1) and conv2d.dilation == (1, 1)
            and conv2d.padding_mode == "zeros" and conv2d.groups == conv2d.in_channels == conv2d.out_channels == D
            and not observed(conv2d) and not torch.is_autocast_enabled()
            and all(t is None or (t.dtype == x.dtype and t.device == x.device) for t in (conv2d.weight, conv2d.bias))
            and _lib.lib().ss2d_dwconv3x3_silu_bwd_workspace_bytes(x.shape[0], D, H, W) > 0)
