"""The patch embedding's two layers as one HIP kernel each: Conv2d(3, C, 3, stride 2, padding 1) -> LayerNorm(C) -> GELU
(ss2d_stem_conv_ln_gelu) and Conv2d(48, 96, 3, stride 2, padding 1) -> LayerNorm(96) (ss2d_stem_conv2_ln) on channel-last
activations (classification/models/vmamba.py:1403-1416); and the convolutions between the stages (:1430-1437) on ss2d_conv3x3s2_cl."""
import ctypes

import torch
import torch.nn as nn

from . import _lib
from .linear import TENSOR_KINDS, calls_unseen

_DTYPE_CODE = {torch.bfloat16: _lib.SS2D_BF16, torch.float16: _lib.SS2D_F16}
STEM_WIDTHS = (48, 64)


def stem_fusable(x, conv, norm, act):
    """True when the kernel serves this conv / norm / activation triple on x."""
    return (x.is_cuda and x.dim() == 4 and x.dtype in _DTYPE_CODE and conv.in_channels == 3 and x.shape[1] == 3
            and conv.out_channels in STEM_WIDTHS and tuple(conv.kernel_size) == (3, 3) and tuple(conv.stride) == (2, 2)
            and tuple(conv.padding) == (1, 1) and tuple(conv.dilation) == (1, 1) and conv.groups == 1
            and conv.padding_mode == "zeros" and conv.weight.dtype == x.dtype
            and tuple(norm.normalized_shape) == (conv.out_channels,) and norm.elementwise_affine
            and norm.weight.dtype == x.dtype and getattr(act, "approximate", "none") == "none")


def stem_conv_ln_gelu_hip(x, weight, bias, ln_weight, ln_bias, eps=1e-5):
    """GELU(LayerNorm(conv2d(x, weight, bias, stride 2, padding 1))) for x (B, 3, H, W): returns the channel-last
    activation (B, Ho, Wo, C).  The weight is read through its strides (contiguous or channels-last)."""
    if not x.is_cuda:
        raise NotImplementedError("stem_conv_ln_gelu: vmamba_amd runs on the GPU only")
    if x.dim() != 4 or x.shape[1] != 3 or weight.dim() != 4 or tuple(weight.shape[1:]) != (3, 3, 3):
        raise ValueError("stem_conv_ln_gelu expects x (B, 3, H, W) and weight (C, 3, 3, 3)")
    if x.dtype not in _DTYPE_CODE or weight.dtype != x.dtype:
        raise RuntimeError("stem_conv_ln_gelu: bf16 or fp16 tensors")
    x = x.contiguous()
    B, _, H, W = x.shape
    C = weight.shape[0]
    cast = lambda t: None if t is None else t.to(x.dtype).contiguous()
    bias, ln_weight, ln_bias = cast(bias), cast(ln_weight), cast(ln_bias)
    ptr = lambda t: None if t is None else t.data_ptr()
    y = torch.empty((B, (H - 1) // 2 + 1, (W - 1) // 2 + 1, C), device=x.device, dtype=x.dtype)
    strides = (ctypes.c_int64 * 4)(*weight.stride())
    rc = _lib.launch(x, _lib.lib().ss2d_stem_conv_ln_gelu, x.data_ptr(), weight.data_ptr(), strides, ptr(bias), ptr(ln_weight),
                     ptr(ln_bias), eps, y.data_ptr(), B, H, W, C, _DTYPE_CODE[x.dtype])
    _lib.check(rc, "ss2d_stem_conv_ln_gelu")
    return y


STEM2_SHAPE = (48, 96)
_STEM2_MAX_BYTES = 0x7f000000             # the kernel's offsets into the input are 31 bits


def stem2_fusable(x, conv, norm):
    """True when ss2d_stem_conv2_ln serves this conv / norm pair on x (B, 48, H, W), channel-last in memory: a convolution that
    computes what nn.Conv2d does, in x's own type."""
    own = type(conv)._conv_forward is not nn.Conv2d._conv_forward or "_conv_forward" in vars(conv)
    if own or (torch.is_autocast_enabled() and torch.get_autocast_dtype("cuda") != x.dtype):
        return False
    return (x.is_cuda and x.dim() == 4 and x.dtype in _DTYPE_CODE and x.shape[1] == conv.in_channels
            and (conv.in_channels, conv.out_channels) == STEM2_SHAPE and tuple(conv.kernel_size) == (3, 3)
            and tuple(conv.stride) == (2, 2) and tuple(conv.padding) == (1, 1) and tuple(conv.dilation) == (1, 1)
            and conv.groups == 1 and conv.padding_mode == "zeros" and conv.weight.dtype == x.dtype
            and tuple(norm.normalized_shape) == (conv.out_channels,) and norm.elementwise_affine and norm.weight.dtype == x.dtype
            and 0 < x.numel() < _STEM2_MAX_BYTES // 2 and x.permute(0, 2, 3, 1).is_contiguous() and x.data_ptr() % 16 == 0)


def stem_conv2_ln_hip(x, weight, bias, ln_weight, ln_bias, eps=1e-5):
    """LayerNorm(conv2d(x, weight, bias, stride 2, padding 1)) for x (B, H, W, 48) channel-last, weight (96, 48, 3, 3) with any
    strides: returns (B, Ho, Wo, 96)."""
    if not x.is_cuda:
        raise NotImplementedError("stem_conv2_ln: vmamba_amd runs on the GPU only")
    if x.dim() != 4 or weight.dim() != 4 or tuple(weight.shape[1:]) != (x.shape[3], 3, 3):
        raise ValueError("stem_conv2_ln expects x (B, H, W, Cin) and weight (C, Cin, 3, 3)")
    if x.dtype not in _DTYPE_CODE or weight.dtype != x.dtype or weight.device != x.device:
        raise RuntimeError("stem_conv2_ln: bf16 or fp16 tensors on one device")
    x = x.contiguous()
    B, H, W, Cin = x.shape
    C = weight.shape[0]
    small = [None if t is None else t.to(x.dtype).contiguous() for t in (bias, ln_weight, ln_bias)]
    if any(t is not None and (t.shape != (C,) or t.device != x.device) for t in small):
        raise ValueError("stem_conv2_ln: bias and LayerNorm parameters must hold one value per output channel")
    ptr = [None if t is None else t.data_ptr() for t in small]
    y = torch.empty((B, (H - 1) // 2 + 1, (W - 1) // 2 + 1, C), device=x.device, dtype=x.dtype)
    strides = (ctypes.c_int64 * 4)(*weight.stride())
    rc = _lib.launch(x, _lib.lib().ss2d_stem_conv2_ln, x.data_ptr(), weight.data_ptr(), strides, *ptr, eps, y.data_ptr(), B, H, W,
                     Cin, C, _DTYPE_CODE[x.dtype])
    _lib.check(rc, "ss2d_stem_conv2_ln")
    return y


def conv_tiles_fusable(x, conv):
    """True when ss2d_conv3x3s2_cl stands for this convolution's product at inference on x (B, C, H, W), channel-last in memory, and is the
    faster one: a plain 3 x 3 convolution of stride 2 in x's own type whose operators nothing sees."""
    if type(x) not in TENSOR_KINDS or x.dtype not in _DTYPE_CODE or not x.is_cuda or x.dim() != 4 or type(conv) is not nn.Conv2d or "_conv_forward" in vars(conv):
        return False
    B, C, H, W = x.shape
    return (conv_tiles_pays(B * ((H + 1) // 2) * ((W + 1) // 2), C) and C == conv.in_channels and C % 32 == 0 and conv.out_channels % 8 == 0
            and tuple(conv.kernel_size) == (3, 3) and tuple(conv.stride) == (2, 2) and tuple(conv.padding) == (1, 1) and tuple(conv.dilation) == (1, 1)
            and conv.groups == 1 and conv.padding_mode == "zeros" and type(conv.weight) in TENSOR_KINDS and conv.weight.dtype == x.dtype
            and conv.weight.device == x.device and (nn.Conv2d._conv_forward, nn.functional.conv2d) == _CONV_CALLS and calls_unseen()
            and x.permute(0, 2, 3, 1).is_contiguous() and x.data_ptr() % 16 == 0)


_CONV_CALLS = nn.Conv2d._conv_forward, nn.functional.conv2d


def conv_tiles_pays(M, C):
    """True from the number of output positions on where ss2d_conv3x3s2_cl, with the copy of its weights into (N, 3, 3, C), is ahead of the
    library.  us in bf16, library / kernel, C -> 2 C: 96 at 6272 positions 24 / 24, at 12 544 29 / 24, at 100 352 93 + 36 / 60; 192 at 784 32 / 39, at 3136
    42 / 39, at 25 088 93 / 43; 384 at 784 66 / 69, at 3136 82 / 69, at 6272 134 / 72.  Fewer positions leave a workgroup alone with 9 C terms."""
    return M >= (3136 if C >= 192 else 6272)


def conv_tiles_hip(x, weight, bias=None):
    """conv2d(x, weight, bias, stride 2, padding 1) for x (B, H, W, C) channel-last, weight (N, C, 3, 3) with any strides: (B, Ho, Wo, N)."""
    if not x.is_cuda:
        raise NotImplementedError("conv_tiles_hip: vmamba_amd runs on the GPU only")
    if x.dim() != 4 or weight.dim() != 4 or tuple(weight.shape[1:]) != (x.shape[3], 3, 3):
        raise ValueError("conv_tiles_hip expects x (B, H, W, C) and weight (N, C, 3, 3)")
    if x.dtype not in _DTYPE_CODE or weight.dtype != x.dtype or weight.device != x.device:
        raise RuntimeError("conv_tiles_hip: bf16 or fp16 tensors on one device")
    x, w = x.contiguous(), weight.permute(0, 2, 3, 1).contiguous()
    B, H, W, C = x.shape
    N = weight.shape[0]
    bias = None if bias is None else bias.to(x.dtype).contiguous()
    if bias is not None and (bias.shape != (N,) or bias.device != x.device):
        raise ValueError("conv_tiles_hip: one bias value per output channel")
    y = x.new_empty((B, (H + 1) // 2, (W + 1) // 2, N))
    rc = _lib.launch(x, _lib.lib().ss2d_conv3x3s2_cl, x.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), y.data_ptr(), B, H, W, C, N,
                     _DTYPE_CODE[x.dtype])
    _lib.check(rc, "ss2d_conv3x3s2_cl")
    return y
