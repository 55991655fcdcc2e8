"""A channel-last VSS block of few positions as one call into the library (ss2d_block_fwd): LayerNorm + in_proj, depthwise
convolution + SiLU, forward_core, out_proj + add, and with fewer still LayerNorm + fc1 + GELU, fc2 + add (classification/models/vmamba.py:1225-1229).

The kernels and results are those of the separate calls, but for out_proj at width 96 on more than 24 576 positions
of maps that are no multiple of 32 (ss2d_linear_rows here, ss2d_linear_cl there); the host's share of a block goes from 100-120 us to about 40, which is what a
model on a few images waits for.
"""
from operator import attrgetter

import torch
import torch.nn as nn

from . import _lib
from .core import core_fits, padded_map_size
from .linear import _DTYPE_CODE, TENSOR_KINDS, LINEAR_ROWS_MOST, linear_rows_pays
from .norm import LayerNorm, operators_seen
from .ss2d import SS2D, HipLayers

# what the call stands for: replaced on the class or the instance, they are called instead
_STEPS = ("forward", "forward_core", "forward_core_fused", "finish_core", "_inference_constants", "_forward_core_native")
_class_steps = attrgetter(*_STEPS)
_CLASS_STEPS = _class_steps(SS2D)
_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")


def _plain(module, cls):
    """True for a module of exactly this class whose calls nothing sees or replaces."""
    if type(module) is not cls:
        return False
    own = vars(module)
    return "forward" not in own and not any(own[name] for name in _HOOKS)


def vss_block_hip(block, mlp_cls, x, residual=None):
    """``block`` on x (B, H, W, C) as one call: (block(x), True), or (x + op(norm(x)), False) where the MLP has too many positions for
    it; with ``residual``, x is norm(residual) already.  None where that does not stand for its modules: autograd, autocast or operators
    that something sees, layers of other kinds, types, sizes or memory, too many positions (linear_rows_pays), a map that has to be padded."""
    code = _DTYPE_CODE.get(x.dtype)
    if (code is None or torch.is_grad_enabled() or not x.is_cuda or x.dim() != 4 or not x.is_contiguous() or torch.is_autocast_enabled()
            or nn.modules.module._has_any_global_hook() or operators_seen()):
        return None
    B, H, W, C = x.shape
    M = B * H * W
    if not 0 < M * C * C <= LINEAR_ROWS_MOST:
        return None
    get = block._modules.get
    op, mlp, norm, norm2 = get("op"), get("mlp"), get("norm"), get("norm2")
    if not (_plain(op, SS2D) and _plain(mlp, mlp_cls) and _plain(norm, LayerNorm) and _plain(norm2, LayerNorm)):
        return None
    if (op.layers is not HipLayers or op.channel_first or mlp.channel_first or not mlp.fused or not op.fused_core or not op.disable_z
            or op.d_state != 1 or not vars(op).keys().isdisjoint(_STEPS) or _class_steps(SS2D) != _CLASS_STEPS):
        return None
    get = op._modules.get
    in_proj, conv, out_norm, out_proj = get("in_proj"), get("conv2d"), get("out_norm"), get("out_proj")
    get = mlp._modules.get
    fc1, act, fc2 = get("fc1"), get("act"), get("fc2")
    if not (all(_plain(layer, nn.Linear) for layer in (in_proj, out_proj, fc1, fc2)) and _plain(conv, nn.Conv2d) and _plain(out_norm, LayerNorm)
            and _plain(act, nn.GELU) and act.approximate == "none"):
        return None
    layers = (in_proj, out_proj, fc1, fc2, norm, norm2, out_norm, conv)
    weight = tuple([layer._parameters.get("weight") for layer in layers])
    bias = tuple([layer._parameters.get("bias") for layer in layers])
    own = op._parameters
    x_proj, dt_proj = own.get("x_proj_weight"), own.get("dt_projs_weight")
    if weight[0] is None or weight[2] is None or dt_proj is None:
        return None
    D, hidden = weight[0].shape[0], weight[2].shape[0]
    if (norm.normalized_shape != (C,) or norm2.normalized_shape != (C,) or out_norm.normalized_shape != (D,)
            or conv.padding != (1, 1) or conv.stride != (1, 1) or conv.dilation != (1, 1) or conv.padding_mode != "zeros"
            or C % 16 or D % 16 or hidden % 16 or C > 768 or D > 3072 or hidden > 3072 or M * D * C > LINEAR_ROWS_MOST
            or not core_fits(H, W, x.dtype) or padded_map_size(H, W, x.dtype) is not None):
        return None
    whole = linear_rows_pays(M, hidden, C)
    consts = op._inference_constants(0)
    out = _lib.host().block(TENSOR_KINDS, x, residual, weight, bias, x_proj, dt_proj, consts["As"], consts["Ds"], consts["dt_bias"],
                            (norm.eps, norm2.eps, out_norm.eps), whole)
    if out is None:
        return None
    if type(out) is int:
        _lib.check(out, "ss2d_block_fwd")
    return out, whole
