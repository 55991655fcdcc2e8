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
    weight = [layer._parameters.get("weight") for layer in (in_proj, out_proj, fc1, fc2, norm, norm2, out_norm, conv)]
    bias = [layer._parameters.get("bias") for layer in (in_proj, out_proj, fc1, fc2, norm, norm2, out_norm, conv)]
    own = op._parameters
    x_proj, dt_proj = own.get("x_proj_weight"), own.get("dt_projs_weight")
    index = x.get_device()
    if residual is not None and residual.shape != x.shape:
        return None
    for t in (x, x if residual is None else residual, x_proj, dt_proj, *weight):
        if t is None or type(t) not in TENSOR_KINDS or t.dtype != x.dtype or t.get_device() != index or not t.is_contiguous() or t.data_ptr() % 16:
            return None
    w_in, w_out, w_1, w_2, w_n1, w_n2, w_on, w_c = weight
    D, hidden, R = w_in.shape[0], w_1.shape[0], dt_proj.shape[2]
    for t, n in zip(bias, (D, C, hidden, C, C, C, D, D)):           # (torch would broadcast one of another size)
        if t is not None and (type(t) not in TENSOR_KINDS or t.numel() != n or t.dtype != x.dtype or t.get_device() != index
                              or not t.is_contiguous() or t.data_ptr() % 16):
            return None
    if (tuple(w_in.shape) != (D, C) or tuple(w_out.shape) != (C, D) or tuple(w_1.shape) != (hidden, C) or tuple(w_2.shape) != (C, hidden)
            or norm.normalized_shape != (C,) or norm2.normalized_shape != (C,) or out_norm.normalized_shape != (D,)
            or w_n1.numel() != C or w_n2.numel() != C or w_on.numel() != D
            or tuple(w_c.shape) != (D, 1, 3, 3) or tuple(x_proj.shape) != (4, R + 2, D) or tuple(dt_proj.shape) != (4, D, R) or R == 0
            or conv.padding != (1, 1) or conv.stride != (1, 1) or conv.dilation != (1, 1) or conv.padding_mode != "zeros"):
        return None
    if (C % 16 or D % 16 or hidden % 16 or C > 768 or D > 3072 or hidden > 3072 or M * D * C > LINEAR_ROWS_MOST
            or not core_fits(H, W, x.dtype) or padded_map_size(H, W, x.dtype) is not None):
        return None
    whole = linear_rows_pays(M, hidden, C)
    consts = op._inference_constants(0)
    As, Ds, dt_bias = consts["As"], consts["Ds"], consts["dt_bias"]
    for t in (As, Ds, dt_bias):
        if t.get_device() != index or t.numel() != 4 * D or not t.is_contiguous():
            return None
    out = torch.empty_like(x)
    ptr = [None if t is None else t.data_ptr() for t in bias]
    p = _lib.BlockParams(
        _lib.ForwardCoreParams(B, D, H, W, R, H, W, code, code, 1, 1, out_norm.eps, None, x_proj.data_ptr(), dt_proj.data_ptr(), As.data_ptr(),
                               Ds.data_ptr(), dt_bias.data_ptr(), w_on.data_ptr(), ptr[6], None, None),
        C, hidden, norm.eps, norm2.eps, x.data_ptr(), None if residual is None else residual.data_ptr(),
        w_n1.data_ptr() if residual is None else None, ptr[4] if residual is None else None, w_in.data_ptr(), ptr[0], w_c.data_ptr(), ptr[7],
        w_out.data_ptr(), ptr[1], w_n2.data_ptr(), ptr[5], w_1.data_ptr() if whole else None,
        ptr[2], w_2.data_ptr() if whole else None, ptr[3], out.data_ptr())
    L = _lib.lib()
    need = L.ss2d_block_workspace_bytes(p)
    if need == _lib.SS2D_ENOTSUP:
        return None
    _lib.check(min(need, 0), "ss2d_block_workspace_bytes")
    workspace = torch.empty(need, dtype=torch.uint8, device=x.device)
    rc = _lib.launch(x, L.ss2d_block_fwd, p, workspace.data_ptr(), need)
    if rc == _lib.SS2D_ENOTSUP:
        return None
    _lib.check(rc, "ss2d_block_fwd")
    return out, whole
