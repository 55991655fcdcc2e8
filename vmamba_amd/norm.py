"""Channel LayerNorm on the HIP kernels of libss2d_hip.so (ss2d_layer_norm / ss2d_layer_norm_cf).

``LayerNorm`` is nn.LayerNorm for (..., C) activations, ``LayerNorm2d`` the reference's channel-first
variant (classification/models/vmamba.py:52-57).  Same parameters (``weight``, ``bias``, ``eps``) as the
torch modules, so state_dicts are interchangeable.  GPU tensors only: there is no CPU path here.
"""
import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

from . import _lib

_DTYPE_CODE = {torch.float32: _lib.SS2D_F32, torch.bfloat16: _lib.SS2D_BF16, torch.float16: _lib.SS2D_F16}


def _params(weight, bias):
    if weight is not None and bias is not None and weight.dtype != bias.dtype:
        bias = bias.to(weight.dtype)
    wdt = weight.dtype if weight is not None else (bias.dtype if bias is not None else torch.float32)
    return (weight.contiguous() if weight is not None else None, bias.contiguous() if bias is not None else None, wdt)


def layer_norm_hip(x, weight, bias, eps=1e-5, out_dtype=None):
    """LayerNorm over the last axis of a contiguous GPU tensor."""
    if not x.is_cuda:
        raise NotImplementedError("layer_norm_hip: vmamba_amd runs on the GPU only")
    x = x.contiguous()
    C = x.shape[-1]
    weight, bias, wdt = _params(weight, bias)
    y = torch.empty(x.shape, device=x.device, dtype=out_dtype or x.dtype)
    rc = _lib.launch(x, _lib.lib().ss2d_layer_norm, x.data_ptr(), weight.data_ptr() if weight is not None else None,
                     bias.data_ptr() if bias is not None else None, y.data_ptr(), x.numel() // max(C, 1), C, eps,
                     _DTYPE_CODE[x.dtype], _DTYPE_CODE[wdt], _DTYPE_CODE[y.dtype])
    _lib.check(rc, "ss2d_layer_norm")
    return y


def add_layer_norm_fusable(x, residual):
    """True when ss2d_add_layer_norm takes these rows (vectorisable: C % 8 == 0, C <= 1024)."""
    C = x.shape[-1]
    return (x.is_cuda and x.dtype in _DTYPE_CODE and residual.dtype == x.dtype and residual.shape == x.shape
            and C % 8 == 0 and C <= 1024)


def add_layer_norm_hip(x, residual, weight, bias, eps=1e-5):
    """(x + residual, LayerNorm(x + residual)) over the last axis in one pass; the sum is rounded to x.dtype first, as
    the separate add would leave it."""
    if not x.is_cuda:
        raise NotImplementedError("add_layer_norm_hip: vmamba_amd runs on the GPU only")
    if residual.shape != x.shape or residual.dtype != x.dtype:
        raise ValueError("add_layer_norm_hip: residual must have the shape and dtype of x")
    x, residual = x.contiguous(), residual.contiguous()
    C = x.shape[-1]
    weight, bias, wdt = _params(weight, bias)
    total, y = torch.empty_like(x), torch.empty_like(x)
    rc = _lib.launch(x, _lib.lib().ss2d_add_layer_norm, x.data_ptr(), residual.data_ptr(),
                     weight.data_ptr() if weight is not None else None, bias.data_ptr() if bias is not None else None,
                     total.data_ptr(), y.data_ptr(), x.numel() // max(C, 1), C, eps, _DTYPE_CODE[x.dtype], _DTYPE_CODE[wdt],
                     _DTYPE_CODE[y.dtype])
    _lib.check(rc, "ss2d_add_layer_norm")
    return total, y


def bias_layer_norm_fusable(dtype, C):
    """True when ss2d_bias_layer_norm takes rows of C channels of this dtype (vectorisable: C % 8 == 0, C <= 1024)."""
    return dtype in _DTYPE_CODE and C % 8 == 0 and C <= 1024


def bias_layer_norm_hip(x, pre_bias, weight, bias, eps=1e-5):
    """LayerNorm(x + pre_bias) over the last axis in one pass, pre_bias one value per channel; the sum is rounded to
    x.dtype first, as the separate add would leave it."""
    if not x.is_cuda:
        raise NotImplementedError("bias_layer_norm_hip: vmamba_amd runs on the GPU only")
    C = x.shape[-1]
    if pre_bias.shape != (C,):
        raise ValueError("bias_layer_norm_hip: pre_bias must hold one value per channel")
    x = x.contiguous()
    weight, bias, wdt = _params(weight, bias)
    pre_bias = pre_bias.to(wdt).contiguous()
    y = torch.empty_like(x)
    rc = _lib.launch(x, _lib.lib().ss2d_bias_layer_norm, x.data_ptr(), pre_bias.data_ptr(),
                     weight.data_ptr() if weight is not None else None, bias.data_ptr() if bias is not None else None,
                     y.data_ptr(), x.numel() // max(C, 1), C, eps, _DTYPE_CODE[x.dtype], _DTYPE_CODE[wdt], _DTYPE_CODE[y.dtype])
    _lib.check(rc, "ss2d_bias_layer_norm")
    return y


def layer_norm_cf_hip(x, weight, bias, eps=1e-5, out_channel_last=False, out_dtype=None):
    """LayerNorm over axis 1 of a channel-first (B, C, *spatial) GPU tensor.

    Returns (B, *spatial, C) when ``out_channel_last`` else (B, C, *spatial)."""
    if not x.is_cuda:
        raise NotImplementedError("layer_norm_cf_hip: vmamba_amd runs on the GPU only")
    x = x.contiguous()
    B, C = x.shape[0], x.shape[1]
    spatial = tuple(x.shape[2:])
    L = 1
    for s in spatial:
        L *= s
    weight, bias, wdt = _params(weight, bias)
    shape = (B, *spatial, C) if out_channel_last else (B, C, *spatial)
    y = torch.empty(shape, device=x.device, dtype=out_dtype or x.dtype)
    rc = _lib.launch(x, _lib.lib().ss2d_layer_norm_cf, x.data_ptr(), weight.data_ptr() if weight is not None else None,
                     bias.data_ptr() if bias is not None else None, y.data_ptr(), B, C, L, eps, _DTYPE_CODE[x.dtype],
                     _DTYPE_CODE[wdt], _DTYPE_CODE[y.dtype], int(bool(out_channel_last)))
    _lib.check(rc, "ss2d_layer_norm_cf")
    return y


def needs_grad(*tensors):
    """True when autograd has to see this call: the HIP LayerNorm / conv kernels are inference kernels, so modules
    route such calls to the differentiable torch operators the reference itself uses."""
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)


def observed(layer):
    """True when something sees or replaces this module's calls -- hooks of its own, global ones, a forward set on the
    instance: a kernel that stands for the module would go past them, so the module has to be called."""
    hooks = (layer._forward_hooks, layer._forward_pre_hooks, layer._backward_hooks, layer._backward_pre_hooks)
    return any(hooks) or nn.modules.module._has_any_global_hook() or "forward" in vars(layer)


# Other kinds of tensors (quantised or sharded weights, subclasses that see the calls they are in) are left to torch's operators.
TENSOR_KINDS = (torch.Tensor, nn.Parameter)


# Elements of the activation from which training in single precision takes this package's own autograd functions for LayerNorm, the MLP and
# the core's projections.  They are Python on the host, up to 10 us a call more than torch's, and a block of fewer elements waits for the host
# -- 1.3 to 1.7 ms a step by box, whatever runs.  A block's step without / with them, us, from 2.1 Mi elements on: 192 x 28 x 28, 16 images (2.3 Mi) 1678 / 1590,
# 384 x 14 x 14, 30 (2.15) 1689 / 1618, 576 x 51 x 38, two (2.13) 1474 / 1392, 736 x 16 x 16, 12 (2.16) 1667 / 1520, 96 x 56 x 56, 8 (2.3) 1713 / 1514; below it goes either way:
# 768 x 7 x 7, 52 (1.87) 1644 / 1698, 736 x 16 x 16, 8 (1.44) 1331 / 1374, 384 x 14 x 14, 20 (1.44) 1653 / 1652, 192 x 28 x 28, 12 (1.72) 1674 / 1595, 576 x 51 x 38, one (1.06) 1285 / 1320.
TRAIN_FROM = 2 << 20


def layer_norm_trains(x, normalized_shape, weight, bias, C=None):
    """True when LayerNormF32 stands for F.layer_norm over the C channels of x (default: its last axis) in training: float32 on the GPU, a
    multiple of 4 channels up to 1024, TRAIN_FROM elements, and operators that nothing sees."""
    if C is None:
        C = x.shape[-1] if x.dim() else 0
    return (type(x) in TENSOR_KINDS and x.is_cuda and x.dtype == torch.float32 and x.numel() >= TRAIN_FROM and tuple(normalized_shape) == (C,) and C % 4 == 0
            and C <= 1024 and all(t is None or (type(t) in TENSOR_KINDS and t.dtype == x.dtype and t.device == x.device and t.is_contiguous()
                                                and t.data_ptr() % 16 == 0) for t in (weight, bias)) and calls_unseen())


def memory_readable(*tensors):
    """True where a backward may hand these tensors (or None) to a kernel by their addresses: memory of their own -- a batch of gradients under
    is_grads_batched or a vectorised jacobian has none, nor does another kind of tensor, and a negated view's is another -- and operators that
    nothing sees now, whatever saw them in the forward."""
    return not operators_seen() and all(t is None or (type(t) in TENSOR_KINDS and torch._C._has_storage(t) and not t.is_neg()) for t in tensors)


class LayerNormF32(torch.autograd.Function):
    """F.layer_norm over the last axis with its backward on ss2d_layer_norm_bwd_f32, which computes the statistics again from x."""

    @staticmethod
    def forward(ctx, x, weight, bias, eps):
        ctx.save_for_backward(x, weight)
        ctx.eps = eps
        return layer_norm_hip(x, weight, bias, eps)

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        wants = ctx.needs_input_grad
        C = x.shape[-1]
        if torch.is_grad_enabled() or not memory_readable(x, weight, dy):          # a second backward goes through the torch operators
            mean = x.mean(-1, keepdim=True)
            centred = x - mean
            rstd = (centred.square().mean(-1, keepdim=True) + ctx.eps).rsqrt()
            xhat, g = centred * rstd, dy if weight is None else dy * weight
            dx = rstd * (g - g.mean(-1, keepdim=True) - xhat * (g * xhat).mean(-1, keepdim=True)) if wants[0] else None
            return dx, (dy * xhat).reshape(-1, C).sum(0) if wants[1] else None, dy.reshape(-1, C).sum(0) if wants[2] else None, None
        x, dy = x.contiguous(), dy.contiguous()
        if (x.data_ptr() | dy.data_ptr()) % 16:                      # (views between 16-byte boundaries)
            x, dy = x.clone(), dy.clone()
        dx = torch.empty_like(x) if wants[0] else None
        dw, db = (torch.empty(C, dtype=x.dtype, device=x.device) if want else None for want in wants[1:3])
        L = _lib.lib()
        need = L.ss2d_layer_norm_bwd_f32_workspace_bytes(C)
        workspace = torch.empty(need, dtype=torch.uint8, device=x.device)
        ptr = lambda t: None if t is None else t.data_ptr()
        rc = _lib.launch(x, L.ss2d_layer_norm_bwd_f32, x.data_ptr(), dy.data_ptr(), ptr(weight), ctx.eps, ptr(dx), ptr(dw), ptr(db), x.numel() // C, C,
                         workspace.data_ptr(), need)
        _lib.check(rc, "ss2d_layer_norm_bwd_f32")
        return dx, dw, db, None


def column_sums(x):
    """x.sum(0) of a float32 matrix (ss2d_column_sums_f32; the library's where autograd or something else follows or the kernel has no variant)."""
    if torch.is_grad_enabled() or not memory_readable(x) or x.dtype != torch.float32 or not x.is_contiguous() or x.numel() == 0 or x.shape[1] % 4 or x.data_ptr() % 16:
        return x.sum(0)
    rows, N = x.shape
    out = torch.empty(N, dtype=x.dtype, device=x.device)
    L = _lib.lib()
    need = L.ss2d_column_sums_f32_workspace_bytes(N)
    workspace = torch.empty(need, dtype=torch.uint8, device=x.device)
    _lib.check(_lib.launch(x, L.ss2d_column_sums_f32, x.data_ptr(), out.data_ptr(), rows, N, workspace.data_ptr(), need), "ss2d_column_sums_f32")
    return out


def _gpu_only(x, what):
    if not x.is_cuda:
        raise NotImplementedError(f"{what}: vmamba_amd runs on the GPU only (got a {x.device.type} tensor)")


class LayerNorm(nn.LayerNorm):
    def forward(self, x):
        _gpu_only(x, "LayerNorm")
        if needs_grad(x, self.weight, self.bias):
            if layer_norm_trains(x, self.normalized_shape, self.weight, self.bias):
                return LayerNormF32.apply(x, self.weight, self.bias, self.eps)
            return F.layer_norm(x, self.normalized_shape, self.weight, self.bias, self.eps)
        return layer_norm_hip(x, self.weight, self.bias, self.eps)


class LayerNorm2d(nn.LayerNorm):
    def forward(self, x):
        _gpu_only(x, "LayerNorm2d")
        if needs_grad(x, self.weight, self.bias):          # vmamba.py:52-57
            return F.layer_norm(x.permute(0, 2, 3, 1), self.normalized_shape, self.weight, self.bias, self.eps).permute(0, 3, 1, 2)
        return layer_norm_cf_hip(x, self.weight, self.bias, self.eps, out_channel_last=False)


_MODES = torch._C._len_torch_dispatch_stack, torch._C._functorch.peek_interpreter_stack, torch._C._len_torch_function_stack


def _calls():
    return nn.Linear.forward, nn.GELU.forward, LayerNorm.forward, F.linear, F.gelu, F.layer_norm


_CALLS = _calls()


def operators_seen():
    """True when the operators that modules call may be seen or replaced, so that a kernel standing for library calls would go past
    it: an active TorchDispatchMode or TorchFunctionMode (flop counters, loggers; not the one behind torch.device and
    set_default_device, which only looks at factories), forward-mode derivatives, torch.func's transforms, or another forward or
    function in the place of torch's or this package's own."""
    dispatch, transforms, functions = _MODES
    if dispatch() or forward_ad._current_level >= 0 or transforms() is not None or _calls() != _CALLS:
        return True
    modes = functions()
    return modes > 0 and any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(modes))


def native_stands(x):
    """True where an operator on x may make and look at its tensors in _lib.host(): nobody who follows its calls expects them from Python."""
    return type(x) in TENSOR_KINDS and x.is_cuda and not torch.compiler.is_compiling() and not operators_seen()


def calls_unseen():
    """True when nothing but autograd follows the operators that are called: no mode or transform (operators_seen), no compiler or tracer."""
    return not (torch.compiler.is_compiling() or torch.jit.is_tracing() or operators_seen() or torch.is_autocast_enabled())
