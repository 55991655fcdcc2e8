"""Narrow channel-last projection on the HIP kernel ss2d_linear_cl: out = [LayerNorm](x) W^T + bias + residual.

Stands in, in a channel-last VSS block of width 96, for norm + in_proj and for out_proj + the residual add
(classification/models/vmamba.py:1225-1228, :648-650, :662) at inference in bf16 / fp16; other widths and fp32
stay on the PyTorch-ROCm operators.  In single-precision training the weight gradient of these projections is a HIP kernel
(ss2d_linear_dw_f32) where that is the faster one.
"""
import torch
import torch.nn as nn

from . import _lib
from .norm import LayerNorm, needs_grad, observed, operators_seen

_DTYPE_CODE = {torch.bfloat16: _lib.SS2D_BF16, torch.float16: _lib.SS2D_F16}
FUSED_SHAPES = ((96, 96),)            # (in_features, out_features)


def linear_fusable(x, weight):
    """True when ss2d_linear_cl takes this call."""
    return (x.is_cuda and x.dtype in _DTYPE_CODE and weight.dtype == x.dtype and weight.dim() == 2
            and (x.shape[-1], weight.shape[0]) in FUSED_SHAPES and weight.shape[1] == x.shape[-1])


def linear_cl_hip(x, weight, bias=None, residual=None, ln_weight=None, ln_bias=None, eps=1e-5):
    """x (..., K) channel-last, weight (N, K); returns [layer_norm(x)] @ weight.T + bias + residual, shape (..., N)."""
    if not x.is_cuda:
        raise NotImplementedError("linear_cl_hip: vmamba_amd runs on the GPU only")
    if x.dtype not in _DTYPE_CODE:
        raise TypeError(f"linear_cl_hip: unsupported dtype {x.dtype}")
    K = x.shape[-1]
    if weight.dim() != 2 or weight.shape[1] != K:
        raise ValueError(f"linear_cl_hip: weight must be (N, {K}), got {tuple(weight.shape)}")
    N = weight.shape[0]
    x = x.contiguous()
    out = torch.empty(x.shape[:-1] + (N,), device=x.device, dtype=x.dtype)
    if residual is not None and (residual.shape != out.shape or residual.dtype != x.dtype):
        raise ValueError("linear_cl_hip: residual must have the shape and dtype of the result")
    small = [None if t is None else t.to(x.dtype).contiguous() for t in (ln_weight, ln_bias, bias)]
    keep = [weight.contiguous(), None if residual is None else residual.contiguous()]
    ptr = lambda t: None if t is None else t.data_ptr()
    rc = _lib.launch(x, _lib.lib().ss2d_linear_cl, x.data_ptr(), ptr(small[0]), ptr(small[1]), float(eps), keep[0].data_ptr(),
                     ptr(small[2]), ptr(keep[1]), out.data_ptr(), x.numel() // K, K, N, _DTYPE_CODE[x.dtype])
    _lib.check(rc, "ss2d_linear_cl")
    return out


# Other kinds of tensors (quantised or sharded weights, subclasses that see the calls they are in) are left to torch's operators.
TENSOR_KINDS = (torch.Tensor, nn.Parameter)


def _rows_params(x, *params):
    """True for (tensor or None, elements) whose memory the kernels can read as it is; a bias that torch would broadcast is not."""
    return all(t is None or (type(t) in TENSOR_KINDS and t.dtype == x.dtype and t.device == x.device and t.numel() == n and t.is_contiguous()
                             and t.data_ptr() % 16 == 0) for t, n in params)


def linear_rows_takes(layer, x):
    """True when ss2d_linear_rows stands for this layer at inference on rows of x's type and device: a plain nn.Linear that nothing
    observes, its parameters of x's own 16-bit dtype, and operators that nothing sees."""
    if type(layer) is not nn.Linear or type(x) not in TENSOR_KINDS or not x.is_cuda or x.dtype not in _DTYPE_CODE or operators_seen():
        return False
    N, K = layer.weight.shape
    return (K % 16 == 0 and 0 < K <= 3072 and N % 8 == 0 and _rows_params(x, (layer.weight, N * K), (layer.bias, N))
            and not needs_grad(x, layer.weight, layer.bias) and not observed(layer) and not torch.is_autocast_enabled())


def linear_rows_fusable(x, layer, norm=None):
    """True when ss2d_linear_rows takes ``layer(x)`` -- ``layer(norm(x))`` with a norm of this package -- and has few enough
    positions to be the faster one (linear_rows_pays)."""
    K = x.shape[-1]
    if type(layer) is not nn.Linear or K == 0 or not linear_rows_pays(x.numel() // K, layer.out_features, K):
        return False
    if not (linear_rows_takes(layer, x) and tuple(layer.weight.shape) == (layer.out_features, K) and x.is_contiguous() and x.data_ptr() % 16 == 0):
        return False
    return norm is None or (type(norm) is LayerNorm and norm.normalized_shape == (K,) and K <= 768 and norm.weight is not None
                            and _rows_params(x, (norm.weight, K), (norm.bias, K)) and not needs_grad(norm.weight, norm.bias) and not observed(norm))


LINEAR_ROWS_MOST = 448 << 20             # M N K of a projection


def few_positions(x):
    """False where no square product of x's type and width can be linear_rows': asked first, so that others pay for nothing else."""
    return x.dtype in _DTYPE_CODE and x.numel() * x.shape[-1] <= LINEAR_ROWS_MOST


def linear_rows_pays(M, N, K):
    """True up to the number of positions where ss2d_linear_rows falls behind what else takes this product.  Its time is 3-5 us for
    the launch and then grows with M N K, every 32 x 32 tile reading its operands from the L2.  Replayed from graphs, us, in bf16,
    with LayerNorm or residual on both sides: 96 -> 96 at 12 544 positions 5.0 against ss2d_linear_cl's 8.0; 192 -> 192 at 3136
    6.0 against the library's 8.6, at 12 544 14.3 / 12.0; 384 -> 384 at 784 6.5 / 9.0, at 1568 8.9 / 9.8, at 3136 13.3 / 11.5;
    768 -> 768 at 196 7.2 / 9.8, at 400 10.6 / 10.2, at 784 15.3 / 11.4.  The rule lies up to 4 us a product beyond the crossing:
    the library's call takes 24 us on the host, and a model on up to 16 images waits for that (3090 us a pass whose kernels run for 1700).
    Replayed from a graph nothing waits, and the rule is the same there, so that a replay has the eager call's bits: two blocks of
    768 x 7 x 7 214 -> 219 at 16 images (eager 405 -> 271), 200 -> 199 at 12.  The MLP (fc1 is asked for, four outputs per input) has fewer
    passes around it to win back: 384 at 400 17.6 / 23.7, at 784 27.5 / 27.5, at 1568 43 / 35; 768 at 49 20.6 / 24.9, at 196 30.2 / 26.4, where the
    host's share (two launches for four library calls of 24 us and two of the package's) still decides.  Widths 96 and 192 have
    ss2d_mlp_fused, whose 128 positions per workgroup leave the chip idle below: 192 at 784 12.1 / 45.2, at 3136 27.2 / 45.5, at
    6272 44.6 / 45.8; 96 at 6272 15.5 / 17.8, at 12 544 25.3 / 18.0."""
    if N >= 4 * K:
        return 0 < M <= 6144 if K <= 192 else 0 < M * N * K <= 480 << 20
    if N == K == 96:                     # ss2d_linear_cl's: with the LayerNorm 7.0 / 8.3 at 25 088, 8.8 / 8.5 at 31 360
        return 0 < M <= 24576
    return 0 < M * N * K <= LINEAR_ROWS_MOST


def linear_rows_hip(x, weight, bias=None, residual=None, ln_weight=None, ln_bias=None, eps=1e-5, gelu=False):
    """x (..., K) channel-last, weight (N, K), one 16-bit dtype: [gelu]([layer_norm(x)] @ weight.T + bias) + residual, shape
    (..., N), for few positions (ss2d_linear_rows)."""
    if not x.is_cuda:
        raise NotImplementedError("linear_rows_hip: vmamba_amd runs on the GPU only")
    if x.dtype not in _DTYPE_CODE:
        raise TypeError(f"linear_rows_hip: unsupported dtype {x.dtype}")
    K = x.shape[-1]
    if weight.dim() != 2 or weight.shape[1] != K:
        raise ValueError(f"linear_rows_hip: weight must be (N, {K}), got {tuple(weight.shape)}")
    N = weight.shape[0]
    for t, n in ((weight, N * K), (bias, N), (ln_weight, K), (ln_bias, K)):
        if t is not None and (t.dtype != x.dtype or t.device != x.device or t.numel() != n or not t.is_contiguous()):
            raise ValueError("linear_rows_hip: contiguous parameters of x's dtype on its device")
    x = x.contiguous()
    out = x.new_empty(x.shape[:-1] + (N,))
    if residual is not None:
        if residual.shape != out.shape or residual.dtype != x.dtype or residual.device != x.device:
            raise ValueError("linear_rows_hip: residual must have the shape, dtype and device of the result")
        residual = residual.contiguous()
    ptr = lambda t: None if t is None else t.data_ptr()
    rc = _lib.launch(x, _lib.lib().ss2d_linear_rows, x.data_ptr(), ptr(ln_weight), ptr(ln_bias), float(eps), weight.data_ptr(),
                     ptr(bias), ptr(residual), out.data_ptr(), x.numel() // K, K, N, int(gelu), _DTYPE_CODE[x.dtype])
    _lib.check(rc, "ss2d_linear_rows")
    return out


def linear_cf_ln_fusable(K, weight, L):
    """True when ss2d_linear_cf_ln takes an fp32 channel-first map (B, K, L) with this 16-bit GPU weight (N, K)."""
    return (weight.is_cuda and weight.dtype in _DTYPE_CODE and weight.dim() == 2 and weight.shape[1] == K
            and (K, weight.shape[0]) in FUSED_SHAPES and L % 32 == 0)


def linear_cf_ln_hip(y, ln_weight, ln_bias, eps, weight, bias=None, residual=None):
    """y (B, K, L) fp32 channel-first (the merged output of the SS2D core), weight (N, K) bf16 / fp16: returns
    layer_norm(y over K, computed in fp32, rounded to the weight's dtype) @ weight.T + bias + residual as the
    channel-last tensor (B, L, N) -- out_norm and out_proj of the block (vmamba.py:641-646, :662) in one kernel."""
    if not y.is_cuda:
        raise NotImplementedError("linear_cf_ln_hip: vmamba_amd runs on the GPU only")
    if y.dtype != torch.float32 or y.dim() != 3 or weight.dtype not in _DTYPE_CODE:
        raise TypeError("linear_cf_ln_hip: y must be (B, K, L) float32 and the weight bf16 or fp16")
    B, K, L = y.shape
    if weight.dim() != 2 or weight.shape[1] != K:
        raise ValueError(f"linear_cf_ln_hip: weight must be (N, {K}), got {tuple(weight.shape)}")
    N, dt = weight.shape[0], weight.dtype
    y = y.contiguous()
    out = torch.empty((B, L, N), device=y.device, dtype=dt)
    if residual is not None and (residual.numel() != out.numel() or residual.dtype != dt):
        raise ValueError("linear_cf_ln_hip: residual must have the size and dtype of the result")
    small = [None if t is None else t.to(dt).contiguous() for t in (ln_weight, ln_bias, bias)]
    if small[0] is None:
        raise ValueError("linear_cf_ln_hip: the LayerNorm weight is required")
    keep = [weight.contiguous(), None if residual is None else residual.contiguous()]
    ptr = lambda t: None if t is None else t.data_ptr()
    rc = _lib.launch(y, _lib.lib().ss2d_linear_cf_ln, y.data_ptr(), ptr(small[0]), ptr(small[1]), float(eps),
                     keep[0].data_ptr(), ptr(small[2]), ptr(keep[1]), out.data_ptr(), B, L, K, N, _DTYPE_CODE[dt])
    _lib.check(rc, "ss2d_linear_cf_ln")
    return out


def linear_dw_hip(x, dy):
    """dy^T x for x (M, K) and dy (M, N), float32, contiguous: the weight gradient of a projection (ss2d_linear_dw_f32)."""
    if not (x.is_cuda and dy.device == x.device and x.dtype == dy.dtype == torch.float32 and x.dim() == dy.dim() == 2
            and x.shape[0] == dy.shape[0]):
        raise ValueError("linear_dw_hip expects float32 x (M, K) and dy (M, N) on one GPU")
    x, dy = x.contiguous(), dy.contiguous()
    (M, K), N = x.shape, dy.shape[1]
    need = _lib.lib().ss2d_linear_dw_f32_workspace_bytes(M, N, K)
    _lib.check(min(need, 0), "ss2d_linear_dw_f32_workspace_bytes")
    workspace = torch.empty(need, dtype=torch.uint8, device=x.device)
    dw = torch.empty((N, K), device=x.device, dtype=x.dtype)
    rc = _lib.launch(x, _lib.lib().ss2d_linear_dw_f32, x.data_ptr(), dy.data_ptr(), dw.data_ptr(), M, N, K, workspace.data_ptr(), need)
    _lib.check(rc, "ss2d_linear_dw_f32")
    return dw


def linear_dw_pays(layer, x):
    """True when LinearDw stands for ``layer(x)`` in training: a plain nn.Linear without bias, hooks or autocast, on float32
    positions many enough and with outputs few enough that the library leaves most of the chip idle.  12 544 positions, library
    against kernel in us: 384 x 384 outputs 77 against 54; 576 x 576 104 against 106.  96 x 96 over 200 704: 443 against 141;
    384 x 384 over 3136: 25 against 28."""
    if not (type(layer) is nn.Linear and layer.bias is None and x.is_cuda and x.dim() >= 2 and x.dtype == torch.float32):
        return False
    weight = layer.weight
    N, K = weight.shape
    return (torch.is_grad_enabled() and weight.requires_grad and weight.dtype == x.dtype and weight.device == x.device
            and x.shape[-1] == K and N % 4 == 0 and K % 4 == 0 and 0 < N * K <= 384 * 384 and x.numel() >= 4096 * K
            and not observed(layer) and not torch.is_autocast_enabled())


class LinearDw(torch.autograd.Function):
    """x W^T, plus ``residual`` if one is given, with dW = dy^T x on ss2d_linear_dw_f32."""

    @staticmethod
    def forward(ctx, x, weight, residual):
        ctx.save_for_backward(x, weight)
        if residual is None:
            return nn.functional.linear(x, weight)
        return torch.addmm(residual.reshape(-1, weight.shape[0]), x.reshape(-1, weight.shape[1]), weight.t()).view(residual.shape)

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        N, K = weight.shape
        dy2, x2 = dy.reshape(-1, N), x.reshape(-1, K)
        dx = torch.mm(dy2, weight).view(x.shape) if ctx.needs_input_grad[0] else None
        dw = None
        if ctx.needs_input_grad[1]:
            # the library's product where the kernel does not stand for it: under a second backward (it has no gradient of its
            # own), and for views that start between 16-byte boundaries, which contiguous() leaves where they are
            x2, dy2 = x2.contiguous(), dy2.contiguous()
            kernel = not torch.is_grad_enabled() and (x2.data_ptr() | dy2.data_ptr()) % 16 == 0
            dw = linear_dw_hip(x2, dy2) if kernel else torch.mm(dy2.t(), x2)
        return dx, dw, dy if ctx.needs_input_grad[2] else None
