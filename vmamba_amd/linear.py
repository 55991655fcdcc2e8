"""Narrow channel-last projection on the HIP kernel ss2d_linear_cl: out = [LayerNorm](x) W^T + bias + residual.

Stands in, in a channel-last VSS block of width 96, for norm + in_proj and for out_proj + the residual add
(classification/models/vmamba.py:1225-1228, :648-650, :662) at inference in bf16 / fp16; other widths and fp32
stay on the PyTorch-ROCm operators.  In single-precision training the products of these projections and of the MLP, and their gradients,
are HIP kernels (ss2d_product_f32, ss2d_linear_dw_f32) where those are the faster ones.
"""
import torch
import torch.nn as nn

from . import _lib
from .norm import TENSOR_KINDS, TRAIN_FROM, LayerNorm, calls_unseen, column_sums, memory_readable, needs_grad, observed, operators_seen

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


def linear_tiles_fusable(x, layer, act=None):
    """True when ss2d_linear_tiles stands for ``layer(x)`` -- ``act(layer(x))``, act exact GELU that nothing observes -- at inference on
    contiguous rows of x and is the faster one (linear_tiles_pays)."""
    if type(layer) is not nn.Linear or type(x) not in TENSOR_KINDS or x.dtype not in _DTYPE_CODE:
        return False
    if act is not None and not (type(act) is nn.GELU and act.approximate == "none" and not observed(act)):
        return False
    N, K = layer.weight.shape
    return (x.shape[-1] == K and K % 32 == 0 and K > 0 and linear_tiles_pays(x.numel() // K, N, K, act is not None) and linear_rows_takes(layer, x)
            and calls_unseen() and x.is_contiguous() and x.data_ptr() % 16 == 0)


def linear_tiles_pays(M, N, K, gelu):
    """True where ss2d_linear_tiles is ahead of the library.  With the GELU, which is a pass over the result there: us in bf16, library
    product and GELU / kernel, four outputs per input: 384 at 3136 positions 21 / 16, at 25 088 91 / 61, at 100 352 354 / 229; 96 at 3136 10 / 11,
    at 12 544 19 / 12; 256 at 3136 16 / 14; 512 at 6272 33 / 36, at 12 544 75 / 48, at 50 176 276 / 159; 640 at 12 544 67 / 70; 768 at 6272 65 / 55, at 12 544
    89 / 92.  Without, the library's larger tiles are ahead but where the contraction is short and the outputs fill tiles of 192: 384 x 384 at
    12 544 positions 11 / 12, at 25 088 25 / 18, at 50 176 41 / 30; 320 x 320 at 25 088 19 / 16; 192 x 192 at 25 088 10 / 10, at 100 352 26 / 23; 256 x 256 at
    50 176 15 / 23; 512 x 512 at 25 088 20 / 28."""
    if gelu:
        return K <= 512 and M >= (12544 if K > 384 else 3136 if K >= 192 else 6272)
    return K <= 384 and (N % 192 == 0 or N % 192 >= 128) and M * N >= 8 << 20


def linear_tiles_hip(x, weight, bias=None, residual=None, gelu=False):
    """x (..., K) channel-last, weight (N, K), one 16-bit dtype: [gelu](x @ weight.T + bias) + residual, shape (..., N), for many positions
    (ss2d_linear_tiles); no residual behind a GELU."""
    if not x.is_cuda:
        raise NotImplementedError("linear_tiles_hip: vmamba_amd runs on the GPU only")
    if x.dtype not in _DTYPE_CODE:
        raise TypeError(f"linear_tiles_hip: unsupported dtype {x.dtype}")
    K = x.shape[-1]
    if weight.dim() != 2 or weight.shape[1] != K:
        raise ValueError(f"linear_tiles_hip: weight must be (N, {K}), got {tuple(weight.shape)}")
    N = weight.shape[0]
    for t, n in ((weight, N * K), (bias, N)):
        if t is not None and (t.dtype != x.dtype or t.device != x.device or t.numel() != n or not t.is_contiguous()):
            raise ValueError("linear_tiles_hip: contiguous parameters of x's dtype on its device")
    x = x.contiguous()
    out = x.new_empty(x.shape[:-1] + (N,))
    if residual is not None:
        if residual.shape != out.shape or residual.dtype != x.dtype or residual.device != x.device:
            raise ValueError("linear_tiles_hip: residual must have the shape, dtype and device of the result")
        residual = residual.contiguous()
    ptr = lambda t: None if t is None else t.data_ptr()
    rc = _lib.launch(x, _lib.lib().ss2d_linear_tiles, x.data_ptr(), weight.data_ptr(), ptr(bias), ptr(residual), out.data_ptr(), x.numel() // K, K, N,
                     int(gelu), _DTYPE_CODE[x.dtype])
    _lib.check(rc, "ss2d_linear_tiles")
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


# ss2d_product_f32: what stands behind the sum
PRODUCT_PLAIN, PRODUCT_GELU, PRODUCT_GELU_GRAD = range(3)


def product_f32_hip(a, b, a_by_columns=False, b_by_columns=False, bias=None, other=None, mode=PRODUCT_PLAIN):
    """sum_k A(m, k) B(n, k) in float32 on the bf16 matrix cores (ss2d_product_f32): a (M, K), or (K, M) by columns, b (N, K) or (K, N),
    contiguous; + bias (N) + other (M, N); PRODUCT_GELU: (the sum with the bias, its GELU); PRODUCT_GELU_GRAD: times GELU'(other)."""
    M, K = a.shape[::-1] if a_by_columns else a.shape
    N = b.shape[1] if b_by_columns else b.shape[0]
    if not a.is_cuda or b.shape[0 if b_by_columns else 1] != K:
        raise ValueError("product_f32_hip: a (M, K) and b (N, K) on one GPU, either stored by columns")
    if any(t is not None and (t.dtype != torch.float32 or t.device != a.device or not t.is_contiguous()) for t in (a, b, bias, other)):
        raise ValueError("product_f32_hip: contiguous float32 tensors on one GPU")
    if (bias is not None and bias.numel() != N) or (other is not None and tuple(other.shape) != (M, N)):
        raise ValueError("product_f32_hip: bias (N), other (M, N)")
    out = a.new_empty((M, N))
    out2 = torch.empty_like(out) if mode == PRODUCT_GELU else None
    L = _lib.lib()
    need = L.ss2d_product_f32_workspace_bytes(M, N, K, a_by_columns, b_by_columns)
    _lib.check(min(need, 0), "ss2d_product_f32_workspace_bytes")
    workspace = torch.empty(need, dtype=torch.uint8, device=a.device) if need else None
    ptr = lambda t: None if t is None else t.data_ptr()
    rc = _lib.launch(a, L.ss2d_product_f32, a.data_ptr(), b.data_ptr(), ptr(bias), ptr(other), out.data_ptr(), ptr(out2), M, N, K,
                     a_by_columns, b_by_columns, mode, ptr(workspace), need)
    _lib.check(rc, "ss2d_product_f32")
    return out if out2 is None else (out, out2)


def product_pays(M, N, K, gradient=False):
    """True where ss2d_product_f32 is ahead of the library's fp32 product, whose rate is 90-100 TFLOP/s at best.  The kernel needs
    workgroups: 384 tiles of 128 x 64 outputs, or shares of a long sum (``gradient``: both operands by columns, K the positions), or 6 G
    products in any cut.  us in a graph, library / kernel: 12 544 x 1536 x 384 146 / 104, x 384 x 1536 147 / 114, x 384 x 384 48 / 34 (588 tiles);
    50 176 x 96 x 96 28 / 18; 1176 x 2048 x 512 38 / 34 (320 tiles, left), 4181 x 384 x 384 16 / 22 (198), 3136 x 768 x 192 13 / 15 (300);
    9408 x 512 x 2048 188 / 148 (592 tiles), 3136 x 512 x 2048 55 / 61 (3.3 G), 2090 x 768 x 3072 79 / 83 (4.9 G).  Gradients: 1536 x 384 over
    12 544 positions 142 / 91, over 4096 50 / 42, 384 x 96 over 50 176 253 / 74, 256 x 1024 over 6272 42 / 38, 768 x 192 over 3136 22 / 28."""
    if gradient:
        return K >= 4096
    return -(-M // 128) * -(-N // 64) >= 384 or M * N * K >= 6 << 30


def _product(a, b, a_by_columns=False, b_by_columns=False, bias=None, other=None, mode=PRODUCT_PLAIN):
    """product_f32_hip where it stands for the library's product, which is taken under a second backward (the kernel has no gradient of its
    own), for tensors whose memory is not theirs (memory_readable), for views that start between 16-byte boundaries and where it is the faster one."""
    M, K = a.shape[::-1] if a_by_columns else a.shape
    N = b.shape[1] if b_by_columns else b.shape[0]
    if (product_pays(M, N, K, a_by_columns and b_by_columns) and not torch.is_grad_enabled() and N % 4 == 0 and (M if a_by_columns else K) % 4 == 0
            and (b_by_columns or K % 4 == 0) and M * N * K > 0 and memory_readable(a, b, bias, other)):
        a, b = a.contiguous(), b.contiguous()
        other = None if other is None else other.contiguous()
        if all(t is None or t.data_ptr() % 16 == 0 for t in (a, b, bias, other)):
            return product_f32_hip(a, b, a_by_columns, b_by_columns, bias, other, mode)
    a, b = a.t() if a_by_columns else a, b if b_by_columns else b.t()
    if mode == PRODUCT_GELU_GRAD:
        return torch.ops.aten.gelu_backward(torch.mm(a, b), other)
    term = bias if other is None else other if bias is None else other + bias
    y = torch.mm(a, b) if term is None else torch.addmm(term, a, b)
    return y if mode == PRODUCT_PLAIN else (y, nn.functional.gelu(y))


def _weight_gradient(dy, x):
    """dy^T x, dy (M, N) and x (M, K).  Up to 384 x 384 outputs ss2d_linear_dw_f32 has the longest sums and ss2d_product_f32, in graphs, some of
    the others: 96 x 96 over 200 704 positions 136 / 158 us, over 50 176 87 / 68, 192 x 192 over 50 176 70 / 72, 384 x 384 over 12 544 51 / 43, 256 x 256 44 / 35."""
    N, K = dy.shape[1], x.shape[1]
    if N * K <= 384 * 384 and x.shape[0] >= 4096 and N % 4 == 0 and K % 4 == 0 and not torch.is_grad_enabled() and memory_readable(x, dy):
        x, dy = x.contiguous(), dy.contiguous()
        if (x.data_ptr() | dy.data_ptr()) % 16 == 0:
            return linear_dw_hip(x, dy)
    return _product(dy, x, True, True)


def _plain_f32(x, *tensors):
    return all(t is None or (type(t) in TENSOR_KINDS and t.dtype == torch.float32 and t.device == x.device) for t in tensors)


def linear_dw_pays(layer, x):
    """True when LinearDw stands for ``layer(x)`` in training: a plain nn.Linear without bias, hooks or autocast, on float32
    positions many enough and with outputs few enough that the library leaves most of the chip idle, or where ss2d_product_f32 is ahead
    of it.  12 544 positions, weight gradient, library against kernel in us: 384 x 384 outputs 72 against 51.
    96 x 96 over 200 704: 435 against 136; 384 x 384 over 6272: 36 against 36, over 4096: 25 against 31."""
    if not (type(layer) is nn.Linear and layer.bias is None and x.is_cuda and x.dim() >= 2 and x.dtype == torch.float32):
        return False
    weight = layer.weight
    N, K = weight.shape
    return (torch.is_grad_enabled() and type(weight) in TENSOR_KINDS and weight.requires_grad and weight.dtype == x.dtype and weight.device == x.device
            and x.shape[-1] == K and N % 4 == 0 and K % 4 == 0 and N * K > 0 and x.numel() >= 4096 * K
            and (N * K <= 384 * 384 or (x.numel() >= TRAIN_FROM and product_pays(x.numel() // K, N, K))) and not observed(layer) and calls_unseen())


class LinearDw(torch.autograd.Function):
    """x W^T, plus ``residual`` if one is given; dW = dy^T x on ss2d_linear_dw_f32, and ss2d_product_f32 for what it is faster at."""

    @staticmethod
    def forward(ctx, x, weight, residual):
        ctx.save_for_backward(x, weight)
        N, K = weight.shape
        y = _product(x.reshape(-1, K), weight, other=None if residual is None else residual.reshape(-1, N))
        return y.view(x.shape[:-1] + (N,) if residual is None else residual.shape)

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        N, K = weight.shape
        dy2, x2 = dy.reshape(-1, N), x.reshape(-1, K)
        dx = _product(dy2, weight, b_by_columns=True).view(x.shape) if ctx.needs_input_grad[0] else None
        dw = _weight_gradient(dy2, x2) if ctx.needs_input_grad[1] else None
        return dx, dw, dy if ctx.needs_input_grad[2] else None


def mlp_f32_pays(x, fc1, act, fc2):
    """True when MlpF32 stands for ``fc2(act(fc1(x)))`` in training: plain nn.Linear layers and exact GELU that nothing observes, contiguous
    float32 parameters, TRAIN_FROM elements, and a first product that ss2d_product_f32 is ahead in."""
    if not (x.dtype == torch.float32 and x.numel() >= TRAIN_FROM and type(x) in TENSOR_KINDS and x.is_cuda and x.dim() >= 2 and type(fc1) is type(fc2) is nn.Linear
            and type(act) is nn.GELU and act.approximate == "none"):
        return False
    N, K = fc1.weight.shape
    params = (fc1.weight, fc1.bias, fc2.weight, fc2.bias)
    return (needs_grad(x, *params) and x.shape[-1] == K and tuple(fc2.weight.shape)[1:] == (N,) and N % 4 == 0 and K % 4 == 0 and N * K > 0
            and product_pays(x.numel() // K, N, K) and _plain_f32(x, *params) and all(t is None or t.is_contiguous() for t in params)
            and (fc1.bias is None or fc1.bias.numel() == N) and (fc2.bias is None or fc2.bias.numel() == fc2.weight.shape[0])
            and not any(observed(m) for m in (fc1, act, fc2)) and calls_unseen())


class MlpF32(torch.autograd.Function):
    """fc2(GELU(fc1(x))) in single precision: GELU behind the first product, its derivative behind the second one's input gradient."""

    @staticmethod
    def forward(ctx, x, w1, b1, w2, b2):
        pre, act = _product(x.reshape(-1, x.shape[-1]), w1, bias=b1, mode=PRODUCT_GELU)
        ctx.save_for_backward(x, w1, b1, w2, pre, act)
        return _product(act, w2, bias=b2).view(x.shape[:-1] + (w2.shape[0],))

    @staticmethod
    def backward(ctx, dy):
        x, w1, b1, w2, pre, act = ctx.saved_tensors
        x2, dy2 = x.reshape(-1, x.shape[-1]), dy.reshape(-1, dy.shape[-1])
        if torch.is_grad_enabled():                                  # a second backward goes through what stands between, not only through x
            pre = nn.functional.linear(x2, w1, b1)
            act = nn.functional.gelu(pre)
        wants = ctx.needs_input_grad
        dw2 = _weight_gradient(dy2, act) if wants[3] else None
        db2 = column_sums(dy2) if wants[4] else None
        if not any(wants[:3]):
            return None, None, None, dw2, db2
        dpre = _product(dy2, w2, b_by_columns=True, other=pre, mode=PRODUCT_GELU_GRAD)
        dw1 = _weight_gradient(dpre, x2) if wants[1] else None
        db1 = column_sums(dpre) if wants[2] else None
        dx = _product(dpre, w1, b_by_columns=True).view(x.shape) if wants[0] else None
        return dx, dw1, db1, dw2, db2
