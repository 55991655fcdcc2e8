"""CPU-only checks of the C ABI: the library loads, exports what include/ss2d_hip.h declares,
and validates arguments before touching the GPU (no kernel is launched here)."""
import ctypes
import os
import re

import pytest

from vmamba_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_functions():
    text = open(os.path.join(ROOT, "include", "ss2d_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ss2d_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_are_exported():
    names = _declared_functions()
    assert set(names) == set(_lib.EXPORTS), names
    L = ctypes.CDLL(_lib.LIB_PATH)
    for n in names:
        assert hasattr(L, n), n


def test_version_and_strerror():
    assert _lib.lib().ss2d_abi_version() == _lib.ABI_VERSION
    text = open(os.path.join(ROOT, "include", "ss2d_hip.h")).read()
    assert f"#define SS2D_ABI_VERSION {_lib.ABI_VERSION}" in text
    assert _lib.strerror(0) == "ok"
    assert "invalid" in _lib.strerror(_lib.SS2D_EINVAL)
    assert "unknown" in _lib.strerror(12345)


def test_struct_layout_matches_header():
    # 10 int32 + 9 pointers + 14 int64, no padding surprises
    assert ctypes.sizeof(_lib.ScanParams) == 10 * 4 + 9 * 8 + 14 * 8
    assert _lib.ScanParams.u.offset == 40 and _lib.ScanParams.u_batch_stride.offset == 40 + 72


def test_cross_scan_argument_validation():
    L = _lib.lib()
    assert L.ss2d_cross_scan(None, None, 0, 3, 4, 4, 4, None) == _lib.SS2D_OK          # empty: no-op
    assert L.ss2d_cross_scan(None, None, 2, 3, 0, 4, 2, None) == _lib.SS2D_OK
    assert L.ss2d_cross_scan(None, None, 1, 1, 1, 1, 4, None) == _lib.SS2D_EINVAL      # null pointers
    assert L.ss2d_cross_scan(None, None, 1, 1, 1, 1, 3, None) == _lib.SS2D_EINVAL      # element size
    assert L.ss2d_cross_scan(None, None, -1, 1, 1, 1, 4, None) == _lib.SS2D_EINVAL


def test_cross_merge_argument_validation():
    L = _lib.lib()
    assert L.ss2d_cross_merge(None, None, 0, 3, 4, 4, _lib.SS2D_F32, 0, None) == _lib.SS2D_OK
    assert L.ss2d_cross_merge(None, None, 1, 1, 1, 1, _lib.SS2D_F32, 0, None) == _lib.SS2D_EINVAL
    assert L.ss2d_cross_merge(None, None, 1, 1, 1, 1, 7, 0, None) == _lib.SS2D_EINVAL   # dtype
    assert L.ss2d_cross_merge(None, None, 1, 1, 1, 1, _lib.SS2D_F32, 2, None) == _lib.SS2D_EINVAL  # order


def test_cross_scan_flex_workspace_validation():
    """ss2d_cross_scan_flex_ws: argument and workspace checks happen before anything is launched."""
    L = _lib.lib()
    ws = ctypes.c_void_p(256)       # never dereferenced: every call below is refused first
    mixed = (0, 1, 0, 0)            # x channel-first, y channel-last
    assert L.ss2d_cross_scan_flex_ws(None, None, 0, 3, 4, 4, 2, *mixed, None, 0, None) == _lib.SS2D_OK       # empty
    assert L.ss2d_cross_scan_flex_ws(None, None, 1, 3, 4, 4, 3, *mixed, ws, 1 << 20, None) == _lib.SS2D_EINVAL  # element size
    assert L.ss2d_cross_scan_flex_ws(None, None, 1, 3, 4, 4, 2, 0, 2, 0, 0, ws, 1 << 20, None) == _lib.SS2D_EINVAL  # flag
    assert L.ss2d_cross_scan_flex_ws(ws, ws, 1, 3, 4, 4, 2, *mixed, None, 1 << 20, None) == _lib.SS2D_EINVAL    # no workspace
    assert L.ss2d_cross_scan_flex_ws(ws, ws, 1, 3, 4, 4, 2, *mixed, ctypes.c_void_p(260), 1 << 20, None) == _lib.SS2D_EINVAL  # alignment
    need = 1 * 3 * 16 * 2
    assert L.ss2d_cross_scan_flex_ws(ws, ws, 1, 3, 4, 4, 2, *mixed, ws, need - 1, None) == _lib.SS2D_ENOMEM
    assert L.ss2d_cross_scan_flex_ws(ws, ws, 1, 3, 4, 4, 2, 0, 1, 1, 0, ws, 4 * need - 1, None) == _lib.SS2D_ENOMEM  # one-by-one: 4 slices
    assert "workspace" in _lib.strerror(_lib.SS2D_ENOMEM)


def test_scan_argument_validation():
    L = _lib.lib()
    assert L.ss2d_selective_scan_fwd(None, None) == _lib.SS2D_EINVAL
    p = _lib.ScanParams()
    p.batch, p.dim, p.seqlen, p.dstate, p.n_groups, p.delta_dim = 0, 8, 16, 1, 4, 8
    p.in_dtype, p.out_dtype = _lib.SS2D_BF16, _lib.SS2D_F32
    assert L.ss2d_selective_scan_fwd(p, None) == _lib.SS2D_OK               # empty batch
    p.batch = 2
    assert L.ss2d_selective_scan_fwd(p, None) == _lib.SS2D_EINVAL           # null pointers
    p.dstate = 257
    assert L.ss2d_selective_scan_fwd(p, None) == _lib.SS2D_EINVAL           # dstate > 256
    p.dstate, p.n_groups = 1, 3
    assert L.ss2d_selective_scan_fwd(p, None) == _lib.SS2D_EINVAL           # dim % n_groups
    p.n_groups, p.out_dtype = 4, _lib.SS2D_F16
    assert L.ss2d_selective_scan_fwd(p, None) == _lib.SS2D_EINVAL           # out dtype neither f32 nor input


def _scan_plan(batch, dim, L, N, G, in_dtype=_lib.SS2D_BF16, with_x=True, base=1 << 20, query="ss2d_selective_scan_kernel"):
    """ss2d_selective_scan_kernel (or another query) for dense tensors of these sizes at made-up, 256-byte aligned addresses (the query
    reads the struct only)."""
    p = _lib.ScanParams()
    p.batch, p.dim, p.seqlen, p.dstate, p.n_groups, p.delta_dim = batch, dim, L, N, G, dim
    p.in_dtype, p.out_dtype, p.delta_softplus = in_dtype, _lib.SS2D_F32, 1
    p.u, p.delta, p.A, p.B, p.C, p.out = (base * k for k in range(1, 7))
    p.x = base * 7 if with_x else None
    p.u_batch_stride, p.u_d_stride = dim * L, L
    p.delta_batch_stride, p.delta_d_stride = dim * L, L
    p.A_d_stride, p.A_dstate_stride = N, 1
    p.B_batch_stride, p.B_group_stride, p.B_dstate_stride = G * N * L, N * L, L
    p.C_batch_stride, p.C_group_stride, p.C_dstate_stride = G * N * L, N * L, L
    p.out_batch_stride, p.out_d_stride = dim * L, L
    return getattr(_lib.lib(), query)(p)


def test_scan_kernel_choice_does_not_depend_on_the_chunk_state_output():
    """The reference's extension interface always asks for the chunk states `x`
    (selective_scan_oflex.cpp:207-208): every benchmark shape must reach the same kernel with and without it."""
    shapes = {  # batch, dim = 4 * d_inner, L, N -> kernel
        (128, 384, 3136, 1): _lib.SCAN_KERNEL_ROW, (128, 768, 784, 1): _lib.SCAN_KERNEL_ROW,
        (128, 1536, 196, 1): _lib.SCAN_KERNEL_SMALL, (128, 3072, 49, 1): _lib.SCAN_KERNEL_SMALL,
        (64, 768, 3136, 16): _lib.SCAN_KERNEL_CHAN, (4, 384, 65536, 1): _lib.SCAN_KERNEL_ROW4,
        (4, 768, 16384, 1): _lib.SCAN_KERNEL_ROW, (48, 384, 3306, 1): _lib.SCAN_KERNEL_FLAT,
        (16, 384, 100, 1): _lib.SCAN_KERNEL_FLAT,
    }
    for (batch, dim, L, N), kernel in shapes.items():
        for with_x in (False, True):
            assert _scan_plan(batch, dim, L, N, 4, with_x=with_x) == kernel, (batch, dim, L, N, with_x)
    assert _scan_plan(0, 384, 3136, 1, 4) == _lib.SCAN_KERNEL_NONE
    assert _scan_plan(2, 384, 3136, 1, 5) == _lib.SS2D_EINVAL
    assert _lib.lib().ss2d_selective_scan_kernel(None) == _lib.SS2D_EINVAL
    assert len(_lib.SCAN_KERNEL_NAMES) == 6


def test_scan_kernel_launched():
    """ss2d_selective_scan_launched names the kernel that runs: where ss2d_selective_scan_kernel says SS2D_SCAN_KERNEL_FLAT for rows that have a wavefront
    each, it does not; everywhere else the two agree."""
    flat, row = _lib.SCAN_KERNEL_FLAT, _lib.SCAN_KERNEL_ROW
    shapes = {  # batch, dim, L, N, groups -> kernel
        (48, 384, 3306, 1, 4): row, (16, 384, 100, 1, 4): row, (128, 384, 3306, 1, 4): row, (128, 384, 100, 1, 4): flat, (128, 768, 484, 1, 4): flat,
        (16, 384, 2051, 1, 4): row, (25, 99, 135, 16, 1): row, (1, 48, 1003, 16, 1): row, (131, 128, 36, 16, 8): flat, (131, 128, 33, 16, 8): row,
        (257, 160, 210, 16, 8): flat,
    }
    for (batch, dim, L, N, G), kernel in shapes.items():
        for with_x in (False, True):
            assert _scan_plan(batch, dim, L, N, G, with_x=with_x, query="ss2d_selective_scan_launched") == kernel, (batch, dim, L, N, G, with_x)
            assert _scan_plan(batch, dim, L, N, G, with_x=with_x) == flat
    for shape in ((128, 384, 3136, 1, 4), (128, 1536, 196, 1, 4), (64, 768, 3136, 16, 4), (4, 384, 65536, 1, 4), (1, 768, 3307, 1, 4), (2, 6, 2309, 3, 1), (0, 384, 9, 1, 4), (2, 384, 9, 1, 5)):
        assert _scan_plan(*shape) == _scan_plan(*shape, query="ss2d_selective_scan_launched") != flat, shape
    assert _lib.lib().ss2d_selective_scan_launched(None) == _lib.SS2D_EINVAL


def test_scan_channel_per_lane_rule_of_rows_off_the_grid():
    """Both sides of the lines between a channel per lane and positions in lanes, for rows of an odd number of fours in single precision and of an odd length."""
    chan = lambda N, L, batch, dtype=_lib.SS2D_F32: _scan_plan(batch, 384, L, N, 4, in_dtype=dtype, query="ss2d_selective_scan_launched") == _lib.SCAN_KERNEL_CHAN
    for N, L, batches in ((16, 100, (4, 8)), (16, 196, (15, 16)), (16, 484, (49, 50)), (16, 900, (26, 27)), (16, 1332, (31, 32)), (8, 196, (16, 17)), (8, 1028, (31, 32)), (4, 1028, (31, 32)), (4, 1764, (31, 32)),
                          (32, 900, (26, 27)), (32, 3364, (31, 32)), (4, 3364, (106, 107))):
        assert [chan(N, L, batch) for batch in batches] == [False, True], (N, L)
    for N, L, batches in ((4, 1764, (42, 43)), (4, 900, (85, 86)), (16, 1764, (2, 3)), (32, 1332, (2, 3)), (32, 5476, (2, 3))):
        assert [chan(N, L, batch) for batch in batches] == [True, False], (N, L)
    assert not any(chan(4, L, 128) for L in range(404, 512, 8)) and all(chan(4, L, 128) for L in (324, 396, 516, 764))
    assert [chan(16, L, 1) for L in (68, 76, 1028, 1532, 1540, 2044, 2052)] == [True, False, False, False, True, True, False]
    assert [chan(4, 1301, batch, _lib.SS2D_BF16) for batch in (42, 43, 128)] == [False] * 3 and [chan(4, 961, b, _lib.SS2D_BF16) for b in (42, 43, 85, 86)] == [False, True, True, False]
    assert all(chan(N, L, batch) for N in (4, 8, 16, 32) for L in (104, 200, 1336, 3360) for batch in (1, 64))      # whole eights: at any size


def _scan_bwd_plan(batch, dim, L, N, G, dtype=_lib.SS2D_BF16, base=1 << 32):
    """ss2d_selective_scan_bwd_kernel for dense tensors of these sizes at made-up, 256-byte aligned addresses far apart."""
    p = _lib.ScanBwdParams()
    p.batch, p.dim, p.seqlen, p.dstate, p.n_groups, p.delta_dim = batch, dim, L, N, G, dim
    p.in_dtype, p.dout_dtype, p.delta_softplus = dtype, _lib.SS2D_F32, 1
    p.u, p.delta, p.A, p.B, p.C, p.dout, p.du, p.ddelta, p.dA, p.dB, p.dC = (base * k for k in range(1, 12))
    p.u_batch_stride, p.u_d_stride = dim * L, L
    p.delta_batch_stride, p.delta_d_stride = dim * L, L
    p.dout_batch_stride, p.dout_d_stride = dim * L, L
    p.A_d_stride, p.A_dstate_stride = N, 1
    p.B_batch_stride, p.B_group_stride, p.B_dstate_stride = G * N * L, N * L, L
    p.C_batch_stride, p.C_group_stride, p.C_dstate_stride = G * N * L, N * L, L
    return _lib.lib().ss2d_selective_scan_bwd_kernel(p)


def test_scan_bwd_kernel_choice():
    """The query names the kernel that the call would launch, and the status of a call that would be refused."""
    name = lambda *args: _lib.SCAN_BWD_KERNEL_NAMES[_scan_bwd_plan(*args)]
    shapes = {  # batch, dim = 4 * d_inner, L, N -> kernel
        (64, 384, 3136, 1): "one", (64, 768, 784, 1): "one", (16, 768, 784, 16): "chan", (16, 768, 196, 16): "chan", (1, 384, 196, 16): "states",
        (16, 384, 784, 2): "states", (16, 48, 49, 16): "states", (1, 96, 3136, 16): "chan", (2, 16, 300, 40): "rows",
    }
    for (batch, dim, L, N), kernel in shapes.items():
        assert name(batch, dim, L, N, 4) == kernel, (batch, dim, L, N)
    for L in list(range(512, 2600)) + [3025, 3481, 3844, 3969, 65537]:      # every length of the rule's range, not only those that equal segments fill
        assert all(name(1, 256, L, N, 4, dtype) == "chan" for N in (8, 16) for dtype in (_lib.SS2D_BF16, _lib.SS2D_F32)), L
    f32, bf16 = _lib.SS2D_F32, _lib.SS2D_BF16           # 8 states: nearly whole passes of 256 positions
    assert [name(32, 384, L, 8, 4, dtype) for dtype in (f32, bf16) for L in (208, 209, 256, 257)] == ["chan", "states", "states", "chan"] + ["chan"] * 4
    # 8 states, many long rows: where the other kernel's workgroups and passes are full of positions
    for shape, dtype, kernel in (((32, 384, 1369), f32, "states"), ((32, 384, 1024), f32, "chan"), ((31, 384, 1369), f32, "chan"), ((64, 384, 1024), f32, "states"), ((64, 384, 784), f32, "chan"),
                                 ((48, 384, 1024), f32, "chan"), ((64, 768, 484), f32, "states"), ((64, 768, 484), bf16, "states"), ((64, 384, 961), bf16, "chan"), ((64, 768, 441), bf16, "chan")):
        assert name(*shape, 8, 4, dtype) == kernel, (shape, dtype)
        assert name(*shape, 16, 4, dtype) == "chan"
    assert name(0, 384, 3136, 1, 4) == "none"
    assert _scan_bwd_plan(2, 384, 3136, 1, 5) == _lib.SS2D_EINVAL
    assert _scan_bwd_plan(1, 16, 400_000, 40, 4) == _lib.SS2D_ENOTSUP
    assert _lib.lib().ss2d_selective_scan_bwd_kernel(None) == _lib.SS2D_EINVAL


def test_host_api_rejects_cpu_tensors_and_unsupported_modes():
    import torch
    import vmamba_amd as va
    x = torch.zeros(1, 2, 3, 3)
    with pytest.raises(NotImplementedError):
        va.cross_scan_fn(x)
    with pytest.raises(NotImplementedError):
        va.cross_merge_fn(torch.zeros(1, 4, 2, 3, 3))
    with pytest.raises(NotImplementedError):
        va.cross_scan_fn(x, scans=1)
    with pytest.raises(NotImplementedError):
        va.cross_scan_fn(x, force_torch=True)
    u = torch.zeros(1, 4, 8)
    with pytest.raises(RuntimeError):
        va.selective_scan_fn(u, u, torch.zeros(4, 1), torch.zeros(1, 4, 1, 8), torch.zeros(1, 4, 1, 8))
    with pytest.raises(NotImplementedError):
        va.selective_scan_fn(u, u, torch.zeros(4, 1), torch.zeros(1, 4, 1, 8), torch.zeros(1, 4, 1, 8), backend="torch")


def test_block_level_wrappers_have_no_cpu_path():
    """The harness-side kernels (fused MLP, narrow projection, LayerNorm variants, depthwise conv, fused core) raise on
    CPU tensors instead of computing anything there, and their 'fusable' predicates are False off the GPU."""
    import torch
    from vmamba_amd.conv import dwconv3x3_silu_hip
    from vmamba_amd.core import dt_proj_hip, ss2d_core_hip
    from vmamba_amd.linear import linear_cl_hip, linear_fusable
    from vmamba_amd.mlp import mlp_fusable, mlp_fused_hip
    from vmamba_amd.norm import add_layer_norm_fusable, add_layer_norm_hip, layer_norm_cf_hip, layer_norm_hip
    x = torch.zeros(4, 96, dtype=torch.bfloat16)
    w1, w2, w = torch.zeros(384, 96, dtype=torch.bfloat16), torch.zeros(96, 384, dtype=torch.bfloat16), torch.zeros(96, 96, dtype=torch.bfloat16)
    for call in (lambda: mlp_fused_hip(x, w1, None, w2, None), lambda: linear_cl_hip(x, w), lambda: layer_norm_hip(x, None, None),
                 lambda: add_layer_norm_hip(x, x, None, None), lambda: layer_norm_cf_hip(torch.zeros(1, 8, 4), None, None),
                 lambda: dwconv3x3_silu_hip(torch.zeros(1, 4, 4, 8), torch.zeros(8, 1, 3, 3), None, in_channel_last=True)):
        with pytest.raises(NotImplementedError):
            call()
    with pytest.raises(RuntimeError):
        ss2d_core_hip(torch.zeros(1, 2, 3, 3), torch.zeros(4, 2, 1, 9), torch.zeros(4, 1, 9), torch.zeros(4, 1, 9), torch.zeros(8))
    with pytest.raises(RuntimeError):
        dt_proj_hip(torch.zeros(4, 6, 8, dtype=torch.bfloat16), torch.zeros(4, 96, 6, dtype=torch.bfloat16))
    lin1, lin2 = torch.nn.Linear(96, 384).bfloat16(), torch.nn.Linear(384, 96).bfloat16()
    assert not mlp_fusable(x, lin1, lin2) and not linear_fusable(x, w) and not add_layer_norm_fusable(x, x)


def test_torch_extension_shim_loads_and_validates_on_cpu():
    import torch
    from vmamba_amd import oflex_ext
    ext = oflex_ext.load()
    assert hasattr(ext, "fwd") and hasattr(ext, "bwd")
    z = torch.zeros(1, 4, 8)
    with pytest.raises(RuntimeError):       # CPU tensors are refused before anything touches a GPU
        ext.fwd(z, z, torch.zeros(4, 1), torch.zeros(1, 4, 1, 8), torch.zeros(1, 4, 1, 8), None, None, True, 1, True)


def test_x_proj_says_what_it_takes():
    """The conditions of ss2d_x_proj from the sizes alone, and that the call itself refuses the same before any launch."""
    L = _lib.lib()
    applies = lambda B, D, C, H, W, dtype=_lib.SS2D_BF16: L.ss2d_x_proj_applies(B, D, C, H, W, dtype)
    taken = [(1, 96, 8, 56, 56), (2, 768, 50, 7, 7), (0, 96, 8, 56, 56), (4, 96, 38, 64, 2000), (64, 96, 8, 64, 2001), (1, 8, 96, 1, 8)]
    refused = [(1, 12, 8, 56, 56), (1, 96, 97, 56, 56), (1, 96, 8, 1, 7), (1, 96, 38, 64, 2001), (1, 768, 80, 32, 1001), (1, 1 << 20, 8, 64, 64)]
    assert all(applies(*c) == _lib.SS2D_OK for c in taken)
    for c in refused:
        assert applies(*c) == _lib.SS2D_ENOTSUP, c
        B, D, C, H, W = c
        assert L.ss2d_x_proj(256, 256, 256, B, D, C, H, W, H, W, -1, C * H * W, H * W, 4 * C * H * W, _lib.SS2D_BF16, None) == _lib.SS2D_ENOTSUP
    assert applies(1, 96, 8, 56, 56, _lib.SS2D_F32) == _lib.SS2D_ENOTSUP and applies(-1, 96, 8, 56, 56) == _lib.SS2D_EINVAL


def test_x_proj_bounds_the_padded_tail():
    """The last tile writes the added positions behind it, and its index arithmetic is exact below 2^23 items only: a map padded
    far beyond its size is refused before any launch."""
    call = lambda C, H, W, Hp, Wp: _lib.lib().ss2d_x_proj(256, 256, 256, 1, 8, C, H, W, Hp, Wp, -1, C * Hp * Wp, Hp * Wp,
                                                          4 * C * Hp * Wp, _lib.SS2D_BF16, None)
    for args in ((1, 4, 4, 4096, 4096), (8, 8, 8, 8, 1 << 18), (96, 8, 8, 1 << 18, 8)):
        assert call(*args) == _lib.SS2D_ENOTSUP, args


def test_forward_core_says_what_it_takes():
    """Whatever one of the four kernels refuses, the workspace query refuses: nothing has been launched or allocated then."""
    def bytes_of(**kw):
        p = _lib.ForwardCoreParams(batch=2, dim=64, height=8, width=8, rank=4, padded_height=8, padded_width=8, dtype=_lib.SS2D_BF16,
                                   norm_dtype=_lib.SS2D_BF16, normalise=1, eps=1e-5)
        for name in ("x", "x_proj_weight", "dt_proj_weight", "A", "D", "delta_bias", "norm_weight", "norm_bias", "out"):
            setattr(p, name, 4096)
        for name, value in kw.items():
            setattr(p, name, value)
        return _lib.lib().ss2d_forward_core_workspace_bytes(p)
    F32, BF16, F16 = _lib.SS2D_F32, _lib.SS2D_BF16, _lib.SS2D_F16
    taken = [{}, dict(rank=48), dict(norm_dtype=F32), dict(dtype=F32, norm_dtype=F32, rank=24), dict(dtype=F32, rank=24), dict(dtype=F16, norm_dtype=F16),
             dict(dtype=F16, norm_dtype=F32, normalise=0), dict(dtype=F32, norm_dtype=F32, dim=44)]
    refused = [dict(rank=49), dict(dtype=F32, norm_dtype=F32, rank=25), dict(dtype=F16, norm_dtype=F32), dict(norm_dtype=F16), dict(dim=44),
               dict(x_proj_weight=4096 + 8), dict(dim=8000), dict(rank=95), dict(dtype=F32, norm_dtype=F32, rank=48, dim=768, height=7, width=7, padded_height=7, padded_width=7)]
    for kw in taken:
        assert bytes_of(**kw) > 0, kw
    for kw in refused:
        assert bytes_of(**kw) == _lib.SS2D_ENOTSUP, kw


def test_forward_core_of_more_positions_than_the_folded_step_takes():
    """Ranks beyond 32-bit offsets of the core with dt_proj folded in: the plan takes the separate kernels, whose room includes delta
    (4 x 48 channels), instead of finding out behind x_proj."""
    p = _lib.ForwardCoreParams(batch=0, dim=48, height=56, width=56, rank=6, padded_height=56, padded_width=56, dtype=_lib.SS2D_BF16,
                               norm_dtype=_lib.SS2D_BF16, normalise=1, eps=1e-5)
    for name in ("x", "x_proj_weight", "dt_proj_weight", "A", "D", "delta_bias", "norm_weight", "norm_bias", "out"):
        setattr(p, name, 4096)
    most = (2 ** 31 - 1) // (4 * 15 * 56 * 56)               # 3 directions of 4 planes' room, two planes and the positions of one
    for batch, folded in ((most, True), (most + 1, False)):
        p.batch = batch
        positions = batch * 56 * 56
        need, plain = _lib.lib().ss2d_forward_core_workspace_bytes(p), positions * (4 * 8 * 2 + 48 * 4)    # projections, y
        delta = positions * 4 * 48 * 2
        assert plain <= need < plain + delta // 4 if folded else need >= plain + delta, (batch, need)


def test_block_says_what_it_takes():
    """Whatever one of the block's kernels refuses, the workspace query and the call refuse before anything is launched."""
    L = _lib.lib()
    BF16 = _lib.SS2D_BF16

    def both(core={}, **kw):
        p = _lib.BlockParams(core=_lib.ForwardCoreParams(batch=2, dim=64, height=8, width=8, rank=4, padded_height=8, padded_width=8, dtype=BF16,
                                                         norm_dtype=BF16, eps=1e-5), d_model=64, hidden=256, norm_eps=1e-5, norm2_eps=1e-5)
        for name in ("x_proj_weight", "dt_proj_weight", "A", "D", "delta_bias", "norm_weight", "norm_bias"):
            setattr(p.core, name, 4096)
        for name, kind in p._fields_:
            if kind is ctypes.c_void_p and name != "residual":
                setattr(p, name, 4096)
        for name, value in core.items():
            setattr(p.core, name, value)
        for name, value in kw.items():
            setattr(p, name, value)
        # (no room: a call that is taken ends with SS2D_ENOMEM, before any launch)
        return L.ss2d_block_workspace_bytes(p), L.ss2d_block_fwd(p, 4096, 0, None)

    taken = [{}, dict(d_model=768, hidden=3072), dict(fc1_weight=None, hidden=4096), dict(hidden=272), dict(norm_bias=None, fc2_bias=None),
             dict(norm_weight=None, norm_bias=None, residual=4096, d_model=784, fc1_weight=None), dict(core=dict(dtype=_lib.SS2D_F16, norm_dtype=_lib.SS2D_F16))]
    refused = [dict(d_model=100), dict(d_model=392), dict(d_model=784), dict(d_model=8), dict(hidden=100), dict(hidden=264), dict(hidden=3088), dict(hidden=4096),
               dict(core=dict(dim=72)), dict(core=dict(dim=3088)), dict(core=dict(rank=49)), dict(core=dict(dtype=_lib.SS2D_F32)),
               dict(core=dict(norm_weight=4104)), *(dict([(name, 4104)]) for name in ("x", "residual", "in_proj_weight", "in_proj_bias", "out_proj_weight",
                                                                                      "norm2_bias", "fc1_weight", "fc2_weight", "fc2_bias", "out"))]
    wrong = [dict(x=None), dict(out=None), dict(fc2_weight=None), dict(norm2_weight=None), dict(norm_weight=None, norm_bias=None), dict(d_model=0), dict(hidden=-1),
             dict(norm_weight=None, residual=4096), dict(core=dict(batch=0)), dict(core=dict(norm_weight=None))]
    for kw in taken:
        need, rc = both(**kw)
        assert need > 0 and rc == _lib.SS2D_ENOMEM, kw
    for kw in refused:
        assert both(**kw) == (_lib.SS2D_ENOTSUP, _lib.SS2D_ENOTSUP), kw
    for kw in wrong:
        assert both(**kw) == (_lib.SS2D_EINVAL, _lib.SS2D_EINVAL), kw
