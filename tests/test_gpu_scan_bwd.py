"""GPU parity of the selective-scan backward (through the C ABI and through autograd) against float64 autograd of
the CPU restatement.  Tolerance: rtol 2e-3 plus 2e-3 of the gradient's largest magnitude for fp32 inputs (sums over
up to a few thousand positions in fp32 with hardware exp2 / log2); 16-bit inputs: 3e-2."""
import pytest
import torch

from oracle import torch_ref
import vmamba_amd as va
from vmamba_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ["du", "ddelta", "dA", "dB", "dC", "dD", "ddelta_bias"]


def make(seed, batch, dim, G, N, L, dtype, delta_dim=None, softplus=True):
    g = torch.Generator().manual_seed(seed)
    delta_dim = delta_dim or dim
    A = -0.5 * torch.rand(dim, N, generator=g) - 0.05
    if softplus:
        delta = torch.randn(batch, delta_dim, L, generator=g) - 1.0
        bias = torch.randn(delta_dim, generator=g) * 0.5 - 1.0
    else:
        delta = 0.3 * torch.rand(batch, delta_dim, L, generator=g)
        bias = 0.2 * torch.rand(delta_dim, generator=g)
    B = torch.randn(batch, G, N, L, generator=g)
    C = torch.randn(batch, G, N, L, generator=g)
    u = torch.randn(batch, dim, L, generator=g)
    D = torch.randn(dim, generator=g)
    dout = torch.randn(batch, dim, L, generator=g)
    return u.to(dtype), delta.to(dtype), A, B.to(dtype), C.to(dtype), D, bias, dout


def compare(got, want, tol, what):
    for name, g, w in zip(NAMES, got, want):
        if w is None:
            assert g is None, name
            continue
        g, w = g.double().cpu(), w.double()
        assert g.shape == w.shape, (name, g.shape, w.shape)
        scale = w.abs().max().item() + 1e-12
        err = (g - w).abs().max().item()
        assert err <= tol * scale + tol * 1e-3, f"{what} {name}: max err {err} vs scale {scale}"


CASES = [
    # batch, dim, G, N, L, delta_dim, softplus
    (2, 4, 1, 1, 40, None, True),          # one short pass
    (2, 8, 4, 1, 700, None, True),         # two passes, SS2D-like grouping (2 channels per B/C row)
    (1, 4, 2, 4, 1030, None, True),        # three passes, several states
    (2, 6, 2, 3, 513, 3, True),            # delta rows shared by two channels; one element into the second pass
    (1, 4, 1, 16, 300, None, True),        # 16 states
    (2, 4, 2, 2, 600, None, False),        # no softplus
    (1, 3, 1, 1, 9, None, True),           # shorter than a lane's 8 items + 1
    (2, 32, 2, 1, 700, None, True),        # 16 channels per group: dB / dC summed per workgroup in LDS
    (1, 60, 2, 2, 300, None, True),        # 30 channels per group in two chunks of 15, two states
    (1, 27, 1, 1, 520, 9, True),           # 27 channels in chunks of 14 + 13, delta rows shared by three channels
    (1, 24, 1, 1, 3136, None, True),       # one state, 7 passes, 6 channels per wavefront (pass-major kernel)
    (2, 10, 1, 1, 100, None, False),       # the same kernel without softplus, wavefronts with 3 and 2 channels
    (3, 14, 2, 1, 49, None, True),         # rows that fit 64 lanes: one position per lane
    (2, 12, 1, 1, 196, 4, True),           # one pass of 4 positions per lane; delta rows shared by three channels
    (2, 9, 1, 1, 255, None, True),         # the same with rows that are read element by element
    (1, 40, 1, 1, 4100, None, True),       # 9 passes, the last one 4 positions long; workgroups of 4 channels
    (2, 10, 1, 2, 256, None, True),        # exactly one pass; one wavefront with two of its four states
    (1, 8, 2, 5, 257, None, True),         # one position into the second pass; the last wavefront has one state
    (2, 30, 1, 16, 784, None, True),       # 16 states, 4 passes, 30 channels in workgroups of 4 and fewer
    (1, 6, 1, 32, 60, 2, False),           # the most states of this kernel, one position per lane, no softplus
    (1, 4, 2, 40, 300, None, True),        # more: a wavefront per row
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_scan_bwd_fp32_against_float64_autograd(case):
    batch, dim, G, N, L, delta_dim, softplus = case
    print("CASE scan-bwd", case, flush=True)
    u, delta, A, B, C, D, bias, dout = make(sum(map(int, case[:5])), batch, dim, G, N, L, torch.float32, delta_dim, softplus)
    want = torch_ref.selective_scan_grads(u, delta, A, B, C, D, bias, dout, softplus)
    dev = [t.to(DEV) for t in (u, delta, A, B, C, D, bias, dout)]
    got = va.selective_scan_bwd(*dev, None, softplus, 1)
    torch.cuda.synchronize()
    compare(got, want, 2e-3, "abi")
    # optional arguments absent
    want2 = torch_ref.selective_scan_grads(u, delta, A, B, C, None, None, dout, softplus if softplus else False)
    got2 = va.selective_scan_bwd(dev[0], dev[1], dev[2], dev[3], dev[4], None, None, dev[7], None, softplus, 1)
    compare(got2, want2, 2e-3, "no D / bias")


@pytest.mark.parametrize("dim,G", [(8, 4), (16, 1)], ids=["rows", "grouped"])
@pytest.mark.parametrize("dtype,dout_float", [(torch.bfloat16, True), (torch.bfloat16, False), (torch.float16, True)])
def test_scan_bwd_16bit_inputs(dtype, dout_float, dim, G):
    print("CASE scan-bwd-16", dtype, dout_float, dim, G, flush=True)
    u, delta, A, B, C, D, bias, dout = make(5, 2, dim, G, 1, 1200, dtype)
    dout = dout if dout_float else dout.to(dtype)
    want = torch_ref.selective_scan_grads(u.float(), delta.float(), A, B.float(), C.float(), D, bias, dout.float(), True)
    got = va.selective_scan_bwd(*[t.to(DEV) for t in (u, delta, A, B, C, D, bias, dout)], None, True, 1)
    assert got[0].dtype == dtype and got[1].dtype == dtype and got[3].dtype == dtype and got[2].dtype == torch.float32
    compare(got, want, 3e-2, "16-bit")


@pytest.mark.parametrize("dtype,dout_float", [(torch.bfloat16, True), (torch.float16, False)])
@pytest.mark.parametrize("N,L", [(1, 196), (1, 49), (1, 1100), (16, 784), (16, 196), (16, 49), (3, 333)])
def test_scan_bwd_16bit_row_lengths(N, L, dtype, dout_float):
    """Every positions-per-lane variant of the register-summing kernels with 16-bit rows (bound: as above)."""
    print("CASE scan-bwd-16-rows", N, L, dtype, dout_float, flush=True)
    u, delta, A, B, C, D, bias, dout = make(N + L, 2, 20, 2, N, L, dtype)
    dout = dout if dout_float else dout.to(dtype)
    want = torch_ref.selective_scan_grads(u.float(), delta.float(), A, B.float(), C.float(), D, bias, dout.float(), True)
    got = va.selective_scan_bwd(*[t.to(DEV) for t in (u, delta, A, B, C, D, bias, dout)], None, True, 1)
    compare(got, want, 3e-2, "16-bit")


# Rows that are no whole 16-byte pieces, read as dwords: one, two and three elements into a group of four and of eight, rows on odd elements and on
# even ones, one state and three; float64 as above.
@pytest.mark.parametrize("dtype,dout_float", [(torch.float32, True), (torch.bfloat16, True), (torch.bfloat16, False), (torch.float16, True)])
@pytest.mark.parametrize("N,L", [(1, 65), (1, 254), (1, 255), (1, 257), (1, 331), (1, 1030), (3, 67), (3, 301)])
def test_scan_bwd_odd_rows(N, L, dtype, dout_float):
    print("CASE scan-bwd-odd-rows", N, L, dtype, dout_float, flush=True)
    u, delta, A, B, C, D, bias, dout = make(N + L, 2, 10, 2, N, L, dtype)
    dout = dout if dout_float else dout.to(dtype)
    want = torch_ref.selective_scan_grads(u.float(), delta.float(), A, B.float(), C.float(), D, bias, dout.float(), True)
    got = va.selective_scan_bwd(*[t.to(DEV) for t in (u, delta, A, B, C, D, bias, dout)], None, True, 1)
    compare(got, want, 1e-4 if dtype == torch.float32 else 3e-2, "odd rows")


# A channel per lane (scan_bwd_chan.hip): rows of one segment (up to 72 positions, many of them), of two, and of many; the last chunk of 8 positions with
# 1, 3, 7 and 8 of them; 16, 33, 50 and 51 channels per group (1 and 2 in the last wavefront, idle wavefronts); 4, 8 and 16 states; delta rows
# shared; rows off the dword grid.  Bound in single precision: sums of up to 1030 terms and 51 channels, each term good to a few 2^-23 -- 1e-4 of the largest gradient.
CHANNEL_CASES = [
    (64, 64, 1, 16, 72, None, True), (64, 64, 1, 16, 73, None, True), (64, 66, 2, 8, 33, None, True), (64, 64, 1, 8, 7, None, False), (128, 64, 1, 4, 57, None, True),
    (64, 64, 1, 16, 128, None, True), (1, 96, 2, 16, 512, None, True), (1, 50, 1, 8, 515, 10, True), (1, 16, 1, 4, 1030, None, True), (2, 51, 1, 16, 779, 17, True),
    (1, 33, 1, 16, 600, None, False), (1, 80, 1, 16, 1000, None, True),
]


@pytest.mark.parametrize("case", CHANNEL_CASES, ids=lambda c: "x".join(str(v) for v in c))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_scan_bwd_channel_per_lane(case, dtype):
    batch, dim, G, N, L, delta_dim, softplus = case
    print("CASE scan-bwd-chan", case, dtype, flush=True)
    u, delta, A, B, C, D, bias, dout = make(sum(map(int, case[:5])), batch, dim, G, N, L, dtype, delta_dim, softplus)
    dout = dout.to(dtype) if L % 3 == 0 else dout
    want = torch_ref.selective_scan_grads(u.float(), delta.float(), A, B.float(), C.float(), D, bias, dout.float(), softplus)
    got = va.selective_scan_bwd(*[t.to(DEV) for t in (u, delta, A, B, C, D, bias, dout)], None, softplus, 1)
    compare(got, want, 1e-4 if dtype == torch.float32 else 3e-2, "channel per lane")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scan_bwd_channel_per_lane_strided_views(dtype):
    """Rows at odd distances and from odd elements on, B and C views of one projection: the bits of the contiguous call, but for the atomics' order."""
    print("CASE scan-bwd-chan-views", dtype, flush=True)
    batch, dim, N, L = 2, 50, 16, 600
    u, delta, A, B, C, D, bias, dout = [t.to(DEV) for t in make(3, batch, dim, 1, N, L, dtype)]
    want = va.selective_scan_bwd(u, delta, A, B, C, D, bias, dout, None, True, 1)

    def view(t, pitch):
        rows = t.reshape(-1, t.shape[-1])
        store = torch.full((rows.shape[0] * pitch + 1,), float("nan"), device=DEV, dtype=t.dtype)
        out = store[1:].view(rows.shape[0], pitch)[:, :L]
        out.copy_(rows)
        return out.unflatten(0, t.shape[:-1])

    proj = torch.cat([B, C], 2).contiguous()
    args = (view(u, L + 5), view(delta, L + 1), A, proj[:, :, :N], view(C, L + 3), D, bias, view(dout, L + 7))
    got = va.selective_scan_bwd(*args, None, True, 1)
    for name, g, w in zip(NAMES, got, want):
        if name in ("du", "ddelta"):
            assert torch.equal(g, w), name
        else:
            assert torch.allclose(g.float(), w.float(), rtol=1e-2 if dtype == torch.bfloat16 else 1e-5, atol=1e-5 * w.float().abs().max().item()), name


def test_scan_bwd_channel_per_lane_keeps_channels_apart():
    """A NaN of one channel reaches that channel's rows and the sums over channels, not the other channels' rows: lanes without a channel, which read the
    last one's constants, included."""
    batch, dim, N, L = 1, 50, 16, 600
    u, delta, A, B, C, D, bias, dout = [t.to(DEV) for t in make(4, batch, dim, 1, N, L, torch.float32)]
    want = va.selective_scan_bwd(u, delta, A, B, C, D, bias, dout, None, True, 1)
    u[0, 49, 300] = float("nan")
    got = va.selective_scan_bwd(u, delta, A, B, C, D, bias, dout, None, True, 1)
    for i in (0, 1):
        assert torch.equal(got[i][:, :49], want[i][:, :49])
    assert bool(got[1][0, 49, :301].isnan().any()) and bool(got[2][:49].isfinite().all())


def test_selective_scan_fn_trains():
    """autograd through selective_scan_fn (csms6s.py:112-126): gradients reach every input."""
    print("CASE scan-autograd", flush=True)
    u, delta, A, B, C, D, bias, dout = make(9, 2, 8, 4, 1, 640, torch.float32)
    want = torch_ref.selective_scan_grads(u, delta, A, B, C, D, bias, dout, True)
    leaves = [t.to(DEV).requires_grad_(True) for t in (u, delta, A, B, C, D, bias)]
    y = va.selective_scan_fn(*leaves, True, True)
    y.backward(dout.to(DEV))
    compare([t.grad for t in leaves], want, 2e-3, "autograd")


def test_scan_bwd_rejections():
    u, delta, A, B, C, D, bias, dout = [t.to(DEV) for t in make(1, 1, 4, 1, 1, 16, torch.float32)]
    with pytest.raises(RuntimeError):
        va.selective_scan_bwd(u, delta, A, B, C, D, bias, dout[:, :2], None, True, 1)
    with pytest.raises(RuntimeError):
        va.selective_scan_bwd(u, delta, A.double(), B, C, D, bias, dout, None, True, 1)
    with pytest.raises(RuntimeError):
        va.selective_scan_bwd(u.cpu(), delta, A, B, C, D, bias, dout, None, True, 1)
    p = _lib.ScanBwdParams()
    assert _lib.lib().ss2d_selective_scan_bwd(p, None) == _lib.SS2D_EINVAL           # dstate 0
    assert _lib.lib().ss2d_selective_scan_bwd(None, None) == _lib.SS2D_EINVAL


def test_cleared_accumulators_and_rounded_pair():
    """ss2d_clear and ss2d_round_pair at their edges: sizes around a thread's 16 bytes and a workgroup's 16 KB, the words behind
    a buffer untouched, the same bits as torch's conversion."""
    import ctypes
    from vmamba_amd import _lib
    sizes = [1, 3, 4, 5, 4095, 4096, 4097, 12291]
    store = [torch.full((n + 4,), 7.0, device="cuda") for n in sizes]
    ptrs, nbytes = (ctypes.c_void_p * 8)(*(t.data_ptr() for t in store)), (ctypes.c_int64 * 8)(*(4 * n for n in sizes))
    assert _lib.launch(store[0], _lib.lib().ss2d_clear, ptrs, nbytes, 8) == _lib.SS2D_OK
    for t, n in zip(store, sizes):
        assert bool((t[:n] == 0).all()) and bool((t[n:] == 7).all())
    assert _lib.launch(store[0], _lib.lib().ss2d_clear, ptrs, nbytes, 9) == _lib.SS2D_EINVAL
    for dtype in (torch.bfloat16, torch.float16):
        for n0, n1 in ((1, 2048), (2047, 9), (2049, 0), (5000, 4096)):
            a, b = torch.randn(n0, device="cuda") * 300, torch.randn(max(n1, 1), device="cuda")
            a[0] = float("inf")
            x, y = (torch.full((n + 8,), 7.0, device="cuda", dtype=dtype) for n in (n0, n1))
            assert _lib.launch(a, _lib.lib().ss2d_round_pair, a.data_ptr(), x.data_ptr(), n0, b.data_ptr(), y.data_ptr(), n1,
                               _lib.SS2D_BF16 if dtype == torch.bfloat16 else _lib.SS2D_F16) == _lib.SS2D_OK
            assert torch.equal(x[:n0], a.to(dtype)) and torch.equal(y[:n1], b[:n1].to(dtype))
            assert bool((x[n0:] == 7).all()) and bool((y[n1:] == 7).all())


class _Watching(torch.overrides.TorchFunctionMode):
    """Sees the operators that are called: the Python route makes the tensors."""

    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _same(got, want):
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        assert a is None or (a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,delta_dim,has_D,has_bias", [(1, 24, True, True), (16, 24, False, True), (2, 24, True, False), (1, 6, False, False)])
def test_operators_made_in_the_extension_equal_those_made_from_python(N, delta_dim, has_D, has_bias, dtype):
    """The three operators forwards and backwards on dense, strided and transposed tensors: the same bits, sizes, strides and types.   (dA, dB, dC and the
    two vectors are sums of atomics over few positions: one wavefront's order.)"""
    from vmamba_amd.csms6s import selective_scan_bwd, selective_scan_fwd
    g = torch.Generator().manual_seed(71)
    rand = lambda *s: torch.randn(*s, generator=g).to("cuda", dtype)
    u, B, C, dout = rand(2, 30, 60)[:, 3:27, 8:58], rand(2, 4, N, 50), rand(2, 4, N + 1, 50)[:, :, :N], rand(2, 24, 50)
    delta, A = rand(2, delta_dim, 50) * 0.3, -torch.rand(24, N, generator=g).cuda()
    D, bias = (torch.rand(24, generator=g).cuda() if has_D else None), (torch.rand(delta_dim, generator=g).cuda() if has_bias else None)
    x, ys = rand(2, 6, 5, 10), rand(2, 4, 6, 5, 10)
    calls = [lambda: selective_scan_fwd(u, delta, A, B, C, D, bias, True, 1, True, True), lambda: selective_scan_fwd(u, delta, A, B, C, D, bias, False, 1, False, False),
             lambda: selective_scan_bwd(u, delta, A, B, C, D, bias, dout, None, True)[:2], lambda: selective_scan_bwd(u, delta, A, B, C, D, bias, dout.float(), None, False)[:2],
             lambda: [va.cross_scan_fn(x)], lambda: [va.cross_scan_fn(x.transpose(2, 3))], lambda: [va.cross_merge_fn(ys)], lambda: [va.cross_merge_fn(ys.transpose(3, 4))]]
    for call in calls:
        got = call()
        with _Watching():
            _same(got, call())
    sums = lambda: selective_scan_bwd(u, delta, A, B, C, D, bias, dout, None, True)[2:]
    got = sums()
    with _Watching():
        want = sums()
    for a, b in zip(got, want):
        assert (a is None) == (b is None) and (a is None or (a.dtype == b.dtype and a.shape == b.shape and torch.allclose(a.float(), b.float(), rtol=2e-2, atol=1e-4 * b.abs().max().item())))


def test_operators_made_in_the_extension_refuse_what_python_refuses():
    from vmamba_amd.csms6s import selective_scan_bwd, selective_scan_fwd
    u, A, B = torch.zeros(1, 8, 16, device="cuda"), torch.zeros(8, 1, device="cuda"), torch.zeros(1, 2, 1, 16, device="cuda")
    bad = [(u, u[:, :, :15], A, B, B), (u, u.half(), A, B, B), (u, u, A.half(), B, B), (u, u, A, B[:, :, :, ::2], B), (u.transpose(1, 2), u, A, B, B), (u, u, A, B, B.cpu()),
           (u, u, A, B, B, torch.zeros(7, device="cuda")), (u, u, A, B, B, None, torch.zeros(8, device="cuda", dtype=torch.half))]
    for args in bad:
        args = args + (None,) * (7 - len(args))
        with pytest.raises(RuntimeError):
            selective_scan_fwd(*args, True)
        with pytest.raises(RuntimeError):
            selective_scan_bwd(*args, u, None, True)
    with pytest.raises(RuntimeError):
        selective_scan_bwd(u, u, A, B, B, None, None, u.half()[:, :, :8], None, True)
    with pytest.raises(ValueError):
        va.cross_scan_fn(u)
    with pytest.raises(TypeError):
        va.cross_merge_fn(torch.zeros(1, 4, 2, 3, 3, device="cuda", dtype=torch.float64))


def bwd_kernel_of(u, delta, A, B, C, dout):
    """Name of the kernel the library picks for these tensors once they sit on the GPU."""
    from vmamba_amd.csms6s import scan_bwd_kernel_name
    u, delta, A, B, C, dout = (t.to(DEV) for t in (u, delta, A, B, C, dout))
    return scan_bwd_kernel_name(u, delta, A, B, C, dout, torch.empty(u.shape, device=DEV, dtype=u.dtype), torch.empty(u.shape, device=DEV, dtype=u.dtype))


# lengths that no equal segments fill: what is left for the last one would be shorter than its states
UNEVEN_CASES = [(1, 17, 1, 16, 529, None, True), (1, 32, 2, 16, 729, None, False), (1, 20, 1, 16, 961, 10, True), (1, 16, 1, 8, 585, None, True)]


@pytest.mark.parametrize("case", CHANNEL_CASES + UNEVEN_CASES, ids=lambda c: "x".join(str(v) for v in c))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_scan_bwd_channel_per_lane_is_the_kernel_that_runs(case, dtype):
    batch, dim, G, N, L, delta_dim, softplus = case
    u, delta, A, B, C, D, bias, dout = make(sum(map(int, case[:5])), batch, dim, G, N, L, dtype, delta_dim, softplus)
    assert bwd_kernel_of(u, delta, A, B, C, dout) == bwd_kernel_of(u, delta, A, B, C, dout.to(dtype)) == "chan"


@pytest.mark.parametrize("case", UNEVEN_CASES, ids=lambda c: "x".join(str(v) for v in c))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_scan_bwd_channel_per_lane_uneven_segments(case, dtype):
    test_scan_bwd_channel_per_lane(case, dtype)


@pytest.mark.parametrize("L", [600, 72])
def test_scan_bwd_channel_per_lane_lanes_without_a_channel_add_nothing(L):
    """33 channels per group: 15 lanes of the third wavefront have none.  The last channel's bias alone would let their decay overflow (softplus off,
    exp(-20 * -30)), where its own steps are small; an infinite C makes g of a zero dout NaN.  dB and dC are the real channels' sums."""
    print("CASE scan-bwd-chan-idle-lanes", L, flush=True)
    batch, dim, N = 96 if L == 72 else 1, 33, 16
    u, delta, A, B, C, D, bias, dout = make(6, batch, dim, 1, N, L, torch.float32, softplus=False)
    A[32], bias[32] = -20.0, -30.0
    delta[:, 32] += 30.0
    assert bwd_kernel_of(u, delta, A, B, C, dout) == "chan"
    want = torch_ref.selective_scan_grads(u, delta, A, B, C, D, bias, dout, False)
    got = va.selective_scan_bwd(*[t.to(DEV) for t in (u, delta, A, B, C, D, bias, dout)], None, False, 1)
    compare(got[3:5], want[3:5], 1e-4, "overflowing decay")
    u, delta, A, B, C, D, bias, dout = make(6, batch, dim, 1, N, L, torch.float32, softplus=False)
    u, B, C, dout = [t.abs() + 0.1 for t in (u, B, C, dout)]
    C[0, 0, 5, L - 1] = float("inf")
    got = va.selective_scan_bwd(*[t.to(DEV) for t in (u, delta, A, B, C, D, bias, dout)], None, False, 1)
    assert bool((got[3][0, 0, 5] == float("inf")).all()) and bool(got[3][0, 0, :5].isfinite().all()) and bool(got[4].isfinite().all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,L", [(4, 680), (8, 1000), (16, 700)])
def test_scan_bwd_channel_per_lane_infinite_states(N, L, dtype):
    """An infinite state and an infinite adjoint go through segments whose decays multiply to 0, as they would position by position (every one of them is
    above exp(-6)): infinities, not NaN, and only where they belong."""
    print("CASE scan-bwd-chan-infinite", N, L, dtype, flush=True)
    dim, inf, first, last = 16, float("inf"), 100, L - 90
    u, delta, A, B, C, D, bias, dout = make(8, 1, dim, 1, N, L, dtype, softplus=False)
    u, B, C, dout = [t.abs() + 0.125 for t in (u, B, C, dout)]                  # every sum is one of positive terms
    A, delta, bias, D = torch.full_like(A, -1.0), 5.0 + delta.abs(), torch.zeros_like(bias), D.abs()
    call = lambda: [t.double().cpu() for t in va.selective_scan_bwd(*[t.to(DEV) for t in (u, delta, A, B, C, D, bias, dout)], None, False, 1)]
    u[0, 3, first] = inf
    assert bwd_kernel_of(u, delta, A, B, C, dout) == "chan"
    du, ddelta, dA, dB, dC = call()[:5]
    assert bool((dC[0, 0, :, first:] == inf).all()) and bool(dC[0, 0, :, :first].isfinite().all())
    assert bool((dB[0, 0, :, first] == inf).all()) and bool(dB[0, 0, :, :first].isfinite().all()) and bool(dB[0, 0, :, first + 1:].isfinite().all())
    assert bool(du.isfinite().all()) and bool((ddelta[0, 3, first + 1:] == -inf).all()) and bool(ddelta[0, 3, :first].isfinite().all())
    assert not bool(dA[3].isfinite().any()) and bool(dA[:3].isfinite().all()) and bool(ddelta[0, 4:].isfinite().all())
    u[0, 3, first], dout[0, 5, last] = 1.0, inf
    du, ddelta, dA, dB, dC = call()[:5]
    assert bool((du[0, 5, :last + 1] == inf).all()) and bool(du[0, 5, last + 1:].isfinite().all()) and bool(du[0, :5].isfinite().all())
    assert bool((dB[0, 0, :, :last + 1] == inf).all()) and bool(dB[0, 0, :, last + 1:].isfinite().all())
    assert bool((dC[0, 0, :, last] == inf).all()) and bool(dC[0, 0, :, :last].isfinite().all()) and bool(ddelta[0, :5].isfinite().all())


@pytest.mark.parametrize("N,delta_dim", [(1, 24), (16, 24), (1, 6)])
def test_operators_are_made_in_the_extension(N, delta_dim, monkeypatch):
    """The extension makes what it is asked for, strided tensors included; what it leaves to Python are transposed maps and delta rows shared in the backward; and
    it is not asked where someone follows the operators."""
    from vmamba_amd.csms6s import selective_scan_bwd, selective_scan_fwd
    rand = lambda *s: torch.rand(*s, device="cuda")
    u, B, C, dout = rand(2, 30, 60)[:, 3:27, 8:58], rand(2, 4, N, 50), rand(2, 4, N + 1, 50)[:, :, :N], rand(2, 24, 50)
    delta, A, D, bias, x, ys = rand(2, delta_dim, 50), -rand(24, N), rand(24), rand(delta_dim), rand(2, 6, 5, 10), rand(2, 4, 6, 5, 10)
    made = []                                                   # of every call of the extension: whether it made the result
    for name in ("scan_fwd", "scan_bwd", "cross_scan", "cross_merge"):
        def counted(*args, _native=getattr(_lib.host(), name)):
            result = _native(*args)
            made.append(result is not None)
            return result
        monkeypatch.setattr(_lib.host(), name, counted)
    calls = [(lambda: selective_scan_fwd(u, delta, A, B, C, D, bias, True, 1, True, True), True), (lambda: selective_scan_bwd(u, delta, A, B, C, D, bias, dout, None, True), delta_dim == 24),
             (lambda: va.cross_scan_fn(x), True), (lambda: va.cross_scan_fn(x.transpose(2, 3)), False), (lambda: va.cross_merge_fn(ys), True),
             (lambda: va.cross_merge_fn(ys.transpose(3, 4)), False)]
    for call, native in calls:
        made.clear()
        call()
        assert made == [native]
        with _Watching():
            call()
        assert made == [native]


@pytest.mark.parametrize("L", [209, 225, 256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_scan_bwd_eight_states_of_nearly_a_pass(L, dtype):
    """209 to 256 positions of 8 states: a channel per lane in 16 bits, positions in lanes in single precision.  Of the images that the rule asks for the
    first three have a gradient; the others' is 0 and so is all that comes of it.  (Bounds as for CHANNEL_CASES.)"""
    print("CASE scan-bwd-eight-states", L, dtype, flush=True)
    u, delta, A, B, C, D, bias, dout = make(9 * L, 3, 48, 1, 8, L, dtype)
    want = torch_ref.selective_scan_grads(u.float(), delta.float(), A, B.float(), C.float(), D, bias, dout.float(), True)
    u, delta, B, C, dout = [t.repeat(72, *[1] * (t.dim() - 1)) for t in (u, delta, B, C, dout)]
    dout[3:] = 0
    assert bwd_kernel_of(u, delta, A, B, C, dout) == ("states" if dtype == torch.float32 else "chan")
    got = va.selective_scan_bwd(*[t.to(DEV) for t in (u, delta, A, B, C, D, bias, dout)], None, True, 1)
    assert not any(bool(got[i][3:].any()) for i in (0, 1, 3, 4))
    compare([t[:3] if i in (0, 1, 3, 4) else t for i, t in enumerate(got)], want, 1e-4 if dtype == torch.float32 else 3e-2, "eight states")
