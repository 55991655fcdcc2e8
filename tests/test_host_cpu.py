"""CPU checks of the host-side model code (no kernels run): shapes, parameter inventory and the
projection identity the SS2D core relies on."""
import pytest
import torch

from oracle.ss2d_core_ref import RefSS2D
from vmamba_amd.ss2d import SS2D
from vmamba_amd.vssm import vmamba_tiny_s1l8


def test_parameter_inventory_matches_reference_shapes():
    m = SS2D(d_model=96, d_state=1, ssm_ratio=1.0)
    K, D, R, N = 4, 96, 6, 1
    assert m.x_proj_weight.shape == (K, R + 2 * N, D)        # vmamba.py:468
    assert m.dt_projs_weight.shape == (K, D, R)              # vmamba.py:225
    assert m.dt_projs_bias.shape == (K, D)
    assert m.A_logs.shape == (K * D, N) and m.Ds.shape == (K * D,)
    assert torch.equal(m.Ds, torch.ones(K * D))
    dt = torch.nn.functional.softplus(m.dt_projs_bias)
    assert dt.min() >= 1e-3 * 0.999 and dt.max() <= 0.1 * 1.001  # dt log-uniform in [1e-3, 0.1]
    m16 = SS2D(d_model=96, d_state=16, ssm_ratio=2.0, disable_z=False)
    assert torch.allclose(m16.A_logs[5].exp(), torch.arange(1, 17).float())
    assert m16.in_proj.weight.shape == (2 * 192, 96)


def test_vmamba_tiny_parameter_count():
    assert sum(p.numel() for p in vmamba_tiny_s1l8().parameters()) == 30249064   # analyze/tp.py:162


def test_grouped_conv_equals_einsum():
    # x_proj/dt_proj as grouped conv1d == the einsum form (vmamba.py:605-608 vs :610-615)
    torch.manual_seed(0)
    m = SS2D(d_model=16, d_state=2, ssm_ratio=1.0)
    xs = torch.randn(2, 4, 16, 30)
    dts, Bs, Cs = m.project(xs)
    x_dbl = torch.einsum("bkdl,kcd->bkcl", xs, m.x_proj_weight)
    r, Bs2, Cs2 = torch.split(x_dbl, [m.dt_rank, 2, 2], dim=2)
    dts2 = torch.einsum("bkrl,kdr->bkdl", r, m.dt_projs_weight).reshape(2, -1, 30)
    assert torch.allclose(dts, dts2, atol=1e-5) and torch.allclose(Bs, Bs2, atol=1e-5) and torch.allclose(Cs, Cs2, atol=1e-5)


def test_reference_core_runs_on_cpu():
    torch.manual_seed(0)
    m = RefSS2D(d_model=8, d_state=1).eval()
    with torch.no_grad():
        y = m(torch.randn(1, 8, 5, 6))
    assert y.shape == (1, 8, 5, 6) and torch.isfinite(y).all()


def test_vssm_state_dict_uses_reference_key_names_and_loads_legacy_checkpoints():
    """State-dict keys are the reference's (classification/models/vmamba.py:1356-1363, 1402-1437, 1487-1490), and the
    key prefixes of its older training code are renamed on load (vmamba.py:1557-1564)."""
    import torch
    from oracle.ss2d_core_ref import reference_vmamba_tiny
    from vmamba_amd.vssm import VSSM

    torch.manual_seed(0)
    small = dict(depths=(1, 2), dims=(16, 32), num_classes=5)
    src = VSSM(**small, channel_first=False, layers=__import__("oracle.ss2d_core_ref", fromlist=["TorchLayers"]).TorchLayers)
    keys = set(src.state_dict().keys())
    block = {"norm.weight", "norm.bias", "op.x_proj_weight", "op.A_logs", "op.Ds", "op.dt_projs_weight", "op.dt_projs_bias",
             "op.in_proj.weight", "op.conv2d.weight", "op.out_norm.weight", "op.out_norm.bias", "op.out_proj.weight",
             "norm2.weight", "norm2.bias", "mlp.fc1.weight", "mlp.fc1.bias", "mlp.fc2.weight", "mlp.fc2.bias"}
    want = {f"patch_embed.{i}.{p}" for i in (0, 2, 5, 7) for p in ("weight", "bias")}
    want |= {f"layers.{i}.blocks.{j}.{k}" for (i, j) in ((0, 0), (1, 0), (1, 1)) for k in block}
    want |= {f"layers.0.downsample.{i}.{p}" for i in (1, 3) for p in ("weight", "bias")}
    want |= {f"classifier.{m}.{p}" for m in ("norm", "head") for p in ("weight", "bias")}
    assert keys == want
    assert len(reference_vmamba_tiny().state_dict()) == 276

    # a checkpoint written with the old names
    legacy = {}
    for k, v in src.state_dict().items():
        k = k.replace(".norm.", ".ln_1.") if ".blocks." in k and ".norm." in k and ".op." not in k else k
        k = k.replace(".op.", ".self_attention.")
        k = k.replace("patch_embed.0.", "patch_embed.proj.").replace("patch_embed.2.", "patch_embed.norm.")
        k = k.replace("classifier.norm.", "norm.").replace("classifier.head.", "head.")
        legacy[k] = v.clone()
    assert set(legacy) != keys
    dst = VSSM(**small, channel_first=False, layers=src.layers[0].blocks[0].op.layers)
    result = dst.load_state_dict(legacy, strict=True)
    assert not result.missing_keys and not result.unexpected_keys
    for (ka, a), (kb, b) in zip(src.state_dict().items(), dst.state_dict().items()):
        assert ka == kb and torch.equal(a, b)
    # channel-first models store 1x1-conv weights; a channel-last checkpoint loads into them (vmamba.py:47-49)
    cf = VSSM(**small, channel_first=True, layers=src.layers[0].blocks[0].op.layers)
    cf.load_state_dict(src.state_dict(), strict=True)
    assert torch.equal(cf.layers[0].blocks[0].mlp.fc1.weight, src.layers[0].blocks[0].mlp.fc1.weight)


def test_gelu_table_is_what_the_generator_writes_and_matches_erf():
    """The fused MLP kernel's GELU table: the committed include equals a fresh render, and its entries are
    0.5 erf(x / sqrt 2) at the bf16 grid (checked against scipy's erf, an independent implementation)."""
    import importlib.util, os, re, struct
    import numpy as np
    from scipy.special import erf
    here = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vmamba_amd", "csrc")
    spec = importlib.util.spec_from_file_location("gen_gelu_table", os.path.join(here, "gen_gelu_table.py"))
    gen = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(gen)
    text = open(os.path.join(here, "gelu_table.inc")).read()
    assert text == gen.render()
    bits = np.array([int(h, 16) for h in re.findall(r"0x([0-9a-f]{8})u", text)], dtype=np.uint32)
    assert bits.size == gen.HI_BITS - gen.LO_BITS == 2176
    vals = bits.view(np.float32).astype(np.float64)
    x = (np.arange(gen.LO_BITS, gen.HI_BITS, dtype=np.uint32) << 16).view(np.float32).astype(np.float64)
    assert x[0] == 2.0 ** -14 and x[-1] < 8.0 and x[-1] > 7.9
    want = 0.5 * erf(x / np.sqrt(2.0))
    assert np.all(np.abs(vals - want) <= 2.0 ** -24 * np.maximum(want, 1e-30) * 1.01)      # fp32 rounding of the exact value
    assert vals[-1] == 0.5 and np.all(np.diff(vals) >= 0)
    # the identity the kernel uses: gelu(x) = 0.5 x + |x| E(|x|), both signs
    for s in (1.0, -1.0):
        g = 0.5 * s * x + x * vals
        assert np.allclose(g, 0.5 * s * x * (1.0 + erf(s * x / np.sqrt(2.0))), rtol=0, atol=1e-6)


def test_inference_constants_are_kept_per_batch_size_and_follow_the_parameters():
    """A = -exp(A_logs) etc. (vmamba.py:619-623) are cached per batch size -- the sub-batches of a runner alternate with
    whole batches -- and recomputed when a parameter changes or autograd is on."""
    m = SS2D(d_model=8, d_state=1, ssm_ratio=1.0, dt_rank=2, channel_first=False)
    with torch.no_grad():
        c2, c3 = m._inference_constants(2), m._inference_constants(3)
        assert m._inference_constants(2) is c2 and m._inference_constants(3) is c3
        assert c2["Wx"].shape[0] == 2 * 4 and c3["Wx"].shape[0] == 3 * 4
        assert torch.equal(c2["As"], -m.A_logs.float().exp())
        for b in range(4, 10):                                   # the cache stays small
            m._inference_constants(b)
        assert len(m._const_cache) <= 4
        m.A_logs.add_(0.5)                                       # in-place update bumps the version: everything stale
        fresh = m._inference_constants(2)
        assert fresh is not c2 and torch.equal(fresh["As"], -m.A_logs.float().exp())
        assert all(k[0] == 2 for k in m._const_cache)
    assert m._inference_constants(2) is not m._inference_constants(2)      # under autograd nothing is kept


def test_with_layout_keeps_keys_values_and_mode():
    """VSSM.with_layout: the channel-last twin of a channel-first model holds the same state_dict (names, shapes, values)
    -- a Linear2d weight (out, in, 1, 1) and the nn.Linear weight (out, in) are one tensor viewed two ways
    (vmamba.py:47-49) -- and converts back."""
    from vmamba_amd.vssm import VSSM
    torch.manual_seed(3)
    m = VSSM(depths=(1, 1, 1, 1), dims=(16, 32, 64, 128), d_state=2, ssm_ratio=2.0, num_classes=10, channel_first=True).eval()
    twin = m.with_layout(False)
    assert not twin.training and twin.layers[0].blocks[0].op.channel_first is False
    sd, sd2 = m.state_dict(), twin.state_dict()
    assert list(sd) == list(sd2)
    for k in sd:
        assert sd[k].numel() == sd2[k].numel() and torch.equal(sd[k].reshape(-1), sd2[k].reshape(-1)), k
    back = twin.with_layout(True).state_dict()
    assert all(back[k].shape == sd[k].shape and torch.equal(back[k], sd[k]) for k in sd)
    # shared weights: the same Parameter objects under the same names; a change through one model is seen by the other
    shared = m.with_layout(False, share_weights=True)
    for (k, p), (k2, p2) in zip(m.named_parameters(), shared.named_parameters()):
        assert k == k2 and p is p2
    with torch.no_grad():
        m.classifier.head.weight.mul_(2.0)
    assert shared.classifier.head.weight is m.classifier.head.weight
    m.double()
    assert next(shared.parameters()).dtype == torch.float64


class _OnGpu:
    """A CPU tensor that says it lies on cuda:0: what the wrappers ask before any launch, without a GPU."""
    is_cuda, device = True, torch.device("cuda:0")

    def __init__(self, tensor):
        self._t = tensor

    def __getattr__(self, name):
        return getattr(self._t, name)

    def get_device(self):
        return 0


def test_x_proj_wants_its_tensors_on_one_device(monkeypatch):
    """A weight or a result that lies elsewhere is no operand of a kernel: the dispatch rule says no, the wrapper raises."""
    from vmamba_amd import _lib
    from vmamba_amd.core import x_proj_f32_fits, x_proj_f32_hip, x_proj_fits, x_proj_hip
    monkeypatch.setattr(_lib, "launch", lambda *a: (_ for _ in ()).throw(AssertionError("launched")))
    for dtype, fits, run in ((torch.bfloat16, x_proj_fits, x_proj_hip), (torch.float32, x_proj_f32_fits, x_proj_f32_hip)):
        x, weight, out = torch.zeros(1, 16, 4, 4, dtype=dtype), torch.zeros(4, 3, 16, dtype=dtype), torch.zeros(1, 4, 3, 16, dtype=dtype)
        assert not fits(_OnGpu(x), weight) and fits(_OnGpu(x), _OnGpu(weight))
        for w, o in ((weight, _OnGpu(out)), (_OnGpu(weight), out)):
            with pytest.raises(RuntimeError):
                run(_OnGpu(x), w, o)


def test_patch_embedding_kernel_stands_for_plain_convolutions_only():
    """The second layer's kernel goes past Conv2d._conv_forward: a convolution that computes something else there, or one that
    autocast runs in another type, is left to itself."""
    from vmamba_amd.norm import LayerNorm
    from vmamba_amd.stem import stem2_fusable

    class Standardised(torch.nn.Conv2d):
        def _conv_forward(self, x, weight, bias):
            return super()._conv_forward(x, weight - weight.mean((1, 2, 3), keepdim=True), bias)

    x = _OnGpu(torch.zeros(1, 48, 8, 8, dtype=torch.bfloat16).to(memory_format=torch.channels_last))
    make = lambda cls: cls(48, 96, 3, stride=2, padding=1).bfloat16()
    plain, norm = make(torch.nn.Conv2d), LayerNorm(96).bfloat16()
    assert stem2_fusable(x, plain, norm)
    assert not stem2_fusable(x, make(Standardised), norm)
    with torch.autocast("cuda", torch.bfloat16):
        assert not torch.is_autocast_enabled() or stem2_fusable(x, plain, norm)
    plain._conv_forward = lambda *a: None
    assert not stem2_fusable(x, plain, norm)


def test_convolution_function_and_single_call_core_have_no_cpu_path(monkeypatch):
    """Neither may hand a host address to a kernel, whichever of its tensors lies on the CPU."""
    from vmamba_amd import _lib
    from vmamba_amd.conv import DwConv3x3SiLU
    from vmamba_amd.core import forward_core_hip
    monkeypatch.setattr(_lib, "launch", lambda *a: (_ for _ in ()).throw(AssertionError("launched")))
    x, weight = torch.zeros(1, 16, 4, 4), torch.zeros(16, 1, 3, 3)
    with pytest.raises(NotImplementedError):
        DwConv3x3SiLU.apply(x, weight, None, False)
    ctx = torch.autograd.function.FunctionCtx()
    for w, b, error in ((weight, None, TypeError), (_OnGpu(weight.half()), None, TypeError), (_OnGpu(weight), weight[:, 0, 0, 0], TypeError),
                        (_OnGpu(weight[:8]), None, ValueError)):
        with pytest.raises(error):
            DwConv3x3SiLU.forward(ctx, _OnGpu(x), w, b, False)
    with pytest.raises(RuntimeError):
        forward_core_hip(x, torch.zeros(4, 3, 16), torch.zeros(4, 16, 1), *(torch.zeros(64) for _ in range(3)))


def test_observed_layers_are_called_in_training():
    """A layer whose calls something sees -- a hook of its own, a global one, a forward set on the instance -- is called as a
    module in training: no kernel stands for it."""
    from torch.nn.modules import module as nn_module
    from vmamba_amd.conv import dwconv_silu_trainable
    from vmamba_amd.linear import linear_dw_pays
    conv, linear = torch.nn.Conv2d(8, 8, 3, padding=1, groups=8), torch.nn.Linear(8, 8, bias=False)

    def taken():
        x, rows = _OnGpu(torch.zeros(1, 8, 6, 6)), _OnGpu(torch.zeros(4096, 8))
        x.device = rows.device = torch.device("cpu")              # the weights' own
        return [dwconv_silu_trainable(conv, x, False), linear_dw_pays(linear, rows)]
    see = lambda *args: None
    assert taken() == [True, True]
    for register in (nn_module.register_module_forward_hook, nn_module.register_module_forward_pre_hook,
                     nn_module.register_module_full_backward_hook, conv.register_forward_hook, linear.register_full_backward_hook):
        handle = register(see)
        assert taken() == [getattr(register, "__self__", conv) is not conv, getattr(register, "__self__", linear) is not linear]
        handle.remove()
    conv.forward, linear.forward = conv.forward, linear.forward
    assert taken() == [False, False]
    del conv.forward, linear.forward
    assert taken() == [True, True]


def test_single_call_core_leaves_steps_of_an_instance_alone(monkeypatch):
    """A step replaced on the instance is part of what forward_core does, as one of a subclass is: the single call does not stand
    for it."""
    from vmamba_amd import ss2d
    monkeypatch.setattr(ss2d, "forward_core_hip", lambda *args: "called")
    op, x = ss2d.SS2D(d_model=16), _OnGpu(torch.zeros(1, 16, 8, 8))
    with torch.no_grad():
        for step in ("forward_core_fused", "finish_core", "_inference_constants"):
            assert op._forward_core_native(x, True) == "called"
            setattr(op, step, getattr(op, step))
            assert op._forward_core_native(x, True) is None
            delattr(op, step)


def test_operators_seen():
    """What may see or replace the operators that modules call, and what does not."""
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    from vmamba_amd.norm import operators_seen

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert not operators_seen()
    for context in (Functions(), FlopCounterMode(display=False), forward_ad.dual_level()):
        with context:
            assert operators_seen()
    with torch.device("cpu"):
        assert not operators_seen()
        with Functions():
            assert operators_seen()
    seen = []
    for transform in (torch.func.vmap(lambda t: seen.append(operators_seen()) or t), torch.func.grad(lambda t: seen.append(operators_seen()) or t.sum())):
        transform(torch.ones(2))
    assert seen == [True, True]
    forward = torch.nn.Linear.forward
    try:
        torch.nn.Linear.forward = lambda self, x: forward(self, x)
        assert operators_seen()
    finally:
        torch.nn.Linear.forward = forward
    assert not operators_seen()


def test_mlp_backward_of_a_batch_of_gradients():
    """MlpF32's backward takes torch's operators for gradients without memory of their own (sizes the kernels are not asked for)."""
    from vmamba_amd.linear import MlpF32
    torch.manual_seed(0)
    x, w1, b1, w2, b2 = wanted = [torch.randn(*s, requires_grad=True) for s in ((5, 8), (12, 8), (12,), (8, 12), (8,))]
    dys = torch.randn(3, 5, 8)
    want = torch.nn.functional.linear(torch.nn.functional.gelu(torch.nn.functional.linear(x, w1, b1)), w2, b2)
    for got, ref in zip(torch.autograd.grad(MlpF32.apply(*wanted), wanted, dys, is_grads_batched=True), torch.autograd.grad(want, wanted, dys, is_grads_batched=True)):
        assert torch.allclose(got, ref, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("name", ["linear", "gelu", "layer_norm"])
def test_replaced_functions_are_not_passed_by(name, monkeypatch):
    """What LayerNorm and the MLP call in training, replaced by the user: no kernel stands for it."""
    from vmamba_amd.norm import calls_unseen
    function = getattr(torch.nn.functional, name)
    assert calls_unseen()
    monkeypatch.setattr(torch.nn.functional, name, lambda *a, **k: function(*a, **k))
    assert not calls_unseen()


@pytest.mark.parametrize("on", ["class", "instance"])
def test_replaced_projections_get_the_constants_they_had(on, monkeypatch):
    """project_from_map of a subclass, or set on the instance, is called in training with the weights repeated over the images, as at any size."""
    from vmamba_amd import ss2d
    monkeypatch.setattr(ss2d, "projections_train", lambda *args: True)

    class Called(Exception):
        pass

    def project_from_map(self, x, consts):
        raise Called(sorted(consts))

    kind = type("Own", (SS2D,), {"project_from_map": project_from_map}) if on == "class" else SS2D
    op = kind(d_model=16)
    if on == "instance":
        op.project_from_map = lambda x, consts: project_from_map(op, x, consts)
    with pytest.raises(Called) as called:
        op.forward_core(torch.zeros(1, 16, 4, 4))
    assert {"Wx_all", "Wx", "Wdt"} <= set(called.value.args[0])


def test_weights_of_another_kind_are_left_to_their_layer():
    """A weight that is another kind of tensor answers the layer's own call in training: LinearDw would read its memory."""
    from vmamba_amd.linear import linear_dw_pays

    class Kind(torch.Tensor):
        pass

    layer, rows = torch.nn.Linear(8, 8, bias=False), _OnGpu(torch.zeros(4096, 8))
    rows.device = torch.device("cpu")                                # the weight's own
    assert linear_dw_pays(layer, rows)
    layer.weight = torch.nn.Parameter(layer.weight.detach().as_subclass(Kind))
    assert type(layer.weight) is Kind and not linear_dw_pays(layer, rows)
