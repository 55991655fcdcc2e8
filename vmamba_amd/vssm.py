"""VMamba-T-shaped backbone used as the throughput harness (random init, inference).

Layer order and shapes follow VSSM / VSSBlock of classification/models/vmamba.py:1153-1505 for
the ``vmamba_tiny_s1l8`` recipe (:1717-1728): patch-embed v2, downsample v3, depths 2/2/8/2, dims
96/192/384/768, d_state 1, ssm_ratio 1, forward type v05_noz, MLP ratio 4.  As in the reference the
same weights run in two activation layouts: ``channel_first=True`` ("ln2d": (B,C,H,W), 1x1 convs,
LayerNorm2d) and ``channel_first=False`` ("ln": (B,H,W,C), nn.Linear, nn.LayerNorm).  The norm
layers come from ``layers`` (default: this package's HIP LayerNorm kernels); convolutions, the projection and
MLP GEMMs and activations are stock torch; drop-path is the identity at inference.

Module names -- hence state_dict keys -- are the reference's (``patch_embed.{0,2,5,7}``,
``layers.{i}.blocks.{j}.{norm,op,norm2,mlp}``, ``layers.{i}.downsample.{1,3}``, ``classifier.{norm,head}``), and
``VSSM._load_from_state_dict`` applies the reference's renames for checkpoints written by its older training code
(vmamba.py:1531-1570), so a released VMamba checkpoint of this architecture loads with ``load_state_dict``.
"""
from collections import OrderedDict

import torch
import torch.nn as nn

from .block import vss_block_hip
from .linear import TENSOR_KINDS, MlpF32, few_positions, linear_rows_fusable, linear_rows_hip, linear_rows_takes, linear_tiles_fusable, linear_tiles_hip, mlp_f32_pays
from .mlp import mlp_fusable, mlp_fused_hip
from .norm import LayerNorm as HipLayerNorm
from .norm import add_layer_norm_fusable, add_layer_norm_hip, bias_layer_norm_fusable, bias_layer_norm_hip, needs_grad, observed
from .ss2d import SS2D, HipLayers, Linear2d
from .pool import GlobalAvgPool2d
from .stem import conv_tiles_fusable, conv_tiles_hip, stem2_fusable, stem_conv2_ln_hip, stem_conv_ln_gelu_hip, stem_fusable


class Permute(nn.Module):
    def __init__(self, *dims):
        super().__init__()
        self.dims = dims

    def forward(self, x):
        return x.permute(*self.dims)


def _to_cl(channel_first):      # (B,C,H,W) -> block layout
    return nn.Identity() if channel_first else Permute(0, 2, 3, 1)


def _to_cf(channel_first):      # block layout -> (B,C,H,W)
    return nn.Identity() if channel_first else Permute(0, 3, 1, 2)


class ConvNormSequence(nn.Sequential):
    """The patch-embedding and downsampling stacks (vmamba.py:1403-1417, 1430-1437).  Where a Conv2d with a bias is
    followed by the permute to channel-last and this package's LayerNorm, the convolution runs without its bias and
    the LayerNorm kernel adds it on the way in (ss2d_bias_layer_norm): one pass over the activation fewer."""

    def forward(self, x):
        mods = list(self)
        i = 0
        while i < len(mods):
            conv = mods[i]
            if i + 4 < len(mods) and self._stem(x, conv, *mods[i + 1:i + 5]):
                norm = mods[i + 2]                    # conv, LayerNorm and GELU in one kernel; the result is channel-last
                x = stem_conv_ln_gelu_hip(x, conv.weight, conv.bias, norm.weight, norm.bias, norm.eps).permute(0, 3, 1, 2)
                i += 5
            elif i + 2 < len(mods) and self._fusable(x, conv, mods[i + 1], mods[i + 2]):
                norm = mods[i + 2]
                if stem2_fusable(x, conv, norm):      # convolution and LayerNorm in one kernel
                    x = stem_conv2_ln_hip(x.permute(0, 2, 3, 1), conv.weight, conv.bias, norm.weight, norm.bias, norm.eps)
                    i += 3
                    continue
                if conv_tiles_fusable(x, conv):
                    x = conv_tiles_hip(x.permute(0, 2, 3, 1), conv.weight)
                else:
                    x = conv._conv_forward(x, conv.weight, None).permute(0, 2, 3, 1)
                x = bias_layer_norm_hip(x, conv.bias, norm.weight, norm.bias, norm.eps)
                i += 3
            else:
                x = conv(x)
                i += 1
        return x

    @staticmethod
    def _stem(x, conv, to_cl, norm, to_cf, act):
        return (isinstance(conv, nn.Conv2d) and isinstance(to_cl, Permute) and tuple(to_cl.dims) == (0, 2, 3, 1)
                and isinstance(norm, HipLayerNorm) and isinstance(to_cf, Permute) and tuple(to_cf.dims) == (0, 3, 1, 2)
                and isinstance(act, nn.GELU) and stem_fusable(x, conv, norm, act)
                and not needs_grad(x, conv.weight, conv.bias, norm.weight, norm.bias))

    @staticmethod
    def _fusable(x, conv, permute, norm):
        return (isinstance(conv, nn.Conv2d) and conv.bias is not None and isinstance(permute, Permute)
                and tuple(permute.dims) == (0, 2, 3, 1) and isinstance(norm, HipLayerNorm) and norm.elementwise_affine
                and x.is_cuda and x.dim() == 4 and bias_layer_norm_fusable(x.dtype, conv.out_channels)
                and not needs_grad(x, conv.weight, conv.bias, norm.weight, norm.bias))


class Mlp(nn.Module):
    def __init__(self, dim, hidden, channel_first=True, fused=True):
        super().__init__()
        self.channel_first, self.fused = channel_first, fused
        Linear = Linear2d if channel_first else nn.Linear
        self.fc1 = Linear(dim, hidden)
        self.act = nn.GELU()
        self.fc2 = Linear(hidden, dim)

    def takes_norm(self, x, norm=None):
        """True when forward runs a fused kernel for x, which then takes the preceding LayerNorm (``norm``) as a prologue."""
        if norm is not None and few_positions(x) and self._rows(x, norm):
            return True
        return (self.fused and not self.channel_first and mlp_fusable(x, self.fc1, self.fc2)
                and not needs_grad(x, self.fc1.weight, self.fc2.weight, self.fc1.bias, self.fc2.bias))

    def _rows(self, x, norm):
        """True when two launches of ss2d_linear_rows stand for norm, fc1, act, fc2 and the add on x: few positions."""
        return (self.fused and not self.channel_first and linear_rows_fusable(x, self.fc1, norm) and type(self.act) is nn.GELU
                and self.act.approximate == "none" and not observed(self.act) and linear_rows_takes(self.fc2, x)
                and self.fc2.weight.shape[1] == self.fc1.out_features)

    def forward(self, x, residual=None, pre_norm=None):
        """fc2(GELU(fc1(h))) (+ residual), h = x or pre_norm(x) (the block's second LayerNorm, vmamba.py:1229).
        Channel-last 16-bit inference at widths 96 / 192 runs as one HIP kernel that normalises the rows on the way
        in and keeps the hidden activations in registers; few positions behind a norm as two launches of ss2d_linear_rows at
        any width; many positions of a wider layer with the GELU behind fc1's product (ss2d_linear_tiles); single-precision training on the products of ss2d_product_f32 where those are the faster ones (MlpF32); everything else
        on the torch operators.  A residual that the kernels cannot add -- one that autograd has to
        see, of another shape, type, device or kind -- is added by torch behind them."""
        rows = pre_norm is not None and few_positions(x) and self._rows(x, pre_norm)
        one = (not rows and self.fused and not self.channel_first and mlp_fusable(x, self.fc1, self.fc2)
               and not needs_grad(x, self.fc1.weight, self.fc2.weight, self.fc1.bias, self.fc2.bias)
               and (pre_norm is None or (isinstance(pre_norm, nn.LayerNorm) and pre_norm.elementwise_affine
                                         and not needs_grad(pre_norm.weight, pre_norm.bias))))
        add = residual if (rows or one) and residual is not None and (residual is x or self._adds(x, residual)) else None       # by the kernel
        if rows:
            h = linear_rows_hip(x, self.fc1.weight, self.fc1.bias, None, pre_norm.weight, pre_norm.bias, pre_norm.eps, gelu=True)
            y = linear_rows_hip(h, self.fc2.weight, self.fc2.bias, add)
        elif one:
            norm = () if pre_norm is None else (pre_norm.weight, pre_norm.bias, pre_norm.eps)
            y = mlp_fused_hip(x, self.fc1.weight, self.fc1.bias, self.fc2.weight, self.fc2.bias, add, *norm)
        else:
            h = x if pre_norm is None else pre_norm(x)
            if self.fused and not self.channel_first and mlp_f32_pays(h, self.fc1, self.act, self.fc2):
                y = MlpF32.apply(h, self.fc1.weight, self.fc1.bias, self.fc2.weight, self.fc2.bias)
            elif self.fused and not self.channel_first and linear_tiles_fusable(h, self.fc1, self.act):
                y = self.fc2(linear_tiles_hip(h, self.fc1.weight, self.fc1.bias, gelu=True))
            else:
                y = self.fc2(self.act(self.fc1(h)))
        return y if residual is None or add is not None else residual + y

    @staticmethod
    def _adds(x, residual):
        """True when the kernels' own addition stands for ``residual + y``, y of x's shape and type."""
        return (type(residual) in TENSOR_KINDS and residual.shape == x.shape and residual.dtype == x.dtype and residual.device == x.device
                and not needs_grad(residual) and (residual.data_ptr() % 16 == 0 or not residual.is_contiguous()))


_STEPS = SS2D.forward, Mlp.forward, Mlp.takes_norm


class VSSBlock(nn.Module):
    def __init__(self, dim, d_state=1, ssm_ratio=1.0, mlp_ratio=4.0, ss2d_cls=SS2D, channel_first=True, layers=HipLayers,
                 **ss2d_kwargs):
        super().__init__()
        Norm = layers.LayerNorm2d if channel_first else layers.LayerNorm
        self.norm = Norm(dim)
        self.op = ss2d_cls(d_model=dim, d_state=d_state, ssm_ratio=ssm_ratio, channel_first=channel_first, layers=layers,
                           **ss2d_kwargs)
        self.norm2 = Norm(dim)
        self.mlp = Mlp(dim, int(dim * mlp_ratio), channel_first)

    def forward(self, x):
        x, pending = self.step(x, None)
        return x if pending is None else x + pending

    def step(self, x, pending):
        """One block on the residual stream x, with ``pending`` (or None) a term the previous block has not added to x
        yet; returns (x, pending) in the same sense.  Deferring the MLP's residual add lets the next block do it
        together with its first LayerNorm in one kernel (ss2d_add_layer_norm); it is only deferred where that kernel
        exists (channel-last 16-bit inference)."""
        inp, pre = x, self.norm
        if pending is not None:
            if self._fusable_add_norm(x, pending, self.norm):
                x, inp = add_layer_norm_hip(pending, x, self.norm.weight, self.norm.bias, self.norm.eps)
                pre = None
            else:
                x = inp = x + pending
        few = few_positions(x) and Mlp.forward is _STEPS[1]
        native = vss_block_hip(self, Mlp, inp, x if pre is None else None) if few else None       # as one call
        if native is not None:
            x, whole = native
            if whole:
                return x, None
            if self.mlp.takes_norm(x, self.norm2):
                return self.mlp(x, residual=x, pre_norm=self.norm2), None
            return self._pending_mlp(x, self.norm2(x))
        # the fused MLP kernels normalise their input themselves
        if self.mlp.takes_norm(x, self.norm2) if few and self._steps_as_written() else self.mlp.takes_norm(x):
            x = self.op(inp, residual=x, pre_norm=pre)
            return self.mlp(x, residual=x, pre_norm=self.norm2), None
        x, h = self.op(inp, residual=x, pre_norm=pre, post_norm=self.norm2)
        return self._pending_mlp(x, h)

    def _steps_as_written(self):
        """True when nothing sees or replaces the calls of op and mlp, whose arguments and results with few positions are others than
        with many: an MLP of another kind is called with norm2's result, as everywhere beyond widths 96 and 192."""
        op, mlp = self.op, self.mlp
        return (isinstance(mlp, Mlp) and (getattr(type(op), "forward", None), type(mlp).forward, type(mlp).takes_norm) == _STEPS
                and not observed(op) and not observed(mlp))

    def _pending_mlp(self, x, h):
        m = self.mlp(h)
        if self._fusable_add_norm(x, m, self.norm):
            return x, m
        return x + m, None

    def _fusable_add_norm(self, x, term, norm):
        return (not self.op.channel_first and isinstance(norm, nn.LayerNorm) and norm.elementwise_affine
                and add_layer_norm_fusable(x, term) and x.dtype != torch.float32
                and not needs_grad(x, term, norm.weight, norm.bias))


class BlockSequence(nn.Sequential):
    """The blocks of one stage; threads the deferred residual term from block to block (see VSSBlock.step)."""

    def forward(self, x):
        pending = None
        for block in self:
            x, pending = block.step(x, pending)
        return x if pending is None else x + pending


class VSSM(nn.Module):
    def __init__(self, in_chans=3, num_classes=1000, depths=(2, 2, 8, 2), dims=(96, 192, 384, 768), d_state=1,
                 ssm_ratio=1.0, mlp_ratio=4.0, ss2d_cls=SS2D, channel_first=True, layers=HipLayers, **ss2d_kwargs):
        super().__init__()
        self._build_args = dict(in_chans=in_chans, num_classes=num_classes, depths=tuple(depths), dims=tuple(dims), d_state=d_state,
                                ssm_ratio=ssm_ratio, mlp_ratio=mlp_ratio, ss2d_cls=ss2d_cls, layers=layers, **ss2d_kwargs)
        cf = channel_first
        Norm = layers.LayerNorm2d if cf else layers.LayerNorm
        d0 = dims[0]
        self.patch_embed = ConvNormSequence(
            nn.Conv2d(in_chans, d0 // 2, kernel_size=3, stride=2, padding=1), _to_cl(cf), Norm(d0 // 2), _to_cf(cf),
            nn.GELU(),
            nn.Conv2d(d0 // 2, d0, kernel_size=3, stride=2, padding=1), _to_cl(cf), Norm(d0))
        stages = []
        for i, (depth, dim) in enumerate(zip(depths, dims)):
            blocks = [VSSBlock(dim, d_state, ssm_ratio, mlp_ratio, ss2d_cls, cf, layers, **ss2d_kwargs) for _ in range(depth)]
            down = (ConvNormSequence(_to_cf(cf), nn.Conv2d(dim, dims[i + 1], kernel_size=3, stride=2, padding=1), _to_cl(cf),
                                  Norm(dims[i + 1]))
                    if i + 1 < len(dims) else nn.Identity())
            stages.append(nn.Sequential(OrderedDict(blocks=BlockSequence(*blocks), downsample=down)))
        self.layers = nn.ModuleList(stages)
        self.classifier = nn.Sequential(OrderedDict(
            norm=Norm(dims[-1]), permute=_to_cf(cf), avgpool=GlobalAvgPool2d(), flatten=nn.Flatten(1),
            head=nn.Linear(dims[-1], num_classes)))
        self.apply(self._init_weights)

    # key prefixes of checkpoints from the reference's previous training code -> current names (vmamba.py:1557-1564)
    LEGACY_KEYS = (("patch_embed.proj", "patch_embed.0"), ("patch_embed.norm", "patch_embed.2"),
                   ("norm", "classifier.norm"), ("head", "classifier.head"))
    LEGACY_BLOCK_KEYS = (("ln_1", "norm"), ("self_attention", "op"))

    def _load_from_state_dict(self, state_dict, prefix, *args, **kwargs):
        def rename(src, dst):
            for key in [k for k in state_dict if k.startswith(prefix + src)]:
                state_dict[prefix + dst + key[len(prefix + src):]] = state_dict.pop(key)

        for i, stage in enumerate(self.layers):
            for j in range(len(stage.blocks)):
                for src, dst in self.LEGACY_BLOCK_KEYS:
                    rename(f"layers.{i}.blocks.{j}.{src}", f"layers.{i}.blocks.{j}.{dst}")
        for src, dst in self.LEGACY_KEYS:
            rename(src, dst)
        return super()._load_from_state_dict(state_dict, prefix, *args, **kwargs)

    @staticmethod
    def _init_weights(m):
        if isinstance(m, nn.Linear):
            nn.init.trunc_normal_(m.weight, std=0.02)
            if m.bias is not None:
                nn.init.zeros_(m.bias)
        elif isinstance(m, nn.LayerNorm):
            nn.init.ones_(m.weight)
            nn.init.zeros_(m.bias)

    def forward(self, x):
        x = self.patch_embed(x)
        for layer in self.layers:
            x = layer(x)
        return self.classifier(x)

    def with_layout(self, channel_first, share_weights=False):
        """The same model (same device, dtype and mode) with its blocks in the other activation layout.  The reference's
        "ln2d" configurations build channel-first blocks (vmamba.py:1281); the two layouts compute the same function and
        share one state_dict (a Linear2d weight is a view of the nn.Linear one, vmamba.py:47-49), and the channel-last
        build is the one whose projections, MLPs and LayerNorms run on this package's fused kernels.

        The twin holds a copy of the weights, or -- ``share_weights=True`` -- the very same Parameter and buffer objects
        (every parameter has the same shape in both builds), so that loading, casting, moving or training either model
        is seen by the other."""
        twin = VSSM(channel_first=channel_first, **self._build_args)
        if not share_weights:
            twin.load_state_dict(self.state_dict())
            p = next(self.parameters())
            return twin.to(device=p.device, dtype=p.dtype).train(self.training)
        mine = dict(self.named_modules())
        for name, module in twin.named_modules():
            src = mine[name]
            for key in list(module._parameters):
                module._parameters[key] = src._parameters[key]
            for key in list(module._buffers):
                module._buffers[key] = src._buffers[key]
        return twin.train(self.training)


def vmamba_tiny_s1l8(channel_first=True, **kwargs):
    return VSSM(depths=(2, 2, 8, 2), dims=(96, 192, 384, 768), d_state=1, ssm_ratio=1.0, mlp_ratio=4.0,
                channel_first=channel_first, **kwargs)
