"""ss2d_forward_core is the same kernels in the same order as the separate calls: the same bits, over every form it takes."""
import pytest
import torch

from vmamba_amd import ss2d
from vmamba_amd.core import core_fits
from vmamba_amd.ss2d import SS2D

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("channel_first", [False, True])
@pytest.mark.parametrize("B,D,H,W", [(1, 768, 7, 7), (3, 192, 14, 14), (2, 96, 28, 28), (5, 48, 9, 8),
                                     (1, 64, 128, 128), (1, 8, 3, 3),
                                     # embedded in larger maps: in LDS, in tiles, a rank without a masked projection, 3 x 5 where padding does not pay
                                     (2, 96, 19, 19), (3, 64, 25, 42), (1, 96, 57, 58), (1, 192, 33, 35), (1, 384, 34, 33), (1, 768, 33, 33), (1, 32, 123, 125), (1, 800, 9, 9), (2, 16, 3, 5)])
def test_same_bits(B, D, H, W, dtype, channel_first, monkeypatch):
    print("CASE forward_core", B, D, H, W, dtype, channel_first, flush=True)
    torch.manual_seed(H)
    taken, native = [], ss2d.forward_core_hip
    monkeypatch.setattr(ss2d, "forward_core_hip", lambda *a: taken.append(native(*a)) or taken[-1])
    op = SS2D(d_model=D, channel_first=channel_first).to(DEV).to(dtype).eval()
    with torch.no_grad():
        op.out_norm.weight.uniform_(0.5, 1.5)
        op.out_norm.bias.uniform_(-1, 1)
        x = torch.randn(B, D, H, W, device=DEV).to(dtype)
        got, turned = op.forward_core(x), op.forward_core(x.transpose(2, 3))
        mixed = SS2D(d_model=D, channel_first=channel_first).to(DEV).to(dtype).eval()
        mixed.load_state_dict(op.state_dict())
        mixed.out_norm.float()                                     # norm parameters of another type than the map's
        got_mixed = mixed.forward_core(x) if dtype != torch.float16 else None      # (the norm kernel has no such pair)
        # the cases the single call is for are its own, not the separate calls compared with themselves
        if op.dt_rank <= (24 if dtype == torch.float32 else 48) and core_fits(H, W, dtype):
            assert len(taken) == 2 + (got_mixed is not None) and all(t is not None for t in taken)
        else:
            assert all(t is None for t in taken)
        monkeypatch.setattr(SS2D, "_forward_core_native", lambda self, x, normalise: None)
        assert torch.equal(got, op.forward_core(x)) and torch.equal(turned, op.forward_core(x.transpose(2, 3)))
        assert got_mixed is None or torch.equal(got_mixed, mixed.forward_core(x))


def test_who_takes_it(monkeypatch):
    calls = []
    native = ss2d.forward_core_hip
    monkeypatch.setattr(ss2d, "forward_core_hip", lambda *a: calls.append(native(*a)) or calls[-1])
    op = SS2D(d_model=96, channel_first=False).to(DEV).bfloat16().eval()
    x = torch.randn(2, 96, 14, 14, device=DEV).bfloat16()
    with torch.no_grad():
        op.forward_core(x)
        assert len(calls) == 1 and calls[0] is not None
        op.forward_core(x[:0])                                     # empty: the separate kernels' own answers
        SS2D(d_model=96, d_state=2, channel_first=False).to(DEV).bfloat16().eval().forward_core(x)
        assert len(calls) == 1

        class Own(SS2D):
            def finish_core(self, *args):
                return super().finish_core(*args) * 2
        own = Own(d_model=96, channel_first=False).to(DEV).bfloat16().eval()
        own.load_state_dict(op.state_dict())
        assert torch.equal(own.forward_core(x), op.forward_core(x) * 2) and len(calls) == 2
    op.float().forward_core(x.float().requires_grad_())            # autograd: the differentiable operators
    assert len(calls) == 2


def test_on_a_side_stream_and_captured():
    op = SS2D(d_model=192, channel_first=False).to(DEV).bfloat16().eval()
    x = torch.randn(2, 192, 14, 14, device=DEV).bfloat16()
    side = torch.cuda.Stream()
    with torch.no_grad():
        want = op.forward_core(x)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            other = op.forward_core(x)
        torch.cuda.current_stream().wait_stream(side)
        assert torch.equal(other, want)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = op.forward_core(x)
        for _ in range(3):
            x.copy_(torch.randn(2, 192, 14, 14, device=DEV))
            graph.replay()
            eager = op.forward_core(x)
            torch.cuda.synchronize()
            assert torch.equal(y, eager)
