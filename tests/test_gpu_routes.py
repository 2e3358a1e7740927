"""Which calls of the block run in the extension, and that what may not runs as the torch layers it stands for."""
import copy

import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float((a.detach().double() - b.detach().double()).norm() / b.detach().double().norm().clamp_min(1e-30))


def block(dev, width=24, states=3, mlp=2.0, **kw):
    import selective_nd_scan as snd
    torch.manual_seed(11)
    blk = snd.VSSBlock(width, d_state=states, ssm_ratio=1.0, mlp_ratio=mlp, **kw).to(dev)
    for p in blk.parameters():
        p.data.add_(0.02 * torch.randn_like(p))
    return blk


def torch_route(blk):
    """The same block with its scan through scan_fn: every other stage is a torch layer."""
    import selective_nd_scan as snd
    ref = copy.deepcopy(blk)
    ref.op.scan_fn = lambda *a: snd.four_corner_scan(*a)
    return ref


def both(blk, ref, x):
    a, b = (m(xi) for m, xi in ((blk, x), (ref, x)))
    assert rel(a, b) <= 2e-5
    for p, q in zip(torch.autograd.grad(a.square().sum(), list(blk.parameters())), torch.autograd.grad(b.square().sum(), list(ref.parameters()))):
        assert rel(p, q) <= 1e-4


def test_hooks_of_sub_modules_run(gpu_device):
    blk = block(gpu_device)
    x = torch.randn(2, 9, 7, 24, device=gpu_device)
    seen = []
    blk.op.conv2d.register_forward_hook(lambda m, i, o: seen.append("conv") or 2 * o)
    blk.op.out_norm.register_forward_pre_hook(lambda m, i: seen.append("norm"))
    ref = torch_route(blk)
    both(blk, ref, x)
    assert seen.count("conv") == 2 and seen.count("norm") == 2


def test_overridden_scan_inputs_is_used(gpu_device):
    import selective_nd_scan as snd

    class Half(snd.SS2DCrossScan):
        def scan_inputs(self, x):
            u, delta, *rest = super().scan_inputs(x)
            return (u, 0.5 * delta, *rest)

    blk = block(gpu_device)
    blk.op.__class__ = Half
    both(blk, torch_route(blk), torch.randn(2, 9, 7, 24, device=gpu_device))


@pytest.mark.parametrize("conv", [dict(dilation=2, padding=2), dict(padding=1, padding_mode="circular")])
def test_replaced_convolution_is_used(gpu_device, conv):
    blk = block(gpu_device)
    blk.op.conv2d = nn.Conv2d(24, 24, 3, groups=24, **conv).to(gpu_device)
    both(blk, torch_route(blk), torch.randn(2, 9, 7, 24, device=gpu_device))


@pytest.mark.parametrize("norm", [lambda: nn.LayerNorm(24, bias=False), lambda: nn.LayerNorm(24, elementwise_affine=False), lambda: nn.RMSNorm(24)])
def test_replaced_output_norm_is_used(gpu_device, norm):
    blk = block(gpu_device)
    blk.op.out_norm = norm().to(gpu_device)
    both(blk, torch_route(blk), torch.randn(2, 9, 7, 24, device=gpu_device))


def test_weight_pre_hook_of_the_convolution_runs(gpu_device):
    """A module that computes its weight on every call, as weight norm and pruning do."""
    blk = block(gpu_device)
    conv = blk.op.conv2d
    conv.register_forward_pre_hook(lambda m, i: [m.weight.data.fill_(0.25), None][1])
    both(blk, torch_route(blk), torch.randn(2, 9, 7, 24, device=gpu_device))


def test_untouched_block_runs_in_the_extension(gpu_device):
    import torch.nn.utils.parametrize as P
    x = torch.randn(2, 9, 7, 24, device=gpu_device)

    def names(blk):
        y, seen, todo = blk(x), set(), []
        todo.append(y.grad_fn)
        while todo:
            f = todo.pop()
            if f is not None and f not in seen:
                seen.add(f)
                todo += [g for g, _ in f.next_functions]
        return {f.name() for f in seen}

    blk = block(gpu_device)
    assert any("Ss2dFn" in n for n in names(blk))
    P.register_parametrization(blk.op.conv2d, "weight", nn.Identity())
    assert not any("Ss2dFn" in n for n in names(blk))
