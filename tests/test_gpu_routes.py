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


def names(y):
    """The names of the autograd nodes behind y."""
    seen, todo = set(), [y.grad_fn]
    while todo:
        f = todo.pop()
        if f is not None and f not in seen:
            seen.add(f)
            todo += [g for g, _ in f.next_functions]
    return {f.name() for f in seen}


def test_untouched_block_runs_in_the_extension(gpu_device):
    import torch.nn.utils.parametrize as P
    x = torch.randn(2, 9, 7, 24, device=gpu_device)
    blk = block(gpu_device)
    assert any("Ss2dFn" in n for n in names(blk(x)))
    P.register_parametrization(blk.op.conv2d, "weight", nn.Identity())
    assert not any("Ss2dFn" in n for n in names(blk(x)))


def layers(dev):
    """A norm and a linear layer of the block, each beside torch's own with the same parameters."""
    import selective_nd_scan as snd
    torch.manual_seed(14)
    for layer, plain in ((snd.vss_block.TokenNorm(24), nn.LayerNorm(24)), (snd.vss_block.TokenLinear(24, 8), nn.Linear(24, 8))):
        for p in layer.parameters():
            p.data.add_(0.1 * torch.randn_like(p))
        plain.load_state_dict(layer.state_dict())
        yield layer.to(dev, torch.bfloat16), plain.to(dev, torch.bfloat16)


def test_layers_in_forward_mode_and_transforms(gpu_device):
    import torch.autograd.forward_ad as fwad
    x, t = (torch.randn(3, 5, 24, device=gpu_device, dtype=torch.bfloat16) for _ in range(2))
    for layer, plain in layers(gpu_device):
        with fwad.dual_level():
            got, want = (fwad.unpack_dual(m(fwad.make_dual(x, t))).tangent for m in (layer, plain))
        assert torch.equal(got, want)
        assert torch.equal(torch.func.vmap(layer)(x), torch.func.vmap(plain)(x))
        got, want = (torch.func.grad(lambda v: m(v).float().square().sum())(x) for m in (layer, plain))
        assert torch.equal(got, want)


def test_layers_are_seen_by_modes_tracing_and_compilers(gpu_device):
    from torch.utils._python_dispatch import TorchDispatchMode

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Logged(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            seen.append(func.__name__)
            return super().__torch_function__(func, types, args, kwargs or {})

    x = torch.randn(5, 24, device=gpu_device, dtype=torch.bfloat16)
    for layer, name in zip((l for l, _ in layers(gpu_device)), ("layer_norm", "linear")):
        seen = []
        with Log():
            want = layer(x)
        assert any(n in s for s in seen for n in ("layer_norm", "addmm"))
        seen = []
        layer(x.as_subclass(Logged))
        assert name in seen
        traced = torch.jit.trace(layer, (x,), check_trace=False)
        assert name in str(traced.inlined_graph)
        assert rel(torch.compile(layer, backend="eager", fullgraph=True)(x), want) <= 1e-2


def test_compiled_block(gpu_device):
    blk = block(gpu_device)
    both(torch.compile(blk, backend="eager"), blk, torch.randn(2, 9, 7, 24, device=gpu_device))


def test_parameters_that_torch_refuses_stay_refused(gpu_device):
    import selective_nd_scan as snd
    x = torch.randn(5, 24, device=gpu_device)
    with pytest.raises(RuntimeError):
        snd.vss_block.TokenNorm(24).to(gpu_device, torch.float16)(x)
    with pytest.raises(RuntimeError):
        snd.vss_block.TokenLinear(24, 8).to(gpu_device, torch.float16)(x)
    op = block(gpu_device).op
    op.out_norm.to(torch.float16)
    with pytest.raises(RuntimeError):
        op(x.view(1, 1, 5, 24))


def test_many_images(gpu_device):
    """More (image, direction) pairs than a grid of the block's passes has rows."""
    blk = block(gpu_device, width=8, states=1, mlp=0.0)
    x = torch.randn(16384, 1, 1, 8, device=gpu_device)
    y, first = blk(x), blk(x[:16383])
    assert rel(y[:16383], first) <= 2e-5
    # (the gradient of a parameter behind the convolution: torch's own 3x3 backward is slow to set up at this size)
    g, last = (torch.autograd.grad(v.square().sum(), blk.op.A_logs)[0] for v in (y, blk(x[16383:])))
    assert rel(g, torch.autograd.grad(first.square().sum(), blk.op.A_logs)[0] + last) <= 1e-4


def test_deterministic_algorithms(gpu_device):
    """Bit for bit the same parameter gradients from run to run, in the layers and in a block around its scan."""
    import selective_nd_scan as snd
    lin, norm = snd.vss_block.TokenLinear(96, 384).to(gpu_device), snd.vss_block.TokenNorm(96).to(gpu_device)
    x, dy = torch.randn(8000, 96, device=gpu_device), torch.randn(8000, 384, device=gpu_device, dtype=torch.bfloat16)
    blk = block(gpu_device)
    torch.use_deterministic_algorithms(True)
    try:
        def once():
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = lin(norm(x))
            return torch.autograd.grad(y, list(lin.parameters()) + list(norm.parameters()), dy)
        first = once()
        for _ in range(5):
            assert all(torch.equal(a, b) for a, b in zip(first, once()))
        assert not any("Ss2dFn" in n for n in names(blk(x.view(10, 20, 40, 96)[..., :24].contiguous())))
    finally:
        torch.use_deterministic_algorithms(False)


@pytest.mark.parametrize("tokens,M,N", [(300, 64, 32), (300, 33, 32), (40, 1024, 1026)])
@pytest.mark.parametrize("frozen", [(), ("weight",), ("bias",), ("weight", "bias")])
def test_frozen_parameters_of_a_linear_layer(gpu_device, tokens, M, N, frozen):
    """Both sides of the rule for the weight gradient; what is frozen has no gradient, the rest those of torch's layer."""
    import selective_nd_scan as snd
    torch.manual_seed(16)
    layer = snd.vss_block.TokenLinear(N, M).to(gpu_device, torch.bfloat16)
    plain = nn.Linear(N, M).to(gpu_device, torch.float32)
    plain.load_state_dict(layer.state_dict())
    x, dy = torch.randn(tokens, N, device=gpu_device), torch.randn(tokens, M, device=gpu_device)
    for m in (layer, plain):
        for n in frozen:
            getattr(m, n).requires_grad_(False)
    xs = [x.bfloat16().requires_grad_(), x.bfloat16().float().requires_grad_()]
    layer(xs[0]).backward(dy.bfloat16())
    plain(xs[1]).backward(dy.bfloat16().float())
    assert rel(xs[0].grad, xs[1].grad) <= 5e-3          # (results in bf16: half an ulp is 2^-9)
    for n in ("weight", "bias"):
        a, b = getattr(layer, n).grad, getattr(plain, n).grad
        assert (a is None) == (n in frozen) and (a is None or rel(a, b) <= 5e-3)


@pytest.mark.parametrize("tokens,M,N,kernel", [(32769, 1024, 512, True), (32768, 1026, 512, True), (32769, 1026, 512, False), (65, 1024, 768, True),
                                               (65, 1024, 770, False), (65, 31, 34, False)])
def test_rule_for_linear_weight_gradients(gpu_device, tokens, M, N, kernel):
    """The kernel's sums are fp32 (1e-5 by their order), the library's result is rounded to bf16 (2^-9 at most, 1e-3 on average)."""
    from selective_nd_scan.interface import ext
    torch.manual_seed(18)
    x, dy = (torch.randn(tokens, n, device=gpu_device, dtype=torch.bfloat16) for n in (N, M))
    w, b = torch.randn(M, N, device=gpu_device).requires_grad_(), torch.randn(M, device=gpu_device).requires_grad_()
    dw, db = torch.autograd.grad(ext().block_linear(x, w, b, x), (w, b), dy)
    for got, want in ((dw, dy.double().t() @ x.double()), (db, dy.double().sum(0))):
        assert rel(got, want) <= (1e-5 if kernel else 4e-3) and (kernel or rel(got, want) >= 1e-4)


def test_norms_are_float32_where_somebody_else_reads_them(gpu_device):
    """Under autocast a norm's result is rounded to 16 bits only for a linear layer that would do so itself."""
    import selective_nd_scan as snd
    x = torch.randn(2, 9, 7, 24, device=gpu_device)

    def run(blk):
        seen = {}
        for n, m in (("op", blk.op), ("mlp", blk.mlp)):
            m.register_forward_pre_hook(lambda mod, i, n=n: seen.update({n: i[0].dtype}))
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = blk(x)
        return y, seen

    blk = block(gpu_device)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert blk.norm(x).dtype == torch.float32 and blk.norm(x, True).dtype == torch.bfloat16
        plain = blk(x)
    y, seen = run(blk)
    assert seen == dict(op=torch.float32, mlp=torch.float32) and torch.equal(y, plain)
    blk = block(gpu_device)
    inner = blk.op.in_proj
    got = []

    class Wide(nn.Module):                           # a projection that keeps to float32
        def forward(self, v):
            got.append(v.dtype)
            with torch.autocast("cuda", enabled=False):
                return inner(v.float())

    blk.op.in_proj = Wide()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        blk(x)
    assert got == [torch.float32]
