"""The autograd functions at their boundary: what the state of autograd and autocast around a call, or around its
backward, may and may not change."""
import contextlib

import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float((a.detach().double() - b.detach().double()).norm() / b.detach().double().norm().clamp_min(1e-30))


def autocast(dtype):
    return contextlib.nullcontext() if dtype is None else torch.autocast("cuda", dtype=dtype)


def block(dev, **kw):
    import selective_nd_scan as snd
    torch.manual_seed(12)
    blk = snd.VSSBlock(24, d_state=3, ssm_ratio=2.0, mlp_ratio=2.0, **kw).to(dev)
    for p in blk.parameters():
        p.data.add_(0.02 * torch.randn_like(p))
    return blk


@pytest.mark.parametrize("fwd,bwd", [(None, torch.bfloat16), (None, torch.float16), (torch.bfloat16, torch.float16),
                                     (torch.float16, torch.bfloat16), (torch.bfloat16, torch.bfloat16)])
def test_backward_under_another_autocast(gpu_device, fwd, bwd):
    """The types of a backward are its forward's, whatever autocast does where backward() is called."""
    blk = block(gpu_device)
    if fwd is None:                                  # (torch's own linear layers take autocast's type in their backward)
        blk = blk.op
        blk.in_proj, blk.out_proj = nn.Identity(), nn.Identity()
    x = torch.randn(2, 9, 11, 24 if fwd else 96, device=gpu_device)
    dy = torch.randn(2, 9, 11, 24 if fwd else 48, device=gpu_device)
    grads = []
    for state in (None, bwd):
        xi = x.clone().requires_grad_()
        with autocast(fwd):
            y = blk(xi)
        with autocast(state):
            y.backward(dy)
        grads.append([xi.grad] + [p.grad for p in blk.parameters()])
        blk.zero_grad(set_to_none=True)
    # fp32: sums in another order.  16 bits: such a sum that lies at a rounding edge moves by one unit in the last place
    # (2^-8 in bf16) in a share of the values that is below 1e-2.
    for a, b in zip(*grads):
        assert a.dtype == b.dtype and rel(a, b) <= (1e-5 if fwd is None else 1e-3)


class Cast(nn.Module):
    def __init__(self, layer, dtype):
        super().__init__()
        self.layer, self.dtype = layer, dtype

    def forward(self, x):
        return self.layer(x).to(self.dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_in_proj_of_another_type_than_autocast(gpu_device, dtype):
    """What in_proj returns sets the type of the stages up to out_proj: here not autocast's."""
    blk = block(gpu_device)
    x = torch.randn(2, 9, 11, 24, device=gpu_device)
    dy = torch.randn_like(x)

    def run(forward):
        xi = x.clone().requires_grad_()
        forward(xi).backward(dy)
        r = [xi.grad] + [p.grad for p in blk.parameters()]
        blk.zero_grad(set_to_none=True)
        return r

    def cast(xi):
        with autocast(torch.bfloat16):
            return blk(xi)

    want = run(blk)                                  # fp32 throughout
    blk.op.in_proj = Cast(blk.op.in_proj, dtype)
    for a, b in zip(run(cast), want):
        assert rel(a, b) <= 2e-2                     # the roundings of the bf16 layers around


@pytest.mark.parametrize("grad", [torch.no_grad, torch.enable_grad])
def test_forward_mode_of_the_scan_is_refused(gpu_device, grad):
    import selective_nd_scan as snd
    import torch.autograd.forward_ad as fwad
    u, B = torch.randn(1, 8, 6, 6, device=gpu_device), torch.randn(1, 4, 2, 6, 6, device=gpu_device)
    A = -torch.ones(8, 2, device=gpu_device)
    with fwad.dual_level():
        dual = fwad.make_dual(u, torch.randn_like(u))
        with grad(), pytest.raises(RuntimeError, match="forward-mode"):
            snd.selective_nd_scan(dual, u, A, B, B)
        snd.selective_nd_scan(fwad.unpack_dual(dual).primal, u, A, B, B)


@pytest.mark.parametrize("C", [8, 16, 32])
def test_token_norm_refuses_another_last_axis(gpu_device, C):
    import selective_nd_scan as snd
    norm = snd.vss_block.TokenNorm(16).to(gpu_device)
    x = torch.randn(3, 16, C, device=gpu_device)
    if C == 16:
        assert norm(x).shape == x.shape
        return
    with pytest.raises(RuntimeError, match="normalized_shape"):
        norm(x)


def test_layers_refuse_parameters_elsewhere(gpu_device):
    import selective_nd_scan as snd
    from selective_nd_scan.interface import ext
    x = torch.randn(3, 16, device=gpu_device)
    w, b = torch.randn(16), torch.randn(16)
    with pytest.raises(RuntimeError, match="one device"):
        ext().block_norm(x, w, b.to(gpu_device), 1e-5, x)
    with pytest.raises(RuntimeError, match="one device"):
        ext().block_linear(x.bfloat16(), torch.randn(4, 16, device=gpu_device), torch.randn(4), x.bfloat16())
    with pytest.raises(RuntimeError):
        snd.vss_block.TokenNorm(16)(x)


@pytest.mark.parametrize("make,dtype", [(lambda v: (v.TokenNorm(24), nn.LayerNorm(24)), None),
                                        (lambda v: (v.TokenLinear(24, 8), nn.Linear(24, 8)), torch.bfloat16),
                                        (lambda v: (v.TokenLinear(24, 8, bias=False), nn.Linear(24, 8, bias=False)), torch.float16)])
def test_second_derivatives_of_layers(gpu_device, make, dtype):
    """create_graph through a norm or linear layer against torch's own layer in fp32."""
    import selective_nd_scan as snd
    torch.manual_seed(13)
    layer, plain = (m.to(gpu_device) for m in make(snd.vss_block))
    plain.load_state_dict(layer.state_dict())
    x, t = torch.randn(7, 24, device=gpu_device), torch.linspace(-1, 1, plain(torch.zeros(1, 24, device=gpu_device)).shape[-1], device=gpu_device)
    res = []
    for m in (layer, plain):
        xi = x.clone().requires_grad_()
        with autocast(dtype if m is layer else None):
            y = m(xi).float()
        params = [xi] + list(m.parameters())
        first = torch.autograd.grad((y + t).pow(3).sum(), params, create_graph=True)
        res.append([*first, *torch.autograd.grad(sum(g.pow(2).sum() for g in first), params)])
    # 16 bits: y, dy and their products are rounded on the way, three to four roundings of 2^-9 (bf16) in a term
    for a, b in zip(*res):
        assert rel(a, b) <= (1e-4 if dtype is None else 2e-2), rel(a, b)


def test_second_derivative_through_the_scan_is_refused(gpu_device):
    """Gradients under create_graph are those without it; differentiating them again raises instead of dropping terms."""
    import selective_nd_scan as snd
    blk = block(gpu_device)
    x = torch.randn(1, 6, 6, 24, device=gpu_device).requires_grad_()
    u, B = (torch.randn(1, 8, 6, 6, device=gpu_device).requires_grad_(), torch.randn(1, 4, 2, 6, 6, device=gpu_device))
    A = -torch.ones(8, 2, device=gpu_device)
    for leaf, f in ((x, lambda: blk(x)), (u, lambda: snd.selective_nd_scan(u, u, A, B, B, delta_softplus=True))):
        want, = torch.autograd.grad(f().square().sum(), leaf)
        g, = torch.autograd.grad(f().square().sum(), leaf, create_graph=True)
        assert rel(g, want) <= 1e-5
        with pytest.raises(RuntimeError, match="differentiated once"):
            g.square().sum().backward()


@pytest.mark.parametrize("merged", [False, True])
@pytest.mark.parametrize("train", [False, True])
def test_traced_scan(gpu_device, merged, train):
    """jit.trace records the scan as one operation, which runs on the inputs of a later call and has its gradient."""
    import selective_nd_scan as snd
    g = torch.Generator(device=gpu_device).manual_seed(15)
    rn = lambda *s: torch.randn(*s, device=gpu_device, generator=g)
    A = -torch.ones(8, 2, device=gpu_device)
    w = torch.linspace(0.5, 2, 8, device=gpu_device).view(4, 2)

    def f(u, delta, B):
        return (snd.cross_scan_2d(u, delta, A, B, B, merge_weights=w) if merged else snd.selective_nd_scan(u, delta, A, B, B, delta_softplus=True)) + 1

    def inputs(Bt):
        return [t.requires_grad_(train) for t in (rn(Bt, 2 if merged else 8, 6, 7), rn(Bt, 8, 6, 7), rn(Bt, 4, 2, 6, 7))]

    traced = torch.jit.trace(f, inputs(1), check_trace=False)
    x = inputs(2)
    got, want = traced(*x), f(*x)
    assert torch.equal(got, want)
    if train:
        dy = rn(*want.shape)
        for a, b in zip(torch.autograd.grad(got, x, dy), torch.autograd.grad(want, x, dy)):
            assert rel(a, b) <= 1e-5


def saved_through(pack, unpack, f, leaves, dy):
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        y = f()
    return torch.autograd.grad(y, leaves, dy.to(y.dtype))


def hooked_cases(dev):
    """(function, leaves, gradient of the result): the scan, a block and its layers."""
    import selective_nd_scan as snd
    torch.manual_seed(17)
    rn = lambda *s: torch.randn(*s, device=dev)
    u, w, B, A = rn(1, 2, 9, 10).requires_grad_(), rn(4, 2).requires_grad_(), rn(1, 4, 6, 9, 10).requires_grad_(), -torch.rand(8, 6, device=dev) - 0.1
    delta = rn(1, 8, 9, 10)
    yield lambda: snd.cross_scan_2d(u, delta, A, B, B, None, None, True, w), [u, w, B], rn(1, 2, 9, 10)
    op = block(dev).op
    op.in_proj, op.out_proj = nn.Identity(), nn.Identity()
    x = rn(1, 9, 10, 96).requires_grad_()
    yield lambda: op(x), [x] + list(op.parameters()), rn(1, 9, 10, 48)
    t = rn(30, 24).requires_grad_()
    norm, lin = snd.vss_block.TokenNorm(24).to(dev), snd.vss_block.TokenLinear(24, 8).to(dev, torch.bfloat16)
    yield lambda: norm(t), [t] + list(norm.parameters()), rn(30, 24)
    yield lambda: lin(t.bfloat16()), [t] + list(lin.parameters()), rn(30, 8)


def test_saved_tensor_hooks(gpu_device):
    """Tensors saved to the host and brought back give the same gradients; other tensors than were saved are refused."""
    for f, leaves, dy in hooked_cases(gpu_device):
        want = torch.autograd.grad(f(), leaves, dy.to(f().dtype))
        for a, b in zip(saved_through(lambda t: t.cpu(), lambda t: t.to(gpu_device), f, leaves, dy), want):
            assert rel(a, b) <= 1e-5
        for other in (lambda t: t.cpu(), lambda t: t.double(), lambda t: t.flatten()[: max(1, t.numel() // 2)]):
            with pytest.raises((RuntimeError, IndexError)):
                saved_through(lambda t: t, other, f, leaves, dy)


@pytest.mark.parametrize("transform", [lambda f, u: torch.func.grad(lambda v: f(v).sum())(u), lambda f, u: torch.func.vmap(f)(u[None]),
                                       lambda f, u: torch.func.jvp(f, (u,), (torch.ones_like(u),))])
def test_function_transforms_of_the_scan_are_refused(gpu_device, transform):
    import selective_nd_scan as snd
    u, B = torch.randn(1, 8, 6, 6, device=gpu_device), torch.randn(1, 4, 2, 6, 6, device=gpu_device)
    A = -torch.ones(8, 2, device=gpu_device)
    with pytest.raises(RuntimeError):
        transform(lambda v: snd.selective_nd_scan(v, u, A, B, B), u)
