"""A whole block against the same block in float64 on the host, whose scan is the torch restatement of the reference recurrence:
nothing of this repository's kernels is on the other side.  And a block on a stream of its own."""
import copy

import pytest
import torch

from oracle.snd_torch_ref import selective_nd_scan_torch

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float((a.detach().double().cpu() - b.detach()).norm() / b.detach().norm().clamp_min(1e-30))


def reference_scan(u, delta, A, B, C, D, delta_bias, delta_softplus, out_float):
    from selective_nd_scan.cross_scan import flip_groups
    G = B.shape[1]
    out = selective_nd_scan_torch(flip_groups(u.repeat(1, G, 1, 1), G), flip_groups(delta, G), A.double(), flip_groups(B, G), flip_groups(C, G), D.double(),
                                  delta_bias.double(), delta_softplus)
    return flip_groups(out, G)


def make(dev, width, states, kw):
    import selective_nd_scan as snd
    torch.manual_seed(19)
    blk = snd.VSSBlock(width, d_state=states, **kw).to(dev)
    for p in blk.parameters():
        p.data.add_(0.02 * torch.randn_like(p))
    return blk


@pytest.mark.parametrize("width,states,shape,dtype,kw", [
    (8, 1, (2, 9, 7), None, dict(mlp_ratio=2.0)),
    (24, 3, (1, 5, 13), None, dict(ssm_ratio=1.0, merge="sum", conv_bias=False, mlp_ratio=0.0)),
    (33, 16, (1, 7, 6), None, dict(ssm_ratio=1.0, mlp_ratio=1.0, dt_rank=9, bias=True)),
    (16, 6, (3, 4, 5), None, dict(mlp_ratio=2.0)),
    (16, 16, (1, 7, 8), torch.bfloat16, dict(mlp_ratio=2.0)),
    (24, 2, (2, 6, 7), torch.float16, dict(mlp_ratio=2.0)),
])
def test_block_against_the_restatement(gpu_device, width, states, shape, dtype, kw):
    blk = make(gpu_device, width, states, kw)
    ref = copy.deepcopy(blk).double().cpu()
    ref.op.scan_fn = reference_scan
    x, dy = (torch.randn(*shape, width, dtype=torch.float64) for _ in range(2))
    xs = [x.float().to(gpu_device).requires_grad_(), x.float().double().requires_grad_()]
    with torch.autocast("cuda", dtype=dtype or torch.bfloat16, enabled=dtype is not None):
        y = blk(xs[0])
    want = ref(xs[1])
    y.backward(dy.float().to(gpu_device))
    want.backward(dy.float().double())
    # fp32: sums of a few hundred terms, each a few times 2^-24 off.  16 bits: activations are rounded about ten times on the
    # way to a gradient, each time by up to 2^-9 (bf16) or 2^-12 (fp16) of their size.
    tol = 2e-6 if dtype is None else 3e-2 if dtype == torch.bfloat16 else 4e-3
    for (name, p), q in zip([("y", y), ("x", xs[0].grad)] + [(n, p.grad) for n, p in blk.named_parameters()],
                            [want, xs[1].grad] + [q.grad for q in ref.parameters()]):
        assert rel(p, q) <= tol, (name, rel(p, q))


def test_block_on_a_stream_of_its_own(gpu_device):
    """Forward and backward on a side stream, with other work queued on the default stream before and after."""
    blk = make(gpu_device, 24, 3, dict(mlp_ratio=2.0))
    x, dy = torch.randn(2, 20, 20, 24, device=gpu_device), torch.randn(2, 20, 20, 24, device=gpu_device)

    def run():
        xi = x.clone().requires_grad_()
        y = blk(xi)
        return [y.detach(), *torch.autograd.grad(y, [xi] + list(blk.parameters()), dy)]

    want = run()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    junk = torch.randn(4096, 4096, device=gpu_device)
    for _ in range(3):
        junk = junk @ junk * 1e-3                      # the default stream is busy
    with torch.cuda.stream(side):
        got = run()
        for t in got:
            t.record_stream(torch.cuda.current_stream())
    side.synchronize()
    for a, b in zip(got, want):
        assert rel(a, b.double().cpu()) <= 1e-5


@pytest.mark.parametrize("train", [False, True])
def test_block_in_a_graph(gpu_device, train):
    """A block's step captured once: every replay, with eager work in between, gives what the eager step gives on its inputs."""
    blk = make(gpu_device, 24, 3, dict(mlp_ratio=2.0))
    x, dy = torch.randn(2, 12, 11, 24, device=gpu_device), torch.randn(2, 12, 11, 24, device=gpu_device)
    xs = x.clone().requires_grad_(train)

    def step():
        with torch.set_grad_enabled(train):
            y = blk(xs)
        return [y.detach(), *(torch.autograd.grad(y, [xs] + list(blk.parameters()), dy) if train else [])]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        got = step()
    for k in range(4):
        with torch.no_grad():
            xs.copy_(x * (1 + k))
        want = [t.double().cpu() for t in step()]
        for t in got:
            t.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert rel(a, b) <= 1e-5, k
