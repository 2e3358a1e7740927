"""The block's own passes around its scan against the same block built from torch layers (the path every other device and
every replaced scan_fn takes)."""
import copy

import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30))


def plain(blk):
    import selective_nd_scan as snd
    ref = copy.deepcopy(blk)
    ref.op.scan_fn = lambda *a: snd.four_corner_scan(*a)
    for owner in [m for m in ref.modules()]:
        for name, m in list(owner.named_children()):
            if type(m) in (snd.vss_block.TokenNorm, snd.vss_block.TokenLinear):
                m.__class__ = nn.LayerNorm if isinstance(m, nn.LayerNorm) else nn.Linear
    return ref


@pytest.mark.parametrize("width,states,ratio,mlp,shape,dtype,kw", [
    (16, 1, 1.0, 2.0, (2, 1, 1), torch.float32, {}),                                   # one pixel: everything is halo
    (24, 5, 2.0, 0.0, (3, 9, 33), torch.float32, dict(merge="sum")),                   # one column into a second tile, odd pixel count
    (40, 16, 2.0, 2.0, (1, 13, 64), torch.float32, dict(conv_bias=False)),             # 80 channels: 2.5 tiles of 32
    (33, 2, 1.0, 1.0, (2, 5, 31), torch.float32, dict(dt_rank=9, bias=True)),          # odd width, rank 9 of 16
    (96, 16, 2.0, 4.0, (2, 28, 28), torch.bfloat16, {}),
    (66, 3, 2.0, 2.0, (1, 17, 18), torch.float16, dict(dt_rank=40)),
    (512, 4, 2.0, 1.0, (1, 7, 7), torch.bfloat16, {}),                                 # 1024 inner channels
])
def test_block_passes(gpu_device, width, states, ratio, mlp, shape, dtype, kw):
    import selective_nd_scan as snd
    torch.manual_seed(5)
    blk = snd.VSSBlock(width, d_state=states, ssm_ratio=ratio, mlp_ratio=mlp, **kw).to(gpu_device)
    for p in blk.parameters():
        p.data.add_(0.02 * torch.randn_like(p))
    ref = plain(blk)
    x = torch.randn(*shape, width, device=gpu_device)
    g = torch.randn_like(x)
    half = dtype != torch.float32

    def run(m):
        xi = x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=dtype if half else torch.bfloat16, enabled=half):
            y = m(xi)
        y.backward(g)
        return [y.detach(), xi.grad] + [p.grad for p in m.parameters()]

    names = ["y", "x"] + [n for n, _ in blk.named_parameters()]
    for name, a, b in zip(names, run(blk), run(ref)):
        assert a.dtype == b.dtype and a.shape == b.shape
        # (one pixel: the gradient through a LayerNorm of few channels cancels to rounding)
        assert rel(a, b) <= (1e-2 if half else 1e-3 if shape[1:] == (1, 1) else 2e-5), (name, rel(a, b))
    with torch.no_grad(), torch.autocast("cuda", dtype=dtype if half else torch.bfloat16, enabled=half):
        assert rel(blk(x), ref(x)) <= (1e-2 if half else 2e-5)


@pytest.mark.parametrize("tokens,M,N", [(1, 2, 2), (63, 66, 34), (257, 64, 130), (5000, 192, 96)])
def test_linear_weight_gradient(gpu_device, tokens, M, N):
    from selective_nd_scan.interface import ext
    torch.manual_seed(6)
    x = torch.randn(tokens, N, device=gpu_device, dtype=torch.bfloat16)
    w = torch.randn(M, N, device=gpu_device).requires_grad_()
    b = torch.randn(M, device=gpu_device).requires_grad_()
    dy = torch.randn(tokens, M, device=gpu_device, dtype=torch.bfloat16)
    dw, db = torch.autograd.grad(ext().block_linear(x, w, b, x), (w, b), dy)
    assert rel(dw, dy.double().t() @ x.double()) <= 1e-5 and rel(db, dy.double().sum(0)) <= 1e-5


# How a weight gradient is cut: fewer than eight splits of the tokens, eight with one token in the last, ten (a round of eight and two),
# one stage and a bit, many tiles, 34 taken as 32, 21 because of the tiles.  A result is a sum in fp32 of up to 8449 exact products: about
# sqrt(8449) * 2^-24 = 5.5e-6 of its size.
@pytest.mark.parametrize("tokens,M,N", [(1700, 64, 64), (1793, 64, 64), (2560, 130, 66), (65, 64, 64), (300, 1024, 512), (8449, 66, 130), (5400, 768, 192)])
def test_linear_weight_gradient_splits(gpu_device, tokens, M, N):
    from selective_nd_scan.interface import ext
    torch.manual_seed(8)
    x = torch.randn(tokens, N, device=gpu_device, dtype=torch.bfloat16)
    dy = torch.randn(tokens, M, device=gpu_device, dtype=torch.bfloat16)
    w = torch.randn(M, N, device=gpu_device).requires_grad_()
    b = torch.randn(M, device=gpu_device).requires_grad_()
    dw, db = torch.autograd.grad(ext().block_linear(x, w, b, x), (w, b), dy)
    assert rel(dw, dy.double().t() @ x.double()) <= 1e-5 and rel(db, dy.double().sum(0)) <= 1e-5


@pytest.mark.parametrize("C,dtype", [(1, torch.float32), (65, torch.float32), (200, torch.bfloat16), (1024, torch.float32)])
def test_token_norm(gpu_device, C, dtype):
    from selective_nd_scan.interface import ext
    torch.manual_seed(7)
    x = (torch.randn(33, C, device=gpu_device) + 3).to(dtype).requires_grad_()
    g, b = (torch.randn(C, device=gpu_device).requires_grad_() for _ in range(2))
    dy = torch.randn(33, C, device=gpu_device).to(dtype)
    got = ext().block_norm(x, g, b, 1e-5, x)
    r = [t.detach().double().requires_grad_() for t in (x, g, b)]
    want = nn.functional.layer_norm(r[0], (C,), r[1], r[2], 1e-5)
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    assert rel(got, want) <= tol
    for name, a, w in zip("xgb", torch.autograd.grad(got, (x, g, b), dy), torch.autograd.grad(want, r, dy.double())):
        assert (C == 1 and name == "x") or rel(a, w) <= tol or float(w.norm()) < 1e-6, name
