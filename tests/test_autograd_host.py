"""What the extension refuses before it looks at the device its tensors are on."""
import pytest
import torch
import torch.autograd.forward_ad as fwad


@pytest.mark.parametrize("name", ["u", "A", "D", "A_decay", "merge_weights"])
@pytest.mark.parametrize("grad", [False, True])
def test_forward_mode_is_refused(name, grad):
    """A dual tensor has requires_grad == False: without the check it takes the path below autograd and its tangent is lost."""
    from selective_nd_scan.interface import ext
    t = dict(u=torch.randn(1, 2, 5, 6), delta=torch.randn(1, 8, 5, 6), A=-torch.ones(8, 3), B=torch.randn(1, 4, 3, 5, 6),
             C=torch.randn(1, 4, 3, 5, 6), D=torch.ones(8), delta_bias=torch.zeros(8), A_decay=torch.ones(1), merge_weights=torch.ones(4, 2))
    if grad:
        t["delta"].requires_grad_()
    with fwad.dual_level(), pytest.raises(RuntimeError, match="forward-mode"):
        t[name] = fwad.make_dual(t[name], torch.ones_like(t[name]))
        ext().scan(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"], True, True, t["A_decay"], 1, True, t["merge_weights"])


@pytest.mark.parametrize("x,gamma,beta", [((3, 8), 4, 4), ((3, 4), 8, 8), ((3, 8), 8, 4), ((3, 8), 4, 8), ((), 1, 1)])
def test_norm_refuses_another_last_axis(x, gamma, beta):
    """gamma and beta are read along the last axis of x by raw pointer."""
    from selective_nd_scan.interface import ext
    with pytest.raises(RuntimeError, match="last axis"):
        ext().block_norm(torch.randn(x), torch.ones(gamma), torch.ones(beta), 1e-5, torch.empty(0))


@pytest.mark.parametrize("x,w,b", [((3, 8), (6, 4), (6,)), ((3, 8), (6, 8), (5,)), ((3, 8), (6, 8, 1), (6,)), ((), (1, 1), (1,))])
def test_linear_refuses_shapes_that_do_not_fit(x, w, b):
    from selective_nd_scan.interface import ext
    with pytest.raises(RuntimeError, match="do not fit"):
        ext().block_linear(torch.randn(x), torch.randn(w), torch.randn(b), torch.empty(0, dtype=torch.bfloat16))


@pytest.mark.parametrize("name,shape", [("conv_w", (6, 1, 1, 9)), ("conv_b", (5,)), ("wx", (4, 7, 6)), ("wx", (4, 8, 5)), ("wdt", (4, 6, 3)), ("wdt", (3, 6, 2)),
                                        ("dt_bias", (4, 5)), ("A_logs", (23, 3)), ("A_logs", (24, 3, 1)), ("D", (6,)), ("mw", (4, 5)), ("mw", (24,)), ("mw", (6, 4)), ("gamma", (5,)), ("beta", (7,))])
def test_ss2d_refuses_shapes_that_do_not_fit(name, shape):
    from selective_nd_scan.interface import ext
    t = dict(xz=(1, 5, 5, 12), conv_w=(6, 1, 3, 3), conv_b=(6,), wx=(4, 8, 6), wdt=(4, 6, 2), dt_bias=(4, 6), A_logs=(24, 3), D=(24,), mw=(4, 6), gamma=(6,), beta=(6,))
    with pytest.raises(RuntimeError, match="on the GPU"):
        ext().ss2d(*[torch.ones(s) for s in t.values()], 1e-5)
    t[name] = shape
    with pytest.raises(RuntimeError, match="do not fit|2-D"):
        ext().ss2d(*[torch.ones(s) for s in t.values()], 1e-5)
