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
