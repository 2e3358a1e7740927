"""The block's layers on tensors that have no memory of their own: the torch layers they stand for run."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("grad", [False, True])
def test_fake_tensors(dtype, grad):
    from selective_nd_scan.vss_block import TokenLinear, TokenNorm
    with FakeTensorMode(), torch.set_grad_enabled(grad):
        x = torch.empty(3, 5, 8, device="cuda", dtype=dtype)
        y = TokenNorm(8, device="cuda", dtype=dtype)(x)
        assert y.shape == x.shape and y.dtype == dtype
        y = TokenLinear(8, 6, device="cuda", dtype=dtype)(x)
        assert y.shape == (3, 5, 6) and y.dtype == dtype
