"""The functions that the block's passes compute by themselves, one value at a time against float64."""
import ctypes as C

import pytest
import torch

import capi

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -23


class BlockShape(C.Structure):
    _fields_ = [(n, C.c_int32) for n in ("batch", "nrows", "ncols", "inner", "n_groups", "dstate", "rank", "dtype")]


def call(name, *args):
    f = getattr(capi.lib(), name)
    f.argtypes = [C.c_void_p if isinstance(a, torch.Tensor) or a is None else C.c_float if isinstance(a, float) else C.c_int if isinstance(a, int)
                  else C.POINTER(BlockShape) for a in args] + [C.c_void_p]
    capi.check(f(*[a.data_ptr() if isinstance(a, torch.Tensor) else C.byref(a) if isinstance(a, BlockShape) else a for a in args],
                 torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()


def test_decay_rates(gpu_device):
    """A = -exp(A_logs): two units in the last place over the whole range, which every step of the recurrence multiplies by."""
    logs = torch.linspace(-80, 80, 4001, device=gpu_device)
    A, w = torch.empty_like(logs), torch.empty(1, device=gpu_device)
    call("snd_block_params", logs, logs.numel(), torch.ones(1, device=gpu_device), 1, 1, capi.SND_F32, A, w, None)
    want = -logs.double().exp()
    assert float(((A.double() - want) / want).abs().max()) <= 2 * EPS


def test_gate(gpu_device):
    """out = silu(z) where gamma = 0 and beta = 1: exp, one sum and one quotient, three units in the last place."""
    z = torch.linspace(-60, 60, 64 * 32, device=gpu_device).view(64, 32)
    xz = torch.cat([torch.zeros_like(z), z], 1).contiguous()                   # [pixels, 2 * inner]
    y, out = torch.randn(32, 64, device=gpu_device), torch.empty_like(z)
    call("snd_block_gate_fwd", BlockShape(1, 8, 8, 32, 4, 1, 1, capi.SND_F32), y, xz, torch.zeros(32, device=gpu_device), torch.ones(32, device=gpu_device), 1e-5,
         out, None)
    want = z.double() * torch.sigmoid(z.double())
    assert float(((out.double() - want) / want).abs().max()) <= 3 * EPS


def test_convolution_gradient(gpu_device):
    """dx = silu'(pre) where the kernel is one at its centre: s (1 + x (1 - s)).  s and 1 - s are each a rounding or two of 1 off
    where s is close to 1, and x multiplies the latter."""
    pre = torch.linspace(-60, 60, 32 * 64, device=gpu_device).view(32, 64)     # [inner, pixels]
    w = torch.zeros(32, 9, device=gpu_device)
    w[:, 4] = 1
    dxz, dw = torch.zeros(64, 64, device=gpu_device), torch.zeros(32, 9, device=gpu_device)
    call("snd_block_conv_bwd", BlockShape(1, 8, 8, 32, 4, 1, 1, capi.SND_F32), torch.ones_like(pre), pre, torch.zeros(64, 64, device=gpu_device), w, dxz, dw, None)
    x = pre.double()
    s = torch.sigmoid(x)
    err = (dxz[:, :32].t().double() - s * (1 + x * (1 - s))).abs()
    assert float((err / (s * (1 + x.abs()))).max()) <= 4 * EPS
