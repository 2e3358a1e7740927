"""A VSS-style block around the four-corner 2D selective scan: the caller that produces the op's
inputs in a 2D-CrossScan backbone.

The reference repository ships only the kernel (README.md:62-69 points at VMamba / SparseFormer for
the models "with minor modifications such as replacing the backbone and kernel"); this module
follows the upstream VMamba SS2D layout of that caller so the op can be dropped into such a block:

    x [B, H, W, C] -> in_proj -> (x, z) -> depthwise 3x3 conv + SiLU
      -> per direction k: x_proj_k -> (dt_k, B_k, C_k), dt_proj_k -> delta_k          (1x1 maps)
      -> four-corner scan (direction k = scan origin corner k, kernel option directions=1)
      -> fuse the four results with trainable weights (README.md:45) -> LayerNorm -> * SiLU(z) -> out_proj

Because the scan origins are handled inside the kernels, every tensor stays in its natural
orientation: the projections are pointwise, so no flipped (or even repeated) copy of the feature
map is ever built - the four direction groups read the same u.
On the GPU everything between the two outer linear layers runs in the extension (snd_block.hip: convolution + SiLU, the
step-size projection, output norm + gate, weight gradients; the wide products are library GEMMs), forward and backward.
Elsewhere, with another `scan_fn`, where a stage was replaced, overridden or hooked, and under tracing, function transforms,
dispatch modes, deterministic algorithms and with tensor subclasses, it is plain PyTorch.
"""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from .cross_scan import cross_merge, cross_scan_2d
from .interface import ext

_FLOATS = (torch.float32, torch.bfloat16, torch.float16)


def _autocast_like(x):
    """An empty tensor of the type a layer would compute in: autocast's, or x's own."""
    return x.new_empty(0, dtype=torch.get_autocast_dtype("cuda")) if torch.is_autocast_enabled("cuda") else x


def _plain(*tensors):
    """Whether kernels of the extension may stand in for torch layers on these tensors (None: not given)."""
    return (not torch.compiler.is_compiling() and all(t is None or type(t) in (torch.Tensor, nn.Parameter) for t in tensors)
            and ext().plain(tensors))


def _layer_types(like, *params):
    """Whether a torch layer would take these parameters: any floating type under autocast, else that of what it reads."""
    ok = _FLOATS if torch.is_autocast_enabled("cuda") else (like,)
    return all(p is None or p.dtype in ok for p in params)


def _bare(module, cls):
    """Whether calling `module` is cls.forward and nothing else: no subclass, replaced forward or hook that a kernel in its place would pass by."""
    return (type(module) is cls and "forward" not in module.__dict__
            and not (module._forward_pre_hooks or module._forward_hooks or module._backward_pre_hooks or module._backward_hooks)
            and not torch.nn.modules.module._has_any_global_hook())


class TokenNorm(nn.LayerNorm):
    """LayerNorm.  narrow: under autocast on the GPU its result has autocast's type instead of float32, for a reader that casts it to that."""

    def forward(self, x, narrow=False):
        if not (x.is_cuda and x.dtype in _FLOATS and self.normalized_shape == tuple(x.shape[-1:]) and x.shape[-1] <= 1024 and x.numel() > 0
                and self.bias is not None and _layer_types(x.dtype, self.weight, self.bias) and _plain(x, self.weight, self.bias)):
            return super().forward(x)
        like = _autocast_like(x) if narrow else x.new_empty(0, dtype=torch.float32) if torch.is_autocast_enabled("cuda") else x
        return ext().block_norm(x, self.weight, self.bias, self.eps, like)


def _normed(norm, x, *readers):
    """norm(x); narrow if the modules that take its result on its way, `readers`, are the constructor's and end in a linear layer."""
    if torch.is_autocast_enabled("cuda") and _bare(norm, TokenNorm) and all(_bare(m, cls) for m, cls in readers):
        return norm(x, True)
    return norm(x)


class TokenLinear(nn.Linear):
    """Linear layer whose weight gradient, in a 16-bit type on the GPU, is split over the tokens."""

    def forward(self, x):
        if not (x.is_cuda and x.dtype in _FLOATS and x.numel() > 0 and torch.is_grad_enabled() and _layer_types(x.dtype, self.weight, self.bias)
                and _plain(x, self.weight, self.bias)):
            return super().forward(x)
        like = _autocast_like(x)
        if like.dtype not in _FLOATS[1:]:
            return super().forward(x)
        return ext().block_linear(x, self.weight, self.bias, like)


class SS2DCrossScan(nn.Module):
    K = 4  # scan origins: the four corners

    def __init__(self, d_model, d_state=16, ssm_ratio=2.0, dt_rank="auto", d_conv=3, conv_bias=True, bias=False,
                 dt_min=1e-3, dt_max=1e-1, dt_init_floor=1e-4, merge="weighted", scan_fn=None):
        super().__init__()
        self.d_model, self.d_state = d_model, d_state
        self.d_inner = int(ssm_ratio * d_model)
        self.dt_rank = math.ceil(d_model / 16) if dt_rank == "auto" else dt_rank
        self.scan_fn = scan_fn          # None: the scan with the merge fused into it
        K, Di, N, R = self.K, self.d_inner, d_state, self.dt_rank

        self.in_proj = TokenLinear(d_model, 2 * Di, bias=bias)
        self.conv2d = nn.Conv2d(Di, Di, d_conv, padding=(d_conv - 1) // 2, groups=Di, bias=conv_bias)
        # per-direction projections, stacked on a leading K axis
        self.x_proj_weight = nn.Parameter(torch.empty(K, R + 2 * N, Di))
        nn.init.kaiming_uniform_(self.x_proj_weight.view(-1, Di), a=math.sqrt(5))
        self.dt_projs_weight = nn.Parameter(torch.empty(K, Di, R).uniform_(-R ** -0.5, R ** -0.5))
        dt = torch.exp(torch.rand(K, Di) * (math.log(dt_max) - math.log(dt_min)) + math.log(dt_min)).clamp(min=dt_init_floor)
        self.dt_projs_bias = nn.Parameter(dt + torch.log(-torch.expm1(-dt)))        # softplus^-1(dt)
        self.A_logs = nn.Parameter(torch.log(torch.arange(1, N + 1, dtype=torch.float32)).repeat(K * Di, 1))
        self.Ds = nn.Parameter(torch.ones(K * Di))
        self.merge_weights = nn.Parameter(torch.ones(K, Di)) if merge == "weighted" else None
        self.out_norm = nn.LayerNorm(Di)
        self.out_proj = TokenLinear(Di, d_model, bias=bias)

    def scan_inputs(self, x):
        """x [B, Di, H, W] (after conv + activation) -> (u, delta, A, B, C, D, delta_bias) of the op."""
        Bt, Di, H, W = x.shape
        K, N, R = self.K, self.d_state, self.dt_rank
        x_dbl = torch.einsum("bdhw,kcd->bkchw", x, self.x_proj_weight.to(x.dtype))
        dts, Bs, Cs = torch.split(x_dbl, [R, N, N], dim=2)
        delta = torch.einsum("bkrhw,kdr->bkdhw", dts, self.dt_projs_weight.to(x.dtype)).reshape(Bt, K * Di, H, W)
        A = -torch.exp(self.A_logs.float())
        return (x, delta.contiguous(), A, Bs.contiguous(), Cs.contiguous(), self.Ds.float(),
                self.dt_projs_bias.float().reshape(-1))

    def _fused(self, xz):
        """Whether the extension may stand in for what follows in forward(): every stage is still the one the constructor made."""
        conv, norm, Di = self.conv2d, self.out_norm, self.d_inner
        return (self.scan_fn is None and not torch.compiler.is_compiling()
                and not torch.are_deterministic_algorithms_enabled()                 # (its parameter gradients are added up with atomics)
                and getattr(self.scan_inputs, "__func__", None) is SS2DCrossScan.scan_inputs
                and _bare(conv, nn.Conv2d) and _bare(norm, nn.LayerNorm)
                and (conv.kernel_size, conv.stride, conv.padding, conv.dilation, conv.padding_mode) == ((3, 3), (1, 1), (1, 1), (1, 1), "zeros")
                and conv.in_channels == conv.out_channels == conv.groups == Di
                and self.dt_projs_bias.shape == (self.K, Di) and norm.normalized_shape == (Di,) and norm.weight is not None and norm.bias is not None
                and xz.is_cuda and xz.dtype in _FLOATS and xz.numel() > 0 and self.dt_rank <= 64 and self.d_state <= 16
                and xz.shape[0] * self.K < 65536     # (image, direction) pairs: rows of a grid
                and _layer_types(xz.dtype, conv.weight, conv.bias) and _layer_types(torch.float32, norm.weight, norm.bias)
                and _plain(xz, conv.weight, conv.bias, self.x_proj_weight, self.dt_projs_weight, self.dt_projs_bias, self.A_logs, self.Ds,
                           self.merge_weights, norm.weight, norm.bias))

    def forward(self, x):
        """x [B, H, W, d_model] -> [B, H, W, d_model]."""
        xz = self.in_proj(x)
        if self._fused(xz):
            return self.out_proj(ext().ss2d(xz, self.conv2d.weight, self.conv2d.bias, self.x_proj_weight, self.dt_projs_weight, self.dt_projs_bias,
                                            self.A_logs, self.Ds, self.merge_weights, self.out_norm.weight, self.out_norm.bias, self.out_norm.eps))
        x, z = xz.chunk(2, dim=-1)
        x = F.silu(self.conv2d(x.permute(0, 3, 1, 2).contiguous()))
        u, delta, A, Bs, Cs, Ds, dt_bias = self.scan_inputs(x)
        if self.scan_fn is None:                                                      # [B, Di, H, W] fp32
            y = cross_scan_2d(u, delta, A, Bs, Cs, Ds, dt_bias, True, self.merge_weights)
        else:
            ys = self.scan_fn(u, delta, A, Bs, Cs, Ds, dt_bias, True, True)          # [B, K*Di, H, W] fp32
            y = cross_merge(ys, self.merge_weights)
        y = self.out_norm(y.permute(0, 2, 3, 1)).to(z.dtype)
        return self.out_proj(y * F.silu(z))


class VSSBlock(nn.Module):
    """Pre-norm residual block: x + SS2D(LN(x)), then x + MLP(LN(x)) when mlp_ratio > 0."""

    def __init__(self, d_model, d_state=16, ssm_ratio=2.0, mlp_ratio=4.0, **ss2d_kwargs):
        super().__init__()
        self.norm = TokenNorm(d_model)
        self.op = SS2DCrossScan(d_model, d_state=d_state, ssm_ratio=ssm_ratio, **ss2d_kwargs)
        self.mlp = None
        if mlp_ratio > 0:
            hidden = int(mlp_ratio * d_model)
            self.norm2 = TokenNorm(d_model)
            self.mlp = nn.Sequential(TokenLinear(d_model, hidden), nn.GELU(), TokenLinear(hidden, d_model))

    def forward(self, x):
        op, mlp = self.op, self.mlp
        x = x + op(_normed(self.norm, x, (op, SS2DCrossScan), (getattr(op, "in_proj", None), TokenLinear)))
        if mlp is not None:
            first = mlp[0] if type(mlp) is nn.Sequential and len(mlp) > 0 else None
            x = x + mlp(_normed(self.norm2, x, (mlp, nn.Sequential), (first, TokenLinear)))
        return x
