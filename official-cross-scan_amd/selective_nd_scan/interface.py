"""Python face of the 2D-CrossScan selective scan on MI355X.

The reference ships only the pybind pair `fwd` / `bwd`
(kernels/selective_nd_scan/src/cusoflex/selective_scan_oflex.cpp:442-445); the Python function that
backbones call is authored here, on a native autograd function over the same pair, with the argument
order of those bindings (selective_scan_oflex.cpp:179-187).

    out = selective_nd_scan(u, delta, A, B, C, D=None, delta_bias=None,
                            delta_softplus=False, out_float=True, A_decay=None)

    u      [B, D, H, W]        fp32 / fp16 / bf16   (or [B, D/G, H, W]: one map shared by the G groups)
    delta  [B, Dd, H, W]       same dtype, D % Dd == 0
    A      [D, N]              fp32, N <= 16
    B, C   [B, G, N, H, W]     same dtype as u, D % G == 0
    D      [D] fp32, delta_bias [Dd] fp32, A_decay [1] fp32 (all optional)
    out    [B, D, H, W]        fp32 if out_float else u.dtype

With directions=0 every group is scanned from the top-left corner, as the reference kernel does
(selective_scan_fwd_kernel_oflex.cuh:140).  directions=1 starts group g at corner g % 4 inside the
kernels (no flipped copies); cross_scan.py builds the four-corner block on top of it.
"""
import torch

from ._ext import ext


class _TracedScan(torch.autograd.Function):
    """The scan as one operation of a graph that jit.trace records; a call into the extension alone would leave no more of itself
    there than the allocation of its result."""

    @staticmethod
    def forward(ctx, *args):
        ctx.args = [a.detach().requires_grad_(a.requires_grad) if isinstance(a, torch.Tensor) else a for a in args]
        with torch.enable_grad():
            ctx.out = ext().scan(*ctx.args)
        return ctx.out.detach()

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dout):
        leaves = [a for a in ctx.args if isinstance(a, torch.Tensor) and a.requires_grad]
        grads = iter(torch.autograd.grad(ctx.out, leaves, dout, retain_graph=True, allow_unused=True))
        return tuple(next(grads) if isinstance(a, torch.Tensor) and a.requires_grad else None for a in ctx.args)


def _scan(*args):
    return _TracedScan.apply(*args) if torch.jit.is_tracing() else ext().scan(*args)


def fwd(u, delta, A, B, C, D=None, delta_bias=None, delta_softplus=False, out_float=True, A_decay=None,
        directions=0, schedule=-1, merge=False, merge_weights=None):
    """Reference binding `fwd` -> [out, x, x_v, x_sd] (selective_scan_oflex.cpp:179-187,282).
    schedule: block mapping of this call (-1 = the module default, see set_schedule).
    merge: the CrossMerge fused into the output stores: out is [B, D/G, H, W] fp32, the sum over the G
    groups of merge_weights[channel] * (result of the channel) (merge_weights [D] fp32, None = ones)."""
    return ext().fwd(u, delta, A, B, C, D, delta_bias, delta_softplus, out_float, A_decay, directions, schedule,
                     merge, merge_weights)


def bwd(u, delta, A, B, C, D, delta_bias, dout, x, x_v, delta_softplus, A_decay, x_sd, directions=0, schedule=-1,
        merge=False, merge_weights=None):
    """Reference binding `bwd` -> [du, ddelta, dA, dB, dC, dD, ddelta_bias, dA_decay]
    (selective_scan_oflex.cpp:286-297,432-438).  With merge, dout is the gradient of the merged output
    [B, D/G, H, W] and a ninth tensor follows: merge_weights * d merge_weights, per channel [D]."""
    return ext().bwd(u, delta, A, B, C, D, delta_bias, dout, x, x_v, delta_softplus, A_decay, x_sd, directions,
                     schedule, merge, merge_weights)


def set_schedule(mode):
    """Default block mapping of calls that name none: 0 = chosen by shape, 1 = one block per (batch,
    group, 16-channel chunk) plane, 2 = one block per 8-row strip, strips pipelined, 3 = bands of strips,
    4 = the row-segment wavefront kernels (1-4 states).
    Results do not depend on it (only the order of the atomic sums in dA, dB, dC, dD, ddelta_bias does), but a
    bwd must run the kernel family of the fwd whose saved state it is given (modes 1-3 are one family, 4 the other,
    0 picks by shape): the autograd functions see to that themselves; a bwd on another family's state returns NaN
    gradients, never plausible numbers."""
    ext().set_schedule(int(mode))


def get_schedule():
    """The default block mapping (see set_schedule)."""
    return int(ext().get_schedule())


def set_debug(on=True):
    """After every pipelined launch, read the workspace's error word (one stream sync per call) and raise
    if a block-to-block wait timed out.  Also switched on by SND_CHECK_PIPELINE=1 in the environment."""
    ext().set_debug(bool(on))


def init(device=0):
    """Per-device set-up (kernel attributes).  Optional; call it once before capturing launches into a
    HIP graph or launching from several threads."""
    ext().init(int(device))


class SelectiveNdScanFn:
    """selective_nd_scan under the name and call form of an autograd.Function (the function itself, forward and
    backward, is native code in the extension)."""

    @staticmethod
    def apply(u, delta, A, B, C, D=None, delta_bias=None, delta_softplus=False, out_float=True, A_decay=None,
              directions=0):
        return _scan(u, delta, A, B, C, D, delta_bias, delta_softplus, out_float, A_decay, directions, False, None)


def selective_nd_scan(u, delta, A, B, C, D=None, delta_bias=None, delta_softplus=False, out_float=True,
                      A_decay=None, directions=0):
    """Differentiable 2D-CrossScan selective scan (forward and backward run on the HIP kernels).
    directions=1: group g of B/C (and its dim/G channels) is scanned from corner g % 4.
    Where no gradient can be asked for (no_grad, or no input that requires one) the forward saves no state."""
    return _scan(u, delta, A, B, C, D, delta_bias, delta_softplus, out_float, A_decay, directions, False, None)


class SelectiveNdScanMergedFn:
    """The scan with the CrossMerge fused into its output stores: out [B, D/G, H, W] fp32 is the sum over the
    G groups of merge_weights[g, i] * (result of channel g*(D/G) + i)."""

    @staticmethod
    def apply(u, delta, A, B, C, D, delta_bias, delta_softplus, A_decay, directions, merge_weights):
        return _scan(u, delta, A, B, C, D, delta_bias, delta_softplus, True, A_decay, directions, True, merge_weights)


def selective_nd_scan_merged(u, delta, A, B, C, D=None, delta_bias=None, delta_softplus=False, A_decay=None,
                             directions=1, merge_weights=None):
    """selective_nd_scan followed by the merge of the G group results of every feature, in one kernel call:
    returns [B, D/G, H, W] fp32 = sum_g merge_weights[g, i] * out[:, g*(D/G) + i].  merge_weights: None (plain
    sum), [G], [G, 1] or [G, D/G]; differentiable.  The four corners of planes of up to 64 columns are added up inside a
    block with 1-4 states, where their sums fit in its LDS; everywhere else the sum is accumulated with float atomics.
    In either case its last bits depend on the order the groups arrive in."""
    if merge_weights is not None:
        G = B.shape[1]
        if merge_weights.dim() == 1:
            if merge_weights.numel() != G:
                raise ValueError("merge_weights must have shape [G], [G, 1] or [G, D/G]")
        elif tuple(merge_weights.shape) not in ((G, 1), (G, A.shape[0] // G)):
            raise ValueError("merge_weights must have shape [G], [G, 1] or [G, D/G]")
    return _scan(u, delta, A, B, C, D, delta_bias, delta_softplus, True, A_decay, directions, True, merge_weights)
