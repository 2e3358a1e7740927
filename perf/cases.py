"""The work whose speed counts for a user of this framework: the 2D-CrossScan selective scan through its Python entry
points, as a backbone calls it in training and in inference.

A case is a dict of plain values:

    entry      "scan"     selective_nd_scan: every group from the top-left corner
               "corners"  four_corner_scan: group g from corner g % 4, one u per direction
               "merged"   cross_scan_2d: one feature map, four corners, results merged with trainable weights
               "block"    VSSBlock: projections, depthwise convolution, the four-corner scan, gate, MLP
    mode       "train": forward and backward through autograd, every gradient taken; "infer": forward under no_grad
    batch, dim, rows, cols, states, groups    the op's B, D (channels over all groups), H, W, N, K
               (a block: dim is its model width, the scan inside has 4 * ratio * dim channels)
    dtype      of u, delta, B, C ("block": the autocast type)
    out_float  whether out is float32 (the default) or of the inputs' type
    decay      whether A_decay is given
    share      channels that share one delta channel (1: each its own)
"""
import math
import os
import random
import sys

import torch

# the package of the tree that this runs in (its folder's name is no Python identifier)
_PKG = os.path.join(os.getcwd(), "official-cross-scan_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import selective_nd_scan as snd  # noqa: E402


def _case(name, entry, mode, batch, dim, rows, cols, states, dtype, groups=4, out_float=True, decay=False, share=1):
    return dict(name=name, entry=entry, mode=mode, batch=batch, dim=dim, rows=rows, cols=cols, states=states, groups=groups,
                dtype=dtype, out_float=out_float, decay=decay, share=share)


def listed():
    return [
        # one small image in inference: the benchmark's config 0; launches and host work are what it costs
        _case("tiny-infer", "scan", "infer", 1, 64, 14, 14, 16, "float32"),
        # a small batch in training (fine-tuning, a late stage at low resolution), four corners and one map
        _case("small-train", "merged", "train", 2, 384, 14, 14, 16, "bfloat16"),
        # the benchmark's headline: the first stage of a classification backbone at batch 64
        _case("stage1-train", "scan", "train", 64, 192, 56, 56, 16, "float32"),
        # the same stage served in 16 bits: forward only, out in the inputs' type
        _case("stage1-infer", "scan", "infer", 64, 192, 56, 56, 16, "bfloat16", out_float=False),
        # the third stage: small planes, many channels
        _case("stage3-train", "scan", "train", 64, 768, 14, 14, 16, "bfloat16"),
        # detection and segmentation at high resolution: few large planes, not square
        _case("detect-train", "scan", "train", 2, 192, 200, 336, 16, "float32"),
        # crops of gigapixel images: the largest planes
        _case("tile-train", "scan", "train", 1, 256, 512, 512, 16, "bfloat16"),
        # the same with one state per channel (the d_state = 1 backbones)
        _case("tile-n1-train", "scan", "train", 1, 256, 512, 512, 1, "bfloat16"),
        # a d_state = 1 backbone's first stage: one map scanned from four corners, merged with trainable weights
        _case("stage1-n1-merged", "merged", "train", 64, 384, 56, 56, 1, "bfloat16"),
        # the second stage with the merge inside the op and 16 states
        _case("stage2-merged", "merged", "train", 32, 768, 28, 28, 16, "bfloat16"),
        # sizes that divide nothing: an odd crop, 8 states, fp16, decay, delta channels shared in pairs
        _case("ragged-corners", "corners", "train", 3, 152, 61, 83, 8, "float16", decay=True, share=2),
        # a whole block of a backbone under autocast
        _case("block-train", "block", "train", 8, 96, 56, 56, 16, "bfloat16"),
    ]


# A drawn case costs no more than the largest listed one: state cells (batch * dim * rows * cols * states) and pixels
# (batch * dim * rows * cols) stay below half of "tile-train"'s, which leaves room for shapes that cost more per cell.
_MAX_CELLS, _MAX_PIXELS, _MIN_CELLS = 1 << 29, 1 << 25, 1 << 17


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    entry = rng.choice(("scan", "scan", "scan", "corners", "corners", "merged", "merged", "block"))
    mode = rng.choice(("train", "train", "infer"))
    dtype = rng.choice(("float32", "bfloat16", "float16"))
    groups = 4 if entry != "scan" else rng.choice((4, 4, 2, 1))
    share = rng.choice((1, 1, 1, 2)) if entry != "block" else 1
    states = rng.choice((1, 16, _log(rng, 1, 16)))
    while True:
        rows, batch, per_group = _log(rng, 7, 512), _log(rng, 1, 64), _log(rng, 8, 192)
        cols = min(512, max(7, int(round(rows * math.exp(rng.uniform(-0.7, 0.7))))))
        dim = 4 * per_group if entry == "block" else groups * (per_group // share * share)
        pixels = batch * dim * rows * cols * (8 if entry == "block" else 1)
        if pixels <= _MAX_PIXELS and _MIN_CELLS <= pixels * states <= _MAX_CELLS:
            break
    if entry == "block":
        return {k: v for k, v in _case("", entry, mode, batch, dim, rows, cols, states, "bfloat16").items() if k != "name"}
    case = _case("", entry, mode, batch, dim, rows, cols, states, dtype, groups,
                 out_float=entry == "merged" or rng.random() < 0.7, decay=rng.random() < 0.2, share=share)
    del case["name"]
    return case


_TYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    train = case["mode"] == "train"

    def rn(*shape):
        return torch.randn(*shape, device=dev, generator=g)

    Bt, Dm, H, W, N, K = (case[k] for k in ("batch", "dim", "rows", "cols", "states", "groups"))
    dtype = _TYPES[case["dtype"]]
    if case["entry"] == "block":
        with torch.random.fork_rng(devices=[]):
            torch.manual_seed(seed)
            block = snd.VSSBlock(Dm, d_state=N, ssm_ratio=2.0, mlp_ratio=4.0).to(dev)
        x, dy = rn(Bt, H, W, Dm), rn(Bt, H, W, Dm)
        if train:
            x.requires_grad_()
        return dict(case=case, block=block, x=x, dout=dy, leaves=[x] + list(block.parameters()) if train else [])

    merged = case["entry"] == "merged"
    Dd = Dm // case["share"]
    dt = torch.exp(torch.empty(Dd, device=dev).uniform_(math.log(1e-3), math.log(1e-1), generator=g))
    t = dict(u=rn(Bt, Dm // K if merged else Dm, H, W).to(dtype), delta=rn(Bt, Dd, H, W).mul_(0.1).to(dtype),
             A=-torch.arange(1, N + 1, device=dev, dtype=torch.float32).repeat(Dm, 1), B=rn(Bt, K, N, H, W).to(dtype),
             C=rn(Bt, K, N, H, W).to(dtype), D=torch.ones(Dm, device=dev), delta_bias=torch.log(torch.expm1(dt)),
             A_decay=torch.full((1,), 0.95, device=dev) if case["decay"] else None,
             merge_weights=1 + 0.1 * rn(K, Dm // K) if merged else None)
    leaves = []
    if train:
        leaves = [v.requires_grad_() for v in t.values() if v is not None]
    dout = rn(Bt, Dm // K if merged else Dm, H, W).to(torch.float32 if case["out_float"] else dtype) if train else None
    return dict(case=case, t=t, dout=dout, leaves=leaves)


def _forward(s):
    case = s["case"]
    if case["entry"] == "block":
        with torch.autocast("cuda", dtype=_TYPES[case["dtype"]]):
            return s["block"](s["x"])
    t = s["t"]
    args = (t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"], True)
    if case["entry"] == "merged":
        return snd.cross_scan_2d(*args, t["merge_weights"], t["A_decay"])
    scan = snd.selective_nd_scan if case["entry"] == "scan" else snd.four_corner_scan
    return scan(*args, case["out_float"], t["A_decay"])


def run(state):
    if state["case"]["mode"] == "infer":
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    return [out.detach(), *torch.autograd.grad(out, state["leaves"], state["dout"])]


def work(case):
    e = 4 if case["dtype"] == "float32" else 2
    Bt, Dm, HW, N, K = case["batch"], case["dim"], case["rows"] * case["cols"], case["states"], case["groups"]
    train = case["mode"] == "train"
    if case["entry"] == "block":
        # tokens in and out (fp32), weights read once, and their gradients; the products of the layers: in, x, dt, out
        # projections and the MLP, the depthwise convolution, and the scan over 4 * 2 * width channels
        tok, di, rank = Bt * HW, 2 * Dm, math.ceil(Dm / 16)
        weights = Dm * 2 * di + 4 * di * (rank + 2 * N) + 4 * di * rank + di * Dm + 2 * 4 * Dm * Dm + 9 * di
        cells = tok * 4 * di * N
        return {"bytes": 4 * tok * Dm * (4 if train else 2) + 4 * weights * (2 if train else 1),
                "flops": tok * weights * (6 if train else 2) + cells * (62 if train else 17)}
    pu = Bt * (Dm // K if case["entry"] == "merged" else Dm) * HW     # u, and out
    pd, q, cells = Bt * Dm // case["share"] * HW, 2 * Bt * K * N * HW, Bt * Dm * HW * N
    inputs, out = e * (pu + pd + q), (4 if case["out_float"] else e) * pu
    # per state cell: a (2), bu (1), h (7), s (2), out (5) forward; and about 45 in the reverse sweep
    return {"bytes": 2 * (inputs + out) if train else inputs + out, "flops": cells * (62 if train else 17)}


def tolerance(case):
    # float32: sums of a few thousand to a few million terms, accumulated in an order that is not fixed; 16-bit types:
    # the rounding of the gradients (the block: of every layer's activations as well)
    if case["entry"] == "block":
        return {"rel": 1e-2}
    return {"rel": {"float32": 2e-5, "bfloat16": 5e-3, "float16": 1e-3}[case["dtype"]]}
