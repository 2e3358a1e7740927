"""The forward with a wave per state (5 to 16 states, at most 64 columns, few planes): against the float64 oracle and
the tile kernels over what the route accepts - one, two and four planes to a wave and partly filled waves, rows that are no
multiple of a band, mirrored orders, spaced rows, shared delta, both out types, the fused merge, decay, no softplus, infinities, a
captured graph - and the tile backward from the state it saves."""
import ctypes as C

import numpy as np
import pytest
import torch

import capi
from oracle import snd_oracle as O
from oracle_ref import reference
from selective_nd_scan import selective_nd_scan
from test_gpu_fwd import relerr
from test_gpu_wave import NAMES

pytestmark = pytest.mark.gpu

CASES = [
    # Bt, Dm, H, W, N, K, Dd, dtype, kw
    (1, 64, 14, 14, 16, 4, None, torch.float32, {}),
    (2, 24, 1, 1, 5, 4, None, torch.float32, {}),                  # one cell, (below) a plane of one tile: both stay with the tile kernels
    (1, 36, 3, 7, 16, 4, None, torch.float32, dict(corners=True)),
    (2, 24, 9, 1, 5, 4, None, torch.float32, {}),                  # one column
    (1, 24, 1, 9, 5, 4, None, torch.float32, dict(corners=True)),  # one row
    (1, 36, 15, 7, 16, 4, None, torch.float32, dict(corners=True)),  # 9 channels per group: the last wave holds one plane of four
    (1, 20, 4, 16, 8, 2, 10, torch.bfloat16, dict(corners=True)),  # a full quarter wave, one whole band, delta shared in pairs
    (3, 15, 5, 17, 9, 3, None, torch.float16, {}),                 # two planes to a wave, three groups, one row in the last band
    (1, 28, 9, 32, 12, 4, None, torch.float32, dict(corners=True, decay=0.9)),
    (1, 12, 13, 33, 6, 4, None, torch.float32, dict(softplus=False)),
    (1, 8, 30, 64, 15, 4, None, torch.bfloat16, dict(out_float=False, plain=True)),
    (1, 16, 57, 50, 16, 4, None, torch.float32, dict(corners=True)),
    (2, 16, 10, 20, 7, 4, None, torch.float32, dict(spaced=True, corners=True)),
]


def _make(dev, Bt, Dm, H, W, N, K, Dd, dtype, seed=5):
    d = O.make_inputs(Bt, Dm, H, W, N=N, K=K, seed=seed, Dd=Dd)
    t = {k: torch.from_numpy(v).to(dev) for k, v in d.items()}
    for k in ("u", "delta", "B", "C"):
        t[k] = t[k].to(dtype)
    return d, t


def _route(f):
    """Whether the plan says that AUTO's forward of this call is the one with a wave per state."""
    return f.plan.wave_per_state == 1


@pytest.mark.parametrize("Bt,Dm,H,W,N,K,Dd,dtype,kw", CASES)
def test_wave_per_state_matches_oracle_and_tiles(gpu_device, Bt, Dm, H, W, N, K, Dd, dtype, kw):
    print("wave per state", Bt, Dm, H, W, N, K, Dd, dtype, kw, flush=True)
    d, t = _make(gpu_device, Bt, Dm, H, W, N, K, Dd, dtype)
    softplus, decay, plain = kw.get("softplus", True), kw.get("decay"), kw.get("plain", False)
    if not softplus:
        t["delta"] = torch.nn.functional.softplus(t["delta"] - 3.0)
    if kw.get("spaced"):                              # rows, channels and images further apart than they need be
        for k in ("u", "delta", "B", "C"):
            x = torch.full(tuple(t[k].shape[:-2]) + (H + 2, W + 3), float("nan"), device=gpu_device, dtype=dtype)
            x[..., :H, :W] = t[k]
            t[k] = x[..., :H, :W]
    D, bias = None if plain else t["D"], t["delta_bias"] if softplus and not plain else None
    dirs = capi.DIR_CORNERS if kw.get("corners") else capi.DIR_TOPLEFT
    dec = torch.tensor([decay], device=gpu_device) if decay is not None else None
    args = (t["u"], t["delta"], t["A"], t["B"], t["C"], D, bias)
    outs, grads = [], []
    for sched in (capi.SCHED_AUTO, capi.SCHED_PLANE):  # the wave per state, the tile kernels
        f = capi.FwdCall(*args, softplus, kw.get("out_float", True), dec, True, sched, dirs)
        assert _route(f) == (f.plan.n_chunks_x * f.plan.n_chunks_y > 1)
        f.out.fill_(float("nan"))
        for x in (f.x, f.x_v, f.x_sd):                 # (what a launch does not write must not matter to the backward)
            x.fill_(float("nan"))
        f.launch()
        b = capi.BwdCall(*args, t["dout"], f.x, f.x_v, softplus, dec, f.x_sd, capi.SCHED_PLANE, dirs)
        b.launch()
        e = capi.FwdCall(*args, softplus, kw.get("out_float", True), dec, False, sched, dirs)
        e.launch()
        torch.cuda.synchronize()
        assert torch.equal(f.out, e.out)               # saved or not
        outs.append(f.out.float().cpu().numpy())
        grads.append([None if g is None else g.float().cpu().numpy() for g in (b.du, b.ddelta, b.dA, b.dB, b.dC, b.dD, b.dbias, b.ddec)])
    r = {k: t[k].float().cpu().numpy() for k in ("u", "delta", "B", "C")}
    ref, gref = reference(r["u"], r["delta"], d["A"], r["B"], r["C"], None if plain else d["D"], d["delta_bias"] if bias is not None else None,
                       d["dout"], softplus, decay, bool(kw.get("corners")))
    # a state gathers four roundings per cell on its way over at most H + W cells (|a| <= 1), out then the sum over the states; a's own
    # error, about eight roundings, scales with delta * A.  out in 16 bits: half a unit of its last place.
    bound = (4 * (H + W) + N + 16) * 2.0 ** -24 + (2.0 ** -8 if kw.get("out_float") is False else 0.0)
    assert np.isfinite(outs[0]).all()
    assert relerr(outs[0], ref) <= bound
    assert relerr(outs[0], outs[1]) <= 2 * bound
    # the gradients from its saved state: as far from the oracle as from the tile kernels' own, give or take the saved state's bound
    if Dd is None:
        for nm, a, w, r_ in zip(NAMES, grads[0], grads[1], gref):
            if a is not None and np.abs(r_).max() > 1e-12:
                assert relerr(a, r_) <= relerr(w, r_) + bound + (Bt * H * W) ** 0.5 * 2.0 ** -24, nm


@pytest.mark.parametrize("H,W,N", [(15, 7, 16), (10, 30, 6), (6, 50, 9)])
def test_wave_per_state_merge(gpu_device, H, W, N):
    """The four corners of one map added up inside the call, against the same without the merge."""
    Bt, Dm, K = 2, 20, 4
    d, t = _make(gpu_device, Bt, Dm, H, W, N, K, None, torch.float32)
    w = torch.linspace(-1.0, 2.0, Dm, device=gpu_device)
    u = t["u"][:, :Dm // K].contiguous()
    args = (u, t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"])
    m = capi.FwdCall(*args, True, True, None, False, capi.SCHED_AUTO, capi.DIR_CORNERS, True, w)
    assert _route(m)
    m.launch()
    f = capi.FwdCall(u.repeat(1, K, 1, 1), *args[1:], True, True, None, False, capi.SCHED_PLANE, capi.DIR_CORNERS)
    f.launch()
    want = (f.out * w.view(1, -1, 1, 1)).view(Bt, K, Dm // K, H, W).sum(1)
    assert relerr(m.out.cpu().numpy(), want.cpu().numpy()) <= (8 * (H + W) + N + 32) * 2.0 ** -24


@pytest.mark.parametrize("W", [7, 16, 30, 64])
def test_wave_per_state_keeps_infinities_to_their_plane(gpu_device, W):
    Bt, Dm, H, N, K = 1, 24, 9, 8, 4
    _, t = _make(gpu_device, Bt, Dm, H, W, N, K, None, torch.float32)
    args = [t[k] for k in ("u", "delta", "A", "B", "C", "D", "delta_bias")]
    clean = capi.FwdCall(*args, True, True, None, False)
    assert _route(clean)
    clean.launch()
    args[0] = t["u"].clone()
    args[0][0, 7, 2, W // 2] = float("inf")
    f = capi.FwdCall(*args, True, True, None, False)
    f.launch()
    torch.cuda.synchronize()
    keep = torch.arange(Dm, device=gpu_device) != 7
    assert torch.equal(f.out[:, keep], clean.out[:, keep])
    assert not torch.isfinite(f.out[0, 7, 2:, W // 2:]).all() and torch.equal(f.out[0, 7, :2], clean.out[0, 7, :2])


# (run: the cells whose a the scan has multiplied when it first meets the state on their left: 8 lanes of a row of 16, the
# 16-lane rows of a half wave, the upper half wave)
@pytest.mark.parametrize("H,W,N,first,run", [(10, 14, 16, 6, 8), (16, 16, 5, 8, 8), (9, 30, 8, 16, 14), (10, 33, 6, 16, 16), (12, 60, 16, 32, 28)])
@pytest.mark.parametrize("left", [0.0, 1e-30])
def test_wave_per_state_where_products_of_a_overflow(gpu_device, H, W, N, first, run, left):
    """a > 1: along a row the a of neighbouring cells multiply to more than a float holds while the states stay in range, as the
    recurrence has it - nothing on the left (0) or a state so small that the product brings it to about 1e10.  One such channel among
    ordinary ones, whose results do not change."""
    Bt, Dm, K, odd = 1, 24, 4, 8
    d, t = _make(gpu_device, Bt, Dm, H, W, N, K, None, torch.float32)
    lam = 92.0 / run
    t["delta"] = torch.nn.functional.softplus(t["delta"] - 3.0)

    def call(sched):
        f = capi.FwdCall(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], None, False, True, None, True, sched)
        for x in (f.x, f.x_v, f.x_sd):
            x.zero_()
        f.launch()
        torch.cuda.synchronize()
        return f
    plain = call(capi.SCHED_AUTO)
    assert _route(plain)
    plain = plain.out
    t["u"][0, odd] = 0.0
    t["u"][0, odd, H - 2, first - 1] = left
    t["u"][0, odd, H - 2, W - 2] = 1.0
    t["delta"][0, odd], t["A"][odd] = lam, 1.0
    auto, tiles = call(capi.SCHED_AUTO), call(capi.SCHED_PLANE)
    keep = torch.arange(Dm, device=gpu_device) != odd
    assert torch.equal(auto.out[:, keep], plain[:, keep])
    r = {k: t[k].cpu().numpy() for k in ("u", "delta", "A", "B", "C")}
    ref, _ = reference(r["u"], r["delta"], r["A"], r["B"], r["C"], d["D"], None, d["dout"], False, None, False)
    # four roundings per cell, and an exponent's rounding: a product's exponent adds up to 92 or so
    bound = (4 * (H + W) + N + 16 + 2 * 100) * 2.0 ** -24
    for f in (auto, tiles):
        assert bool(torch.isfinite(f.out).all())
        assert relerr(f.out[0, odd].cpu().numpy(), ref[0, odd]) <= bound
    for x in (auto.x, auto.x_v, auto.x_sd.flatten()[:-1]):   # (the last word of x_sd says which family wrote it)
        assert bool(torch.isfinite(x).all())


def test_wave_per_state_in_a_captured_graph(gpu_device):
    _, t = _make(gpu_device, 1, 64, 14, 14, 16, 4, None, torch.float32)
    args = [t[k] for k in ("u", "delta", "A", "B", "C", "D", "delta_bias")]
    f = capi.FwdCall(*args, True, True, None, False)
    assert _route(f)
    f.launch()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        f.launch()
    for k in range(3):
        args[0].mul_(1.5)
        e = capi.FwdCall(*args, True, True, None, False)
        e.launch()
        f.out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(f.out, e.out)


def test_wave_per_state_is_one_launch(gpu_device):
    """The public call without gradients: out and nothing beside it is worked on - no workspace, no clearing launch."""
    _, t = _make(gpu_device, 1, 64, 14, 14, 16, 4, None, torch.float32)
    args = [t[k] for k in ("u", "delta", "A", "B", "C", "D", "delta_bias")]
    with torch.no_grad():
        ref = selective_nd_scan(*args, True)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(g):
            out = selective_nd_scan(*args, True)
    n = C.c_size_t(0)
    assert capi.lib().hipGraphGetNodes(C.c_void_p(g.raw_cuda_graph()), None, C.byref(n)) == 0
    assert n.value == 1
    g.instantiate()
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
