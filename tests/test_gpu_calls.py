"""The host path around the kernels: the passes a call makes as jobs of one launch, the forward that saves no state, and
the choice of lanes per channel for 5-8 states."""
import numpy as np
import pytest
import torch

import capi
from oracle import snd_oracle as O
from oracle import snd_oracle_c as OC
from test_gpu_fwd import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src,dst,outer,rows,cols", [
    (torch.float32, torch.bfloat16, 1, 1, 1), (torch.float32, torch.float16, 1, 1, 4099), (torch.float32, torch.float32, 7, 3, 1),
    (torch.bfloat16, torch.bfloat16, 3, 4, 5 * 49), (torch.float16, torch.float16, 2, 2, 1024), (torch.bfloat16, torch.bfloat16, 5, 16, 260),
])
def test_jobs_clear_and_sum(gpu_device, src, dst, outer, rows, cols):
    """Sums over rows (a cast with one row) against torch in fp32, beside two clears, one with a tail of three words."""
    g = torch.Generator(device=gpu_device).manual_seed(1)
    a = torch.randn(outer, rows, cols, device=gpu_device, generator=g).to(src)
    out = torch.full((outer, cols), 7.0, device=gpu_device, dtype=dst)
    z = torch.ones(16384 // 4 * 3 + 3 + 8, device=gpu_device)
    z2 = torch.ones(64, device=gpu_device)
    dt = {torch.float32: capi.SND_F32, torch.float16: capi.SND_F16, torch.bfloat16: capi.SND_BF16}
    jobs = (capi.Job * 4)(capi.Job(None, None, z.data_ptr(), (z.numel() - 8) * 4, 0, 0, capi.JOB_CLEAR, 0, 0),
                          capi.Job(a.data_ptr(), None, out.data_ptr(), outer, cols, rows, capi.JOB_SUM, dt[src], dt[dst]),
                          capi.Job(None, None, z2.data_ptr(), 0, 0, 0, capi.JOB_CLEAR, 0, 0),          # nothing to do: dropped
                          capi.Job(None, None, z2.data_ptr(), 4, 0, 0, capi.JOB_CLEAR, 0, 0))
    capi.check(capi.lib().snd_run_jobs(jobs, 4, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert (z[:-8] == 0).all() and (z[-8:] == 1).all() and z2[0] == 0 and (z2[1:] == 1).all()
    want = a[:, 0].float()
    for r in range(1, rows):
        want = want + a[:, r].float()
    assert torch.equal(out, want.to(dst))


@pytest.mark.parametrize("n", [1, 65536 * 3 + 1, 2, 65536 * 3 + 2])
def test_rounding_to_bfloat16(gpu_device, n):
    """To nearest even, bit for bit as torch rounds: ties, subnormal values, the largest ones, infinities; a NaN stays one.  Stored one by
    one, and four at a time where the count (n and 22 special values) is a multiple of four."""
    bits = torch.arange(n, device=gpu_device, dtype=torch.int64) * 21845 + (torch.arange(n, device=gpu_device) % 5 - 2) + 0x8000
    special = torch.tensor([0x00008000, 0x00018000, 0x3f808000, 0x3f818000, 0x7f7fffff, 0x7f7f8000, 0x7f800000, 0x7f800001, 0x7fc00000, 1, 0x007fffff],
                           device=gpu_device, dtype=torch.int64)
    bits = torch.cat([bits, special, special + 0x80000000]) & 0xffffffff
    a = torch.where(bits >= 1 << 31, bits - (1 << 32), bits).to(torch.int32).view(torch.float32)
    out = torch.empty(a.numel(), device=gpu_device, dtype=torch.bfloat16)
    job = capi.Job(a.data_ptr(), None, out.data_ptr(), 1, a.numel(), 1, capi.JOB_SUM, capi.SND_F32, capi.SND_BF16)
    capi.check(capi.lib().snd_run_jobs((capi.Job * 1)(job), 1, torch.cuda.current_stream().cuda_stream))
    want, nan = a.to(torch.bfloat16), torch.isnan(a)
    assert torch.equal(torch.isnan(out), nan)
    assert torch.equal(out.view(torch.int16)[~nan], want.view(torch.int16)[~nan])


@pytest.mark.parametrize("src,dst,outer,rows,cols", [
    (torch.float32, torch.float32, 1, 31, 20), (torch.float32, torch.float32, 1, 32, 20),       # either side of the split
    (torch.float32, torch.float32, 3, 33, 1),                                                   # a slice of one row, the last ones of none
    (torch.float32, torch.bfloat16, 2, 129, 15 * 4), (torch.bfloat16, torch.bfloat16, 2, 100, 17 * 4),
    (torch.float16, torch.float16, 5, 3072, 49), (torch.bfloat16, torch.bfloat16, 1, 40, ((1 << 17) - 1) * 4),
    (torch.bfloat16, torch.bfloat16, 1, 40, (1 << 17) * 4), (torch.float32, torch.float16, 1, 8, 1000), (torch.float32, torch.float32, 2, 23, 7),
])
def test_jobs_sum_of_many_rows(gpu_device, src, dst, outer, rows, cols):
    """Rows eight at a time, and dealt to the slices of a block, against float64."""
    g = torch.Generator(device=gpu_device).manual_seed(3)
    a = torch.randn(outer, rows, cols, device=gpu_device, generator=g).to(src)
    out = torch.full((outer * cols + 8,), 7.0, device=gpu_device, dtype=dst)
    dt = {torch.float32: capi.SND_F32, torch.float16: capi.SND_F16, torch.bfloat16: capi.SND_BF16}
    capi.check(capi.lib().snd_run_jobs((capi.Job * 1)(capi.Job(a.data_ptr(), None, out.data_ptr(), outer, cols, rows, capi.JOB_SUM, dt[src], dt[dst])), 1,
                                       torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert (out[-8:] == 7).all()
    want = a.double().sum(1)
    # `rows` additions of half a unit in the last place of fp32 each, and the rounding of the result
    bound = rows * 2.0 ** -24 * a.double().abs().sum(1) + want.abs() * {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dst]
    assert ((out[:-8].view(outer, cols).double() - want).abs() <= bound + 1e-7).all()


@pytest.mark.parametrize("G,rg", [(4, 1), (4, 300), (8, 64)])
def test_jobs_merge_weights(gpu_device, G, rg):
    g = torch.Generator(device=gpu_device).manual_seed(2)
    w = torch.randn(G, rg, device=gpu_device, generator=g)
    w[0, 0] = 0.0
    wdw = torch.randn(G, rg, device=gpu_device, generator=g)
    wdw[0, 0] = 3e-20
    wf = torch.where(w.abs() < 1e-20, torch.full_like(w, 1e-20), w)
    per, grp, fl = torch.empty_like(w), torch.empty(G, device=gpu_device), torch.empty_like(w)
    mk = lambda kind, src, src2, out: capi.Job(src.data_ptr(), src2.data_ptr() if src2 is not None else None, out.data_ptr(), G, rg, 1, kind, 0, 0)
    jobs = (capi.Job * 3)(mk(capi.JOB_WEIGHT, wdw, w, per), mk(capi.JOB_WEIGHT_GROUP, wdw, w, grp), mk(capi.JOB_WEIGHT_FLOOR, w, None, fl))
    capi.check(capi.lib().snd_run_jobs(jobs, 3, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(fl, wf)
    assert torch.allclose(per, wdw / wf, rtol=1e-6)
    assert torch.allclose(grp, (wdw / wf).double().sum(1).float(), rtol=1e-4, atol=1e-4 * float((wdw / wf).abs().max()))


@pytest.mark.parametrize("Bt,Dm,H,W,N,K,dtype,sched", [
    (1, 32, 41, 8, 16, 2, torch.float32, 1),      # one column tile: the row is carried in registers
    (1, 32, 41, 40, 16, 2, torch.float32, 1),     # five: through the block's slab of x_v
    (2, 32, 44, 24, 16, 2, torch.bfloat16, 3),    # bands: a slab each
    (1, 16, 40, 24, 16, 2, torch.float32, 2),     # strips: through the workspace
    (1, 64, 14, 14, 16, 4, torch.float32, 0),
    (70, 16, 21, 14, 7, 4, torch.float16, 0),     # 7x7 tiles, 8-lane kernels
    (66, 16, 17, 12, 8, 4, torch.float32, 0),     # 8-lane kernels, whole four-column chunks
    (65, 16, 24, 20, 6, 4, torch.bfloat16, 0),
    (2, 32, 24, 40, 3, 2, torch.float32, 1),      # 8 lanes for three states
    (1, 32, 40, 24, 4, 2, torch.bfloat16, 2),
    (2, 16, 33, 130, 2, 4, torch.float32, 0),     # row-segment kernels
    (1, 8, 9, 1500, 2, 2, torch.float32, 0),      # wide planes: the column groups hand over through the workspace
])
def test_forward_without_saved_state_is_the_forward(gpu_device, Bt, Dm, H, W, N, K, dtype, sched):
    """What selective_nd_scan returns where no gradient can be asked for, bit for bit what it returns in training."""
    import selective_nd_scan as snd
    d = O.make_inputs(Bt, Dm, H, W, N=N, K=K, seed=3)
    t = {k: torch.from_numpy(v).to(gpu_device) for k, v in d.items()}
    for k in ("u", "delta", "B", "C"):
        t[k] = t[k].to(dtype)
    args = (t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"], True, True, None)
    try:
        snd.set_schedule(sched)
        infer = snd.selective_nd_scan(*args)
        train = snd.selective_nd_scan(t["u"].clone().requires_grad_(), *args[1:])
    finally:
        snd.set_schedule(0)
    assert not infer.requires_grad and train.requires_grad
    assert torch.equal(infer, train.detach())
    with torch.no_grad():
        half = snd.selective_nd_scan(t["u"].clone().requires_grad_(), *args[1:8], False, None)
    assert half.dtype == dtype and not half.requires_grad and relerr(half.float().cpu().numpy(), infer.cpu().numpy()) <= 1e-2


@pytest.mark.parametrize("Bt,H,W,N,dtype", [
    (65, 9, 9, 5, torch.float32),                 # 260 plane chunks: every CU has a block, 8 lanes per channel
    (64, 9, 9, 5, torch.float32),                 # 256: one short of it, 16 lanes
    (66, 14, 21, 8, torch.bfloat16),              # 7x7 tiles
    (66, 17, 12, 8, torch.float32),               # whole four-column chunks
    (67, 10, 13, 6, torch.float16),
])
def test_lanes_per_channel_for_five_to_eight_states(gpu_device, Bt, H, W, N, dtype):
    d = O.make_inputs(Bt, 12, H, W, N=N, K=4, seed=4)                     # 3 channels per group: 13 of 16 are padding
    t = {k: torch.from_numpy(v).to(gpu_device) for k, v in d.items()}
    for k in ("u", "delta", "B", "C"):
        t[k] = t[k].to(dtype)
    args = (t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"])
    f = capi.FwdCall(*args, True, True, None, True, capi.SCHED_AUTO)
    f.launch()
    b = capi.BwdCall(*args, t["dout"], f.x, f.x_v, True, None, f.x_sd, capi.SCHED_AUTO)
    b.launch()
    torch.cuda.synchronize()
    r = {k: t[k].float().cpu().numpy() for k in ("u", "delta", "B", "C")}
    ref = OC.fwd(r["u"], r["delta"], d["A"], r["B"], r["C"], d["D"], d["delta_bias"], True, None, real="f64")
    gref = OC.bwd(r["u"], r["delta"], d["A"], r["B"], r["C"], d["D"], d["delta_bias"], d["dout"], True, None, real="f64")
    assert relerr(f.out.cpu().numpy(), ref) <= 1e-4
    half = dtype != torch.float32
    for nm, a, w in zip(["du", "ddelta", "dA", "dB", "dC", "dD", "ddelta_bias"], [b.du, b.ddelta, b.dA, b.dB, b.dC, b.dD, b.dbias], gref):
        tol = 1e-2 if (half and nm in ("du", "ddelta", "dB", "dC")) else 1e-4
        assert relerr(a.float().cpu().numpy(), w) <= tol, (nm, relerr(a.float().cpu().numpy(), w))


@pytest.mark.parametrize("H,W,N,rg", [(1, 1, 1, 9), (4, 64, 1, 2), (5, 17, 3, 3), (9, 33, 2, 1), (8, 16, 4, 6), (13, 7, 1, 10), (128, 64, 2, 1), (127, 63, 4, 2), (3, 8, 2, 5)])
@pytest.mark.parametrize("save", [True, False])
def test_merge_in_lds(gpu_device, H, W, N, rg, save):
    """One-segment planes merged from the four corners inside the kernel: every element of out is stored (none was cleared)."""
    import ctypes as C
    d = O.make_inputs(2, 4 * rg, H, W, N=N, K=4, seed=6)
    t = {k: torch.from_numpy(v).to(gpu_device) for k, v in d.items()}
    u = t["u"][:, :rg].contiguous()
    w = torch.linspace(-1.0, 2.0, 4 * rg, device=gpu_device)
    args = (u, t["delta"], t["A"], t["B"], t["C"], t["D"], t["delta_bias"], True, True, None)
    f = capi.FwdCall(*args, save, capi.SCHED_WAVEFRONT, capi.DIR_CORNERS, True, w)
    assert capi.lib().snd_fwd_merge_stores(C.byref(f.params.shape), capi.SCHED_WAVEFRONT, capi.DIR_CORNERS) == 1
    f.out.fill_(float("nan"))
    f.launch()
    f0 = capi.FwdCall(*args, True, capi.SCHED_WAVEFRONT, capi.DIR_CORNERS)
    f0.launch()
    torch.cuda.synchronize()
    want = (f0.out.double() * w.double().view(1, -1, 1, 1)).view(2, 4, rg, H, W).sum(1)
    assert relerr(f.out.cpu().numpy(), want.cpu().numpy()) <= 1e-5
