"""The tile backward's dB / dC: neighbouring 8x8 tiles of a strip leave together (an odd tile out at either end leaves alone), the
terms that all states or all channels share are summed per pixel, and each tile's inputs are requested under the tile before it.
Odd and even numbers of tiles, a single one, tiles cut by the plane's edge, vector and element-wise staging, 7x7 tiles, fewer states than lanes,
against the float64 oracle."""
import pytest
import torch

import capi
from oracle_ref import reference
from test_gpu_fwd import relerr
from test_gpu_wave import NAMES, run

pytestmark = pytest.mark.gpu

PAIRS = [
    # Bt, Dm, H, W, N, dtype, kw: 4 groups
    (2, 64, 16, 8, 16, torch.float32, {}),                       # one tile per strip
    (2, 72, 24, 24, 16, torch.float32, {}),                      # three: the last alone; 18 channels, two of them in a block of their own
    (1, 64, 9, 28, 16, torch.float32, {}),                       # four, the last half empty; a strip of one row
    (2, 64, 17, 37, 9, torch.float32, dict(decay=0.9)),          # five, element-wise staging, nine states
    (1, 64, 20, 20, 6, torch.float32, dict(dirs=capi.DIR_CORNERS)),   # eight lanes per channel, vector staging, mirrored
    (1, 64, 11, 19, 5, torch.float32, dict(dirs=capi.DIR_CORNERS, decay=0.9)),
    (1, 64, 12, 24, 3, torch.float32, {}),                       # four lanes per channel
    (2, 64, 14, 14, 16, torch.float32, dict(dirs=capi.DIR_CORNERS)),  # 7x7 tiles
    (1, 64, 16, 72, 16, torch.bfloat16, dict(dirs=capi.DIR_CORNERS)),
    (1, 64, 13, 45, 8, torch.float16, {}),
    (2, 72, 7, 7, 16, torch.float32, dict(dirs=capi.DIR_CORNERS, decay=0.9)),   # planes of a single tile: 7x7, cut, 8x8
    (3, 64, 5, 6, 9, torch.bfloat16, {}),
    (2, 64, 8, 8, 7, torch.float32, dict(dirs=capi.DIR_CORNERS)),
    (2, 64, 8, 8, 16, torch.bfloat16, {}),
    (2, 64, 6, 7, 3, torch.float32, {}),
]


@pytest.mark.parametrize("sched", [capi.SCHED_PLANE, capi.SCHED_STRIPS])
@pytest.mark.parametrize("Bt,Dm,H,W,N,dtype,kw", PAIRS)
def test_tile_pairs_match_the_oracle(gpu_device, Bt, Dm, H, W, N, dtype, kw, sched):
    print("tile pairs", Bt, Dm, H, W, N, dtype, kw, sched, flush=True)
    d, t, f, b = run(gpu_device, Bt, Dm, H, W, N, 4, None, dtype, sched, **kw)
    r = {k: t[k].float().cpu().numpy() for k in ("u", "delta", "B", "C")}
    _, gref = reference(r["u"], r["delta"], d["A"], r["B"], r["C"], d["D"], d["delta_bias"], d["dout"], True, kw.get("decay"),
                        kw.get("dirs") == capi.DIR_CORNERS)
    # An adjoint or a state gathers four roundings per cell on its way over at most H + W cells (|a| <= 1), a gradient then the
    # sums over states, channels or pixels, of which rounding errors add up like the square root of their number; a's own error, about
    # eight roundings, scales with delta * A.  Against the largest value; du, ddelta leave in the inputs' type.
    bound = (4 * (H + W) + N + Dm // 4 + (Bt * H * W) ** 0.5 + 8) * 2.0 ** -24
    for nm, a, w in zip(NAMES, [b.du, b.ddelta, b.dA, b.dB, b.dC, b.dD, b.dbias, b.ddec], gref):
        assert (a is None) == (w is None), nm
        if a is None:
            continue
        tol = bound + ({torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}.get(dtype, 0.0) if nm in ("du", "ddelta") else 0.0)
        e = relerr(a.float().cpu().numpy(), w)
        assert e <= tol, (nm, e, tol)
