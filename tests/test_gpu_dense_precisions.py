"""The sorted contraction of dense half windows in the operand precisions other than the default, at its
edges (footprint clusters at window corners, integer positions with their ninth cells, one step above them,
clipped footprints; one piece and several, one sorted batch and several; one, two and four blocks of eight
terms), against the plain FP32 tile gridder on the same samples.

Bounds, of the peak, n samples of the same sign.  splitc and single round the product of the ES factors
three times to f16 and single the term values once, 4 x 2^-11 of a sample at most, of a sign that the
dithering makes random: 4 x 2^-11 / sqrt(n), which the grid correction amplifies 3 times in the image's
central half and 85 times at its edge.  bf16 keeps 16 bits of either factor and drops the product of the
low halves: 2^-17 + 2^-17 + 2^-18 of a sample, not random where positions repeat, amplified the same way.
Both and the tile gridder add the FP32 sums' 8e-6 (3e-5 at the edge).  A sample lost or counted twice is 1 / n.
"""
import numpy as np
import pytest
import torch

from conftest import announce
from test_gpu_dense import CELL, G, N, SCALE, positions
import svdimager_amd as S

pytestmark = pytest.mark.gpu

CASES = [("corner", 2600, 8, 0), ("corner", 9000, 16, 1 << 20), ("corner", 9000, 20, 4096), ("hot", 300, 32, 0),
         ("hot", 9000, 16, 1 << 20), ("hot", 17000, 8, 1 << 20), ("integers", 6000, 8, 0), ("integers", 6000, 16, 0),
         ("above", 6000, 8, 0), ("above", 6000, 32, 1 << 20), ("first", 9000, 8, 0), ("last", 9000, 16, 0)]


@pytest.mark.parametrize("precision", ["SPLITC", "SINGLE", "BF16"])
@pytest.mark.parametrize("kind,n,terms,cap", CASES)
def test_dense_halves_match_the_tile_gridder(precision, kind, n, terms, cap):
    announce(f"dense {precision} {kind} n={n} terms={terms} cap={cap}")
    rng = np.random.default_rng([n, terms, len(kind)])
    p = positions(kind, n, rng)
    b = np.concatenate([p / np.float32(SCALE), rng.uniform(-3.0, 3.0, (n, 1))], axis=1).astype(np.float32)
    t = lambda a: torch.as_tensor(np.asarray(a, np.float32), device="cuda")
    vre, vim = rng.uniform(0.5, 1.0, n), rng.uniform(-0.25, 0.25, n)
    with S.Context(0) as ctx:
        if cap:
            ctx.set_tuning(G, coop_cap=cap)
        images = []
        for gridder in (S.GRIDDER_TILED, S.GRIDDER_MFMA):
            img, plan = S.FIpipeDevice(ctx, t(b), t(np.eye(3)), t(vre), t(vim), N, CELL, output=S.OUTPUT_SIGNED,
                                       gridder=gridder, num_terms=terms, mfma_precision=getattr(S, "PRECISION_" + precision))
            torch.cuda.synchronize()
            assert plan["gridder"] == gridder
            images.append(img.cpu().numpy().astype(np.float64))
    ref, got = images
    peak = np.abs(ref).max()
    c = slice(N // 4, 3 * N // 4)
    sample = 2.5 * 2.0**-17 if precision == "BF16" else 4 * 2.0**-11 / np.sqrt(n)
    central, whole = np.abs(got - ref)[c, c].max() / peak, np.abs(got - ref).max() / peak
    print(f"central {central:.1e} of {3 * sample + 8e-6:.1e}, whole {whole:.1e} of {85 * sample + 3e-5:.1e}, 1/n {1 / n:.1e}", flush=True)
    assert np.isfinite(got).all() and peak > 0
    assert central <= 3 * sample + 8e-6
    assert whole <= 85 * sample + 3e-5
