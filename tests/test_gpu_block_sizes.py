"""The window binning's block sizes (rows per block by the snapshot's rows and channels, samples per
thread of preprocessed input) against the tile gridder, whose binning is separate code: row counts
around a block of 64 rows and above, channel counts around the groups of threads that share a row,
and from 16384 rows on rows read four at a time, a multiple of 4 and with one to three left over.

Tolerance: both gridders sum n <= 70000 samples of the same sign in FP32, errors of at most about
sqrt(n) 2^-24 of a cell's sum (1.6e-5, averaged away in the image's central half); a sample lost or
counted twice is 1 / n >= 1.4e-5 of the peak, so the bound there is 8e-6 as for fewer samples.
"""
import numpy as np
import pytest
import torch

from conftest import announce
import svdimager_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,channels", [(r, c) for r in (3, 5, 63, 64, 260, 1021, 1024) for c in (1, 8, 9, 17, 64, 67)] +
                         [(16384, 4), (16385, 1), (16386, 3), (16387, 4), (20000, 2), (33001, 2)])
def test_block_sizes_match_the_tile_gridder(rows, channels):
    announce(f"block sizes rows={rows} channels={channels}")
    N, cell = 96, 1e-4
    rng = np.random.default_rng([rows, channels])
    n = rows * channels
    dev = "cuda"
    t = lambda a, dt=torch.float32: torch.as_tensor(np.asarray(a), dtype=dt, device=dev)
    uvw = rng.normal(0.0, 300.0, (rows, 3)) * np.array([1.0, 0.7, 0.02])
    flags = (rng.random(n) < 0.2).astype(np.uint8)
    snap = {"uvw": t(uvw, torch.float64), "freq": t(np.linspace(1e8, 1.5e8, channels), torch.float64), "num_rows": rows,
            "num_channels": channels, "array_center_x": -2565018.0}
    for pol in (0, 3):
        snap[f"vis{pol}_re"], snap[f"vis{pol}_im"] = t(rng.uniform(0.5, 1.0, n)), t(rng.uniform(-0.2, 0.2, n))
        snap[f"flag{pol}"] = t(flags, torch.uint8)
        snap[f"weight{pol}"] = t(rng.uniform(0.5, 1.0, n))
    d = S.DeviceSnapshot(snap, dev)
    imgs = []
    with S.Context(0) as ctx:
        for gridder in (S.GRIDDER_TILED, S.GRIDDER_MFMA):
            img, plan = S.image_snapshot(ctx, d, N, cell, output=S.OUTPUT_SIGNED, gridder=gridder)
            torch.cuda.synchronize()
            assert plan["gridder"] == gridder
            imgs.append(img.cpu().numpy().astype(np.float64))
    peak = np.abs(imgs[0]).max()
    c = slice(N // 4, 3 * N // 4)
    assert np.isfinite(imgs[1]).all()
    assert np.abs(imgs[1] - imgs[0])[c, c].max() <= 8e-6 * peak
    assert np.abs(imgs[1] - imgs[0]).max() <= 3e-5 * peak
