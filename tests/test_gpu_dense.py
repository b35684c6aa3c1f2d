"""The MFMA gridder's sorted contraction of dense half windows (k_win_dense) against the plain FP32
tile gridder, on preprocessed samples whose grid positions are chosen to meet its edges:

* clusters around window corners, with counts at its threshold (256 records), at one sorted batch
  (8192) and beyond, in one piece and in several;
* positions that are exact integers (nine-cell footprints, whose last column goes its own way) and
  one FP32 step above integers (the record encoding rounds them to the integer one cell lower);
* footprints clipped by the grid's first and last rows and columns;
* one, two and four blocks of eight terms.

Tolerance: both gridders sum n <= 20000 unit samples in FP32, so a cell's sum errs by at most about
sqrt(n) 2^-24 of itself (8e-6; the image's central half averages it away, its edge divides by the
grid correction), while one sample lost or counted twice is 1 / n >= 5e-5 of the peak everywhere.
"""
import numpy as np
import pytest
import torch

from conftest import announce
import svdimager_amd as S

pytestmark = pytest.mark.gpu

N = 64
G = 96
SCALE = 2.0 ** -5                   # cell G: grid cells per wavelength, exact in FP32
CELL = SCALE / G


def positions(kind, n, rng):
    """(n, 2) grid positions in cells, FP32 (multiples of the FP32 step, exact in cell G bin)."""
    centre = np.array([8.0, -8.0])                 # 16-cell window corners lie at 16 k - 48
    p = rng.normal(0.0, 3.0, (n, 2)) + centre
    if kind == "hot":
        p = rng.uniform(-0.5, 0.5, (n, 2)) + np.array([-4.25, 3.75])
    elif kind == "integers":
        p = np.rint(p)
    elif kind == "above":
        p = np.nextafter(np.rint(p).astype(np.float32), np.float32(1e9))
    elif kind == "first":
        p = np.abs(rng.normal(0.0, 3.0, (n, 2))) - 51.0
    elif kind == "last":
        p = 50.0 - np.abs(rng.normal(0.0, 3.0, (n, 2)))
    return np.asarray(p, np.float32)


@pytest.mark.parametrize("kind,n,terms,cap", [
    ("corner", 240, 8, 0), ("corner", 2600, 8, 0), ("corner", 20000, 8, 0), ("corner", 20000, 16, 1 << 20),
    ("corner", 20000, 32, 0), ("corner", 9000, 20, 4096), ("hot", 8192, 8, 1 << 20), ("hot", 8193, 1, 1 << 20),
    ("hot", 300, 12, 0), ("integers", 6000, 8, 0), ("integers", 6000, 16, 0), ("above", 6000, 8, 0),
    ("above", 6000, 32, 1 << 20), ("first", 12000, 8, 0), ("last", 12000, 16, 0),
])
def test_dense_halves_match_the_tile_gridder(kind, n, terms, cap):
    announce(f"dense {kind} n={n} terms={terms} cap={cap}")
    rng = np.random.default_rng([n, terms, len(kind)])
    p = positions(kind, n, rng)
    b = np.concatenate([p / np.float32(SCALE), rng.uniform(-3.0, 3.0, (n, 1))], axis=1).astype(np.float32)
    assert np.float32(CELL) * np.float32(G) == np.float32(SCALE)
    t = lambda a: torch.as_tensor(np.asarray(a, np.float32), device="cuda")
    vre, vim = rng.uniform(0.5, 1.0, n), rng.uniform(-0.25, 0.25, n)
    vin = t(np.eye(3))
    with S.Context(0) as ctx:
        if cap:
            ctx.set_tuning(G, coop_cap=cap)
        images = []
        for gridder in (S.GRIDDER_TILED, S.GRIDDER_MFMA):
            img, plan = S.FIpipeDevice(ctx, t(b), vin, t(vre), t(vim), N, CELL, output=S.OUTPUT_SIGNED,
                                       gridder=gridder, num_terms=terms)
            torch.cuda.synchronize()
            assert plan["gridder"] == gridder
            images.append(img.cpu().numpy().astype(np.float64))
    ref, got = images
    peak = np.abs(ref).max()
    c = slice(N // 4, 3 * N // 4)
    assert np.isfinite(got).all() and peak > 0
    assert np.abs(got - ref)[c, c].max() <= 8e-6 * peak
    assert np.abs(got - ref).max() <= 3e-5 * peak
