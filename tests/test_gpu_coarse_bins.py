"""Coarse binning of the MFMA gridder (bins past its LDS histogram: eight row classes binned together,
then sorted by class) against the plain FP32 tile gridder, on the grids where it can go wrong:

* 2304^2 and 2343^2 (the last coarse bin of a window column is partial; odd side), 8- and 4-row classes;
* coarse bins of one piece (512 records), exactly one, one more, and of many pieces;
* footprints clipped by the grid's edges, positions on integers and one FP32 step above them, at
  multiples of 64 rows, where the coarse bins meet;
* several slabs, and planes too small to hold the records (the bins themselves in LDS bands).

Tolerance: as for the dense halves, n <= 20000 unit samples summed in FP32 by both gridders: 8e-6 of
the peak in the central half and 3e-5 at the edge, while one sample lost or counted twice is
1 / n >= 5e-5 of the peak everywhere.
"""
import numpy as np
import pytest
import torch

from conftest import announce
import svdimager_amd as S

pytestmark = pytest.mark.gpu


def positions(kind, n, G, rng):
    p = rng.uniform(-G / 2 - 6, G / 2 + 6, (n, 2))
    if kind == "hot":
        p = rng.uniform(-20.0, 20.0, (n, 2))
    elif kind == "one-bin":
        p = np.stack([rng.uniform(8.0, 50.0, n) + (64 * 10 - G // 2), rng.uniform(4.0, 11.0, n) + (16 * 40 - G // 2)], 1)
    elif kind == "borders":                        # first footprint cells around multiples of 64 rows
        p[:, 0] = 64 * rng.integers(1, G // 64, n) - G // 2 + 4 + rng.integers(-1, 2, n)
        up = rng.random(n) < 0.5
        p = p.astype(np.float32)
        p[up] = np.nextafter(p[up], np.float32(1e9))
    elif kind == "edges":
        p = np.where(rng.random((n, 2)) < 0.5, -G / 2 - 3.9, G / 2 - 4.5) + rng.uniform(0.0, 8.0, (n, 2))
    return np.asarray(p, np.float32)


@pytest.mark.parametrize("kind,n,N,terms,class_log2,r3", [
    ("wide", 20000, 1536, 8, 0, 1.0), ("wide", 20000, 1562, 3, 0, 1.0), ("hot", 20000, 1536, 8, 0, 1.0),
    ("hot", 20000, 1562, 9, 2, 1.0), ("one-bin", 512, 1536, 8, 0, 1.0), ("one-bin", 513, 1536, 8, 0, 1.0),
    ("one-bin", 20000, 1562, 8, 0, 1.0), ("borders", 20000, 1536, 8, 0, 1.0), ("borders", 20000, 1562, 8, 2, 1.0),
    ("edges", 20000, 1562, 8, 0, 1.0), ("wide", 20000, 1024, 8, 0, 6.0e4), ("hot", 20000, 1024, 8, 0, 6.0e4),
])
def test_coarse_bins_match_the_tile_gridder(kind, n, N, terms, class_log2, r3):
    announce(f"coarse {kind} n={n} N={N} terms={terms} class={class_log2} r3={r3}")
    G = (3 * N + 1) // 2
    cell = np.float32(2e-5)
    rng = np.random.default_rng([n, N, len(kind)])
    p = positions(kind, n, G, rng)
    b = np.concatenate([p / (cell * np.float32(G)), rng.uniform(-r3, r3, (n, 1))], axis=1).astype(np.float32)
    t = lambda a: torch.as_tensor(np.asarray(a, np.float32), device="cuda")
    vre, vim = rng.uniform(0.5, 1.0, n), rng.uniform(-0.25, 0.25, n)
    with S.Context(0) as ctx:
        if class_log2:
            ctx.set_tuning(G, class_log2=class_log2)
        images = []
        for gridder in (S.GRIDDER_TILED, S.GRIDDER_MFMA):
            img, plan = S.FIpipeDevice(ctx, t(b), t(np.eye(3)), t(vre), t(vim), N, float(cell), output=S.OUTPUT_SIGNED,
                                       gridder=gridder, num_terms=terms)
            torch.cuda.synchronize()
            assert plan["gridder"] == gridder
            assert plan["num_slabs"] > 2 or r3 < 2.0
            images.append(img.cpu().numpy().astype(np.float64))
    ref, got = images
    peak = np.abs(ref).max()
    c = slice(N // 4, 3 * N // 4)
    assert np.isfinite(got).all() and peak > 0
    assert np.abs(got - ref)[c, c].max() <= 8e-6 * peak
    assert np.abs(got - ref).max() <= 3e-5 * peak


def test_records_in_bands_when_the_planes_are_small():
    """More samples than the planes can hold records of (one term at 3 slabs of 1024^2): the bands."""
    announce("coarse: planes too small")
    N, n, terms = 1562, 1_400_000, 1
    G, cell = (3 * N + 1) // 2, np.float32(2e-5)
    assert 2 * n * 16 > terms * 8 * G * G and (G + 15) // 16 * ((G + 7) // 8) > 36864
    rng = np.random.default_rng(5)
    p = rng.uniform(-G / 2, G / 2, (n, 2)).astype(np.float32)
    b = np.concatenate([p / (cell * np.float32(G)), rng.uniform(-1.0, 1.0, (n, 1))], axis=1).astype(np.float32)
    t = lambda a: torch.as_tensor(np.asarray(a, np.float32), device="cuda")
    # (Random phases: every pixel is a sum of n terms of random sign, so errors are set against the
    # rms of the image, by the same bound as above: a lost sample is 1 / sqrt(n) >= 8e-4 of it.)
    ph = rng.uniform(0.0, 2.0 * np.pi, n)
    with S.Context(0) as ctx:
        imgs = []
        for gridder in (S.GRIDDER_TILED, S.GRIDDER_MFMA):
            img, _ = S.FIpipeDevice(ctx, t(b), t(np.eye(3)), t(np.cos(ph)), t(np.sin(ph)), N, float(cell),
                                    output=S.OUTPUT_SIGNED, gridder=gridder, num_terms=terms)
            torch.cuda.synchronize()
            imgs.append(img.cpu().numpy().astype(np.float64))
    c = slice(N // 4, 3 * N // 4)
    rms = np.sqrt((imgs[0][c, c] ** 2).mean())
    assert rms > 0
    assert np.abs(imgs[1] - imgs[0])[c, c].max() <= 1e-4 * rms
