"""The MFMA gridder where its dense halves make more pieces than there are partial slots, so that the
work shape is made coarser on the device, against the plain FP32 tile gridder: many dense halves
(the threshold rises), one half of many pieces (the pieces grow), both, and fewer than the slots.

Tolerance: both gridders sum n <= 70000 samples of the same sign in FP32, errors of at most about
sqrt(n) 2^-24 of a cell's sum (1.6e-5, averaged away in the image's central half, divided by the grid
correction at its edge); a sample lost or counted twice is 1 / n >= 1.4e-5 of the peak everywhere.
"""
import numpy as np
import pytest
import torch

from conftest import announce
import svdimager_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,N,n,terms,coop_min,class_log2", [
    ("wide", 64, 20000, 8, 32, 2), ("wide", 64, 70000, 8, 32, 3), ("wide", 128, 70000, 32, 32, 2),
    ("hot", 16, 60000, 32, 256, 2), ("hot", 16, 70000, 8, 32, 3), ("mixed", 64, 70000, 32, 32, 2),
    ("mixed", 30, 50000, 16, 64, 2), ("wide", 64, 70000, 8, 1024, 2),
])
def test_shape_past_the_slots_matches_the_tile_gridder(kind, N, n, terms, coop_min, class_log2):
    announce(f"work shape {kind} N={N} n={n} terms={terms} coop_min={coop_min} class={class_log2}")
    G = (3 * N + 1) // 2
    cell = np.float32(1e-3)
    rng = np.random.default_rng([N, n, terms])
    p = rng.uniform(-G / 2, G / 2, (n, 2))
    hot = np.arange(n) < {"wide": 0, "hot": n, "mixed": n // 2}[kind]
    p[hot] = rng.uniform(-0.5, 0.5, (int(hot.sum()), 2)) + np.array([-4.25, 3.75])
    b = np.concatenate([p / (np.float64(cell) * G), rng.uniform(-3.0, 3.0, (n, 1))], axis=1).astype(np.float32)
    t = lambda a: torch.as_tensor(np.asarray(a, np.float32), device="cuda")
    vre, vim = rng.uniform(0.5, 1.0, n), rng.uniform(-0.25, 0.25, n)
    with S.Context(0) as ctx:
        ctx.set_tuning(G, coop_min=coop_min, coop_cap=4096, class_log2=class_log2)
        images = []
        for gridder in (S.GRIDDER_TILED, S.GRIDDER_MFMA):
            img, plan = S.FIpipeDevice(ctx, t(b), t(np.eye(3)), t(vre), t(vim), N, float(cell), output=S.OUTPUT_SIGNED,
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
