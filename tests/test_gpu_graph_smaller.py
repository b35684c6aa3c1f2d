"""Graph capture of a planned call whose snapshot has fewer rows than the one the context was warmed with
(rows dropped as flagged): the workspace of the larger call must do, whatever other block sizes, bins or
slots the smaller one takes.  The replay is checked against an eager call on the same snapshot.

Tolerance: as for two summation orders of the same gridder, 1e-5 of peak over the image and 1e-6 over the
central half."""
import numpy as np
import pytest
import torch

from conftest import announce, assert_parity
import svdimager_amd as S

pytestmark = pytest.mark.gpu


def _snapshot(uvw, channels):
    n = uvw.shape[0] * channels
    rng = np.random.default_rng(n)
    t = lambda a, dt=torch.float32: torch.as_tensor(np.asarray(a), dtype=dt, device="cuda")
    snap = {"uvw": t(uvw, torch.float64), "freq": t(np.linspace(1e8, 1.2e8, channels), torch.float64),
            "num_rows": uvw.shape[0], "num_channels": channels, "array_center_x": -2565018.0}
    for pol in (0, 3):
        snap[f"vis{pol}_re"], snap[f"vis{pol}_im"] = t(rng.uniform(0.5, 1.0, n)), t(rng.uniform(-0.2, 0.2, n))
        snap[f"flag{pol}"] = torch.zeros(n, dtype=torch.uint8, device="cuda")
        snap[f"weight{pol}"] = None
    return S.DeviceSnapshot(snap, "cuda")


# Fewer rows in more blocks of the binning; fewer rows than blocks of four rows at a time take; records that
# do not fit the planes, then ones that do (coarse bins, with more counts); 25 % more samples than slots are sized by.
@pytest.mark.parametrize("rows,kept,channels,N,terms", [
    (66_000, 65_500, 2, 128, 8), (16_500, 16_300, 9, 128, 8), (33_000, 30_100, 33, 256, 8),
    (1_500_000, 1_000_000, 1, 1562, 1), (20_000, 16_383, 64, 96, 16),
])
def test_capture_with_fewer_rows(rows, kept, channels, N, terms):
    announce(f"capture {kept} of {rows} rows x {channels} at {N}^2, {terms} terms")
    rng = np.random.default_rng([rows, N])
    uvw = rng.normal(0.0, 600.0, (rows, 3)) * np.array([1.0, 0.8, 0.02])
    large, small = _snapshot(uvw, channels), _snapshot(uvw[:kept], channels)
    cell = 2.5e-4
    opts = dict(output=S.OUTPUT_SIGNED, gridder=S.GRIDDER_MFMA, num_terms=terms)
    with S.Context(0) as ctx:
        img = torch.zeros((N, N), dtype=torch.float32, device="cuda")
        _, plan = S.image_snapshot(ctx, large, N, cell, image=img, **opts)
        S.image_snapshot(ctx, large, N, cell, image=img, plan=plan, **opts)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            S.image_snapshot(ctx, small, N, cell, image=img, plan=plan, **opts)
        torch.cuda.synchronize()
        replays = []
        for _ in range(3):
            img.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            replays.append(img.cpu().numpy())
        del graph
        torch.cuda.synchronize()
        S.image_snapshot(ctx, small, N, cell, image=img, plan=plan, **opts)
        torch.cuda.synchronize()
        ref = img.cpu().numpy()
    for got in replays:
        assert np.isfinite(got).all()
        assert_parity(got, ref, "replay vs eager", whole=1e-5, central=1e-6)
