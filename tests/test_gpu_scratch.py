"""The MFMA gridder's scratch, which lies in the buffer of the transformed rows: what a context holds
after a call, and the no-allocation call over several slab batches, whose work shape is the same for each.

Bounds: the context holds the planes, the transformed rows and columns, 32 bytes a sample for records,
24 a row for the rotation, a slot (K 16 x 24 cells) for every 4608 samples, and at most 24 bytes for every
bin of 4 x 16 cells and 256 for every window of 16 x 16 otherwise, plus 2 MiB for what does not grow.  The
no-allocation call runs the kernels of the allocating one; it recomputes two tables (about 15 us) and waits
for its stream, so twice the time is ample, where a work shape that collapses costs several times."""
import time

import numpy as np
import pytest
import torch

from conftest import announce, assert_parity, load_small_snapshot
import svdimager_amd as S
from svdimager_amd import synth

pytestmark = pytest.mark.gpu


def _core_snapshot(rows, channels, seed):
    """A dense core of baselines (wavelengths at 100 MHz) over several slabs of r3."""
    rng = np.random.default_rng(seed)
    n = rows * channels
    uvw = np.concatenate([rng.normal(0.0, 90.0, (rows // 2, 3)), rng.normal(0.0, 900.0, (rows - rows // 2, 3))])
    uvw *= np.array([1.0, 0.8, 0.5])
    t = lambda a, dt=torch.float32: torch.as_tensor(np.asarray(a), dtype=dt, device="cuda")
    snap = {"uvw": t(uvw, torch.float64), "freq": t(np.linspace(1e8, 1.2e8, channels), torch.float64), "num_rows": rows,
            "num_channels": channels, "array_center_x": -2565018.0}
    for pol in (0, 3):
        ph = rng.uniform(0.0, 2.0 * np.pi, n)
        snap[f"vis{pol}_re"], snap[f"vis{pol}_im"] = t(np.cos(ph)), t(np.sin(ph))
        snap[f"flag{pol}"] = torch.zeros(n, dtype=torch.uint8, device="cuda")
        snap[f"weight{pol}"] = None
    return S.DeviceSnapshot(snap, "cuda")


@pytest.mark.parametrize("name", ["small", "core-512", "skalow"])
def test_the_workspace_is_bounded(name):
    announce(f"workspace of {name}")
    if name == "small":
        snap = load_small_snapshot()
        d, N, cell = S.DeviceSnapshot(snap, "cuda"), snap["image_size"], snap["cell"]
    elif name == "core-512":
        d, N, cell = _core_snapshot(81_103, 64, 1), 512, 2e-5
    else:
        d, N, cell = S.DeviceSnapshot(synth.make_snapshot(synth.SKALOW, device="cuda"), "cuda"), 1024, synth.SKALOW.cell
    with S.Context(0) as ctx:
        _, plan = S.image_snapshot(ctx, d, N, cell, gridder=S.GRIDDER_MFMA)
        held = ctx.workspace_bytes()
    G, K, planes = (3 * N + 1) // 2, plan["num_terms"], plan["num_terms"] * plan["batch_slabs"]
    n, slabs = d.num_samples, plan["batch_slabs"]
    bound = 8 * planes * (G * G + G * N + N * N) + 32 * n + 24 * d.num_rows + (n // 4608 + 16) * K * 16 * 24 * 8
    bound += slabs * ((G // 4 + 2) * (G // 16 + 2) * 24 + (G // 16 + 1) ** 2 * 256) + (1 << 21)
    assert held <= bound, (held / 2**20, bound / 2**20)


# Five slabs of 3.8 M samples; 5.2 M samples that leave the slots less than they would take otherwise.
@pytest.mark.parametrize("rows,channels,N,cell,terms,slabs", [(80_001, 48, 384, 5e-4, 0, 3), (130_816, 40, 250, 5e-5, 16, 1)])
def test_noalloc_against_the_allocating_call(rows, channels, N, cell, terms, slabs):
    d = _core_snapshot(rows, channels, 2)
    with S.Context(0) as ctx:
        opts = dict(output=S.OUTPUT_SIGNED, gridder=S.GRIDDER_MFMA, num_terms=terms)

        def image(**kw):
            img, plan = S.image_snapshot(ctx, d, N, cell, **opts, **kw)
            torch.cuda.synchronize()
            return img.cpu().numpy(), plan

        def seconds(**kw):
            best = np.inf
            for _ in range(5):
                torch.cuda.synchronize()
                t = time.perf_counter()
                S.image_snapshot(ctx, d, N, cell, **opts, **kw)
                torch.cuda.synchronize()
                best = min(best, time.perf_counter() - t)
            return best
        announce(f"noalloc {rows} x {channels} at {N}^2")
        ref, plan = image(max_batch_slabs=1)
        got, plan_n = image(noalloc=True)
        assert plan["num_slabs"] >= slabs and plan_n["num_slabs"] == plan["num_slabs"]
        assert np.isfinite(got).all()
        assert_parity(got, ref, "noalloc vs allocating", whole=1e-5, central=1e-6)
        a, b = seconds(max_batch_slabs=1), seconds(noalloc=True)
        print(f"allocating {a * 1e3:.2f} ms, no-allocation {b * 1e3:.2f} ms, {plan['num_slabs']} slabs", flush=True)
        assert b <= 2.0 * a
