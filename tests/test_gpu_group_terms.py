"""A grouped planned batch (svdi_image_snapshots_planned) whose snapshots differ in their number of terms,
1 to 20 in one group: the contraction's blocks of eight terms and of sixteen take their jobs in launches of
their own.  Every image against the same planned call alone.

Tolerance: as for two summation orders of the same gridder, 1e-5 of peak over the image and 1e-6 over the
central half."""
import pytest
import torch

from conftest import announce, assert_parity, load_small_snapshot
import svdimager_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("terms", [(8, 16, 8, 20, 1, 9, 8), (16, 8), (8, 9)])
@pytest.mark.parametrize("precision", [S.PRECISION_DEFAULT, S.PRECISION_SINGLE])
def test_groups_of_mixed_terms(terms, precision):
    snap = load_small_snapshot()
    cell = snap["cell"]
    sizes = [(128, 96, 64)[i % 3] for i in range(len(terms))]
    opts = dict(output=S.OUTPUT_SIGNED, gridder=S.GRIDDER_MFMA, mfma_precision=precision)
    with S.Context(0) as ctx:
        ds, plans = [], []
        for i, (N, K) in enumerate(zip(sizes, terms)):
            d = S.DeviceSnapshot(snap, "cuda")
            for k in ("vis0_re", "vis0_im", "vis3_re", "vis3_im"):
                d.tensors[k].mul_(1.0 + 0.1 * i)
            ds.append(d)
            plans.append(S.image_snapshot(ctx, d, N, cell, num_terms=K, **opts)[1])
        assert [p["num_terms"] for p in plans] == list(terms)
        announce(f"group of terms {terms} precision {precision}")
        imgs, _ = S.image_snapshot_batch(ctx, ds, sizes, [cell] * len(sizes), plans=plans, **opts)
        torch.cuda.synchronize()
        for i, (d, N) in enumerate(zip(ds, sizes)):
            one = torch.empty((N, N), dtype=torch.float32, device="cuda")
            S.image_snapshot(ctx, d, N, cell, image=one, plan=plans[i], **opts)
            torch.cuda.synchronize()
            assert_parity(imgs[i].cpu().numpy(), one.cpu().numpy(), f"group [{i}] ({N}^2, {terms[i]} terms) vs alone",
                          whole=1e-5, central=1e-6)
