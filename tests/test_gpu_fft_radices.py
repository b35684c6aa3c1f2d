"""The mixed-radix FFT passes (svdi_fft2_inverse at lengths without a kernel of their own) against
torch's complex128 transform: lengths of one stage (2 .. 16, each radix) and of two to four, with
every radix first, in the middle and last; the longest (8190, 8192); more rows than a workgroup takes
and a partial last tile; windows of one column, of a part of a strip and of the whole plane.

Bound: 2e-6 of the largest output, as for the other lengths (FP32 rounding of an FFT).
"""
import pytest
import torch

from conftest import announce
import svdimager_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,P,lo,count", [(g, 3, 0, g) for g in range(2, 17)] + [
    (22, 5, 3, 1), (26, 2, 0, 25), (77, 3, 10, 61), (143, 2, 0, 143), (169, 1, 1, 167), (182, 3, 30, 122), (210, 4, 35, 140),
    (360, 2, 60, 239), (1001, 1, 100, 801), (1331, 1, 0, 1331), (1848, 2, 308, 1232), (2197, 1, 500, 3), (2205, 1, 367, 1471),
    (3024, 1, 504, 2016), (4096, 1, 683, 2730), (6561, 1, 1000, 130), (8190, 1, 0, 66), (8192, 1, 4000, 65)])
def test_mixed_radix_passes(gpu_ctx, G, P, lo, count):
    announce(f"fft radices G={G} P={P} window={lo}+{count}")
    gen = torch.Generator(device="cuda").manual_seed(G)
    planes = torch.complex(torch.randn(P, G, G, device="cuda", generator=gen),
                           torch.randn(P, G, G, device="cuda", generator=gen)).contiguous()
    rows = min(count, G - lo)
    ours = S.fft2_inverse(gpu_ctx, planes, lo, rows, lo, rows)
    torch.cuda.synchronize()
    for p in range(P):
        ref = torch.fft.ifft2(planes[p].to(torch.complex128), norm="forward")
        scale = float(ref.abs().max())
        err = float((ours[p].to(torch.complex128) - ref[lo:lo + rows, lo:lo + rows]).abs().max()) / scale
        assert err <= 2e-6, (p, err)
