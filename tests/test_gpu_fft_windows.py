"""svdi_fft2_inverse at the sizes of the wavefront passes (G = 1536, 3072, 6144) over windows that
do not fit their blocks of eight columns or their row split: ragged widths, odd first rows and
heights, one element, the plane's last rows and columns, the whole plane.  Reference:
torch.fft.ifft2 of the same complex64 planes.

Bound: max |ours - rocFFT| <= 2e-6 of max |rocFFT| over the plane (both FP32; an FFT's rounding
grows like log2(G) ulp of the output's scale).
"""
import pytest
import torch

from conftest import announce
import svdimager_amd as S

pytestmark = pytest.mark.gpu

WINDOWS = [(0, 0, 0, 0), (1, 3, 5, 9), (2, 8, 8, 8), (7, 1, 11, 1), (-5, 5, -13, 13), (256, 1001, 255, 515)]


@pytest.mark.parametrize("G,P", [(1536, 2), (3072, 2), (6144, 1)])
def test_windows(gpu_ctx, G, P):
    gen = torch.Generator(device="cuda").manual_seed(G)
    planes = torch.complex(torch.randn(P, G, G, device="cuda", generator=gen),
                           torch.randn(P, G, G, device="cuda", generator=gen)).contiguous()
    ref = torch.fft.ifft2(planes, norm="forward")
    scale = float(ref.abs().max())
    for row_lo, rows, col_lo, cols in WINDOWS:
        row_lo, col_lo, rows, cols = row_lo % G, col_lo % G, rows or G, cols or G
        announce(f"fft2_inverse G={G} P={P} rows {row_lo}+{rows} cols {col_lo}+{cols}")
        ours = S.fft2_inverse(gpu_ctx, planes, row_lo, rows, col_lo, cols)
        want = ref[:, row_lo:row_lo + rows, col_lo:col_lo + cols]
        assert float((ours - want).abs().max()) <= 2e-6 * scale
