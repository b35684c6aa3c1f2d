"""svdi_fft2_inverse at lengths with a prime factor above 13: those transformed by a convolution of
length 2^m >= 2 G - 1, at both sides of its powers of two and of the range's ends (G = 38 and 4097
are direct DFTs), over the central window and one at the plane's far corner.  Reference:
torch.fft.ifft2 in complex128.

Bound: max |ours - ref| <= 2e-6 of max |ref|: 2 log2(8192) + 3 = 29 roundings of 2^-24 on the way of
a value, 1.7e-6 if all went one way.
"""
import pytest
import torch

from conftest import announce
import svdimager_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,P", [(51, 3), (38, 3), (53, 2), (453, 5), (511, 2), (513, 2), (1023, 2), (2047, 1),
                                 (2049, 1), (4081, 1), (4097, 1)])
def test_lengths(gpu_ctx, G, P):
    gen = torch.Generator(device="cuda").manual_seed(G)
    planes = torch.complex(torch.randn(P, G, G, device="cuda", generator=gen),
                           torch.randn(P, G, G, device="cuda", generator=gen)).contiguous()
    ref = torch.fft.ifft2(planes.to(torch.complex128), norm="forward")
    scale = float(ref.abs().max())
    N = (2 * G) // 3
    lo = G // 2 - N // 2
    for row_lo, rows, col_lo, cols in [(lo, N, lo, N), (0, G, 0, G), (G - 5, 5, G - 3, 3)]:
        announce(f"fft2_inverse G={G} P={P} rows {row_lo}+{rows} cols {col_lo}+{cols}")
        ours = S.fft2_inverse(gpu_ctx, planes, row_lo, rows, col_lo, cols)
        want = ref[:, row_lo:row_lo + rows, col_lo:col_lo + cols]
        assert float((ours.to(torch.complex128) - want).abs().max()) <= 2e-6 * scale
