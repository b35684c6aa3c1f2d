"""The mixed-radix FFT passes at lengths whose transforms leave room for one workgroup to a CU, which takes
1024 threads then (svdi_fft2_inverse), against torch's complex128 transform: two columns a workgroup and one,
a window that ends within a strip, the plane's corner.

Bound: 2e-6 of the largest output, as for the other lengths (FP32 rounding of an FFT)."""
import pytest
import torch

from conftest import announce
import svdimager_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G", [2500, 5000, 6561, 7000])
def test_one_workgroup_to_a_cu(gpu_ctx, G):
    gen = torch.Generator(device="cuda").manual_seed(G)
    planes = torch.complex(torch.randn(1, G, G, device="cuda", generator=gen),
                           torch.randn(1, G, G, device="cuda", generator=gen)).contiguous()
    ref = torch.fft.ifft2(planes[0].to(torch.complex128), norm="forward")
    scale = float(ref.abs().max())
    for row_lo, rows, col_lo, cols in [(G // 6, G // 3, G // 6 + 1, 131), (G - 9, 9, G - 5, 5)]:
        announce(f"fft threads G={G} rows {row_lo}+{rows} cols {col_lo}+{cols}")
        ours = S.fft2_inverse(gpu_ctx, planes, row_lo, rows, col_lo, cols)
        torch.cuda.synchronize()
        err = float((ours[0].to(torch.complex128) - ref[row_lo:row_lo + rows, col_lo:col_lo + cols]).abs().max()) / scale
        assert err <= 2e-6, err
