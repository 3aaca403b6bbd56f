"""GPU parity of the short row and column passes (several transforms per wave, 2..128 points) at
the sizes where the wave split can go wrong: rows or columns that do not fill a wave, one lane per
transform, widths whose column block is narrower than four, fewer and more planes than the eight
plane subsets of the moment kinds.  FP32 bar of the path: relative L2 <= 1e-5 against FP64."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("H,W", [(2, 2), (4, 2), (2, 8), (8, 4), (16, 24), (24, 16), (48, 32), (32, 96), (96, 48),
                                 (128, 64), (64, 128), (128, 2), (4, 256)])
@pytest.mark.parametrize("prop", ["asm", "fresnel"])
def test_short_transform_nodes_vs_fp64(gpu, H, W, prop):
    from holoflow_amd import hfx

    g = torch.Generator().manual_seed(H * 1000 + W)
    x = torch.complex(torch.randn(3, H, W, generator=g), torch.randn(3, H, W, generator=g))
    p = O.PathParams(H, W, 32, 8, 1, 4, prop, 852e-9, 12e-6, 12e-6, 0.05)
    if prop == "asm":
        got = hfx.AngularSpectrum(3, H, W, p.lambda_m, p.dx_m, p.dy_m, p.z_m)(x.cuda())
        ref = O.angular_spectrum(x, p)
    else:
        got = hfx.Fresnel(3, H, W, p.lambda_m, p.dx_m, p.dy_m, p.z_m)(x.cuda())
        ref = O.fresnel(x, p, output_magnitude=False)
    assert rel_l2(got.cpu().numpy(), ref.numpy()) < TOL


@pytest.mark.parametrize("H,W", [(4, 24), (24, 8), (16, 32), (32, 16), (48, 96), (96, 64), (128, 48), (64, 128)])
@pytest.mark.parametrize("nb,split", [(1, 0), (7, 2), (19, 11)])
@pytest.mark.parametrize("prop", ["asm", "fresnel"])
def test_short_moment_passes_vs_fp64(gpu, H, W, nb, split, prop):
    from holoflow_amd import hfx

    T = 64
    p = O.PathParams(H, W, T, 16, 3, 3 + nb, prop, 852e-9, 12e-6, 12e-6, 0.1, fftshift=True,
                     split_bin=3 + split if split else 0)
    d = hfx.synth_desc(H, W, disk_radius_px=0.39 * min(H, W), seed=H + W)
    ring, _ = hfx.synth_frames(d, 0, T)
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, 16, p.bin_begin, p.bin_end, prop, p.lambda_m, p.dx_m, p.dy_m,
                                           p.z_m, fftshift=True, split_bin=p.split_bin))
    got = plan.moments(ring, 0).cpu().numpy()
    ref = O.doppler_moments(ring.cpu().numpy().view(np.uint16), p, "f64")
    assert got.shape == ref.shape
    assert max(rel_l2(got[i], ref[i]) for i in range(ref.shape[0])) < TOL
