"""The folded FP32 time DFT for windows that are no multiple of 32: last batches of one to four
steps, last steps with one to three zero-weight pairs, the shortest windows with more than eight
bins, the longest that runs folded and the next one that does not, one to four bin tiles, DC and the
T/2 bin in the band, a ring that wraps inside the window.  FP32 bar of the path: relative L2 <= 1e-5
against FP64."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,kb,ke,both", [(8, 0, 8, True), (16, 0, 9, False), (20, 1, 11, False), (28, 2, 14, False),
                                          (36, 0, 19, False), (40, 1, 10, False), (44, 0, 23, False),
                                          (48, 3, 14, False), (52, 0, 27, False), (68, 1, 34, False),
                                          (100, 3, 51, False), (132, 1, 62, False), (252, 100, 127, False),
                                          (260, 4, 20, False), (48, 2, 26, True)])
@pytest.mark.parametrize("H,W,prop", [(24, 48, "asm"), (96, 256, "fresnel")])
def test_fold_any_window_vs_fp64(gpu, H, W, prop, T, kb, ke, both):
    from holoflow_amd import hfx

    p = O.PathParams(H, W, T, 4, kb, ke, prop, 852e-9, 12e-6, 12e-6, 0.1, fftshift=True, both_sidebands=both)
    F = T + 3
    g = torch.Generator(device="cuda").manual_seed(T + W)
    ring = torch.randint(0, 65536, (F, H, W), dtype=torch.int32, device="cuda", generator=g).to(torch.uint16).view(torch.int16)
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, 4, kb, ke, prop, p.lambda_m, p.dx_m, p.dy_m, p.z_m,
                                           fftshift=True, both_sidebands=both))
    got = plan.moments(ring, F - 5)
    win = ring.cpu().numpy().view(np.uint16)[(F - 5 + np.arange(T)) % F]
    ref = O.doppler_moments(win, p, "f64")
    assert max(rel_l2(got[i].cpu().numpy(), ref[i]) for i in range(3)) < 1e-5
