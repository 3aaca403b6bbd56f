"""The pipelined FP32 front with a two-sided band whose planes take several LDS groups, at rows
enough that each workgroup walks more than one (so that the groups of one row, the next row's
time DFT and the row after it interleave), for every window length it is compiled for, the DC bin
in the band, plane counts that split unevenly, and several windows in one launch.  FP32 bar of the
path: relative L2 <= 1e-5 against FP64."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,T,kb,ke,prop", [(512, 1024, 64, 11, 26, "fresnel"), (768, 1024, 32, 0, 8, "asm"),
                                              (256, 1024, 128, 3, 14, "asm"), (768, 768, 64, 2, 13, "fresnel"),
                                              (512, 768, 128, 40, 55, "asm"), (256, 768, 32, 1, 12, "fresnel")])
def test_two_sided_front_vs_fp64(gpu, H, W, T, kb, ke, prop):
    from holoflow_amd import hfx

    p = O.PathParams(H, W, T, T // 4, kb, ke, prop, 852e-9, 12e-6, 12e-6, 0.4, fftshift=True, both_sidebands=True)
    F = T + T // 4
    g = torch.Generator(device="cuda").manual_seed(W + T + kb)
    ring = torch.randint(0, 4096, (F, H, W), dtype=torch.int16, device="cuda", generator=g)
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, T // 4, kb, ke, prop, p.lambda_m, p.dx_m, p.dy_m, p.z_m,
                                           fftshift=True, both_sidebands=True, batch_windows=2))
    first = F - 5
    got = plan.moments(ring, first)
    batch = plan.moments_batch(ring, first, 3)
    assert torch.equal(batch[0], got)
    assert torch.equal(batch[1], plan.moments(ring, (first + T // 4) % F))
    win = ring.cpu().numpy().view(np.uint16)[(first + np.arange(T)) % F]
    ref = O.doppler_moments(win, p, "f64")
    assert max(rel_l2(got[i].cpu().numpy(), ref[i]) for i in range(3)) < 1e-5
