"""The 2048-row column pass of the angular spectrum over a persistent grid: fewer items than the
rule asks for, the smallest launch that loops, items that do not divide evenly over the blocks, planes
of several windows in one launch.
FP32 bar of the path: relative L2 <= 1e-5 against FP64."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,nb", [(8, 1), (1024, 7), (1024, 8), (1024, 9), (512, 17), (768, 13), (256, 32),
                                  (2048, 5)])
def test_long_columns_vs_fp64(gpu, W, nb):
    from holoflow_amd import hfx

    H, T = 2048, 64
    p = O.PathParams(H, W, T, 8, 1, 1 + nb, "asm", 852e-9, 12e-6, 12e-6, 0.3)
    g = torch.Generator(device="cuda").manual_seed(W + nb)
    ring = torch.randint(0, 4096, (T + 8, H, W), dtype=torch.int16, device="cuda", generator=g)
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, 8, 1, 1 + nb, "asm", p.lambda_m, p.dx_m, p.dy_m, p.z_m))
    got = plan.moments(ring, 0)
    ref = O.doppler_moments(ring[:T].cpu().numpy().view(np.uint16), p, "f64")
    assert max(rel_l2(got[i].cpu().numpy(), ref[i]) for i in range(3)) < 1e-5
    batch = plan.moments_batch(ring, 0, 2)
    assert torch.equal(batch[0], got)
    assert torch.equal(batch[1], plan.moments(ring, 8))
