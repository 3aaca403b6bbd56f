"""The inverse moment row pass with the planes of a row split over waves (launches of few rows) at
the sizes where it can go wrong: each compiled length, row counts on both sides of the rule, rows
that do not fill the last block, plane counts around the split, the band split inside and at the
edge of a round of planes.  The sums must not depend on the launch (a window of a batch or a group
is bit-identical to the same window alone).  FP32 bar of the path: relative L2 <= 1e-5 against
FP64."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(2, 256), (96, 256), (512, 256), (24, 512), (512, 512), (768, 512), (1024, 512),
                                 (48, 768), (512, 768), (16, 1024), (512, 1024), (1024, 1024), (2, 2048), (24, 2048),
                                 (512, 2048)])
@pytest.mark.parametrize("nb,split,power2", [(1, 0, False), (3, 1, True), (4, 0, False), (7, 4, False), (9, 0, True)])
def test_moment_rows_vs_fp64(gpu, H, W, nb, split, power2):
    from holoflow_amd import hfx

    T = 32
    p = O.PathParams(H, W, T, 8, 2, 2 + nb, "asm", 852e-9, 12e-6, 12e-6, 0.3, fftshift=True, power2=power2,
                     split_bin=2 + split if split else 0)
    g = torch.Generator(device="cuda").manual_seed(H + W + nb)
    ring = torch.randint(0, 4096, (T + 24, H, W), dtype=torch.int16, device="cuda", generator=g)
    cfg = hfx.MomentConfig(H, W, T, 8, 2, 2 + nb, "asm", p.lambda_m, p.dx_m, p.dy_m, p.z_m, fftshift=True,
                           power2=power2, split_bin=p.split_bin)
    plan = hfx.MomentPlan(cfg)
    got = plan.moments(ring, 0)
    ref = O.doppler_moments(ring[:T].cpu().numpy().view(np.uint16), p, "f64")
    assert max(rel_l2(got[i].cpu().numpy(), ref[i]) for i in range(ref.shape[0])) < 1e-5
    batch = plan.moments_batch(ring, 0, 4)
    for w in range(4):
        assert torch.equal(batch[w], plan.moments(ring, 8 * w))
