"""Angular spectrum with zero padding: the row pass runs the input's rows only and the column pass
takes the others as zeros.  Padding of both axes, of one axis, of a single row or column on each
side, real and complex inputs, every case twice so that the workspace holds the previous result
where nothing is written.  FP32 bar of the path: relative L2 <= 1e-5 against FP64."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-5
SHAPES = [(2, 4, 4, 8), (22, 64, 24, 64), (24, 60, 24, 64), (94, 60, 96, 256), (6, 500, 512, 512),
          (512, 8, 512, 1024), (1022, 44, 1024, 48), (300, 764, 768, 768), (20, 1024, 2048, 1024),
          (24, 1000, 32, 2048)]


@pytest.mark.parametrize("H,W,OH,OW", SHAPES)
@pytest.mark.parametrize("real", [False, True])
def test_padded_node_vs_fp64(gpu, H, W, OH, OW, real):
    from holoflow_amd import hfx

    g = torch.Generator().manual_seed(H * 1000 + W)
    node = hfx.AngularSpectrum(3, H, W, 852e-9, 12e-6, 12e-6, 0.3, in_real=real, pad=(OH, OW))
    p = O.PathParams(H, W, 4, 4, 0, 1, "asm", 852e-9, 12e-6, 12e-6, 0.3, pad=(OH, OW))
    for _ in range(2):
        x = torch.randn(3, H, W, generator=g)
        if not real:
            x = torch.complex(x, torch.randn(3, H, W, generator=g))
        got = node(x.cuda())
        ref = O.angular_spectrum(x.to(torch.complex64), p)
        assert rel_l2(got.cpu().numpy(), ref.numpy()) < TOL


@pytest.mark.parametrize("H,W,OH,OW", SHAPES)
def test_padded_plan_vs_fp64(gpu, H, W, OH, OW):
    from holoflow_amd import hfx

    T = 32
    p = O.PathParams(H, W, T, T, 2, 6, "asm", 852e-9, 12e-6, 12e-6, 0.3, pad=(OH, OW))
    g = torch.Generator(device="cuda").manual_seed(H + W)
    ring = torch.randint(0, 4096, (3 * T, H, W), dtype=torch.int16, device="cuda", generator=g)
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, T, 2, 6, "asm", p.lambda_m, p.dx_m, p.dy_m, p.z_m, pad=(OH, OW)))
    got = [plan.moments(ring, 0)] + list(plan.moments_batch(ring, T, 2))
    frames = ring.cpu().numpy().view(np.uint16)
    for w in range(3):
        ref = O.doppler_moments(frames[w * T:(w + 1) * T], p, "f64")
        assert max(rel_l2(got[w][i].cpu().numpy(), ref[i]) for i in range(3)) < TOL
