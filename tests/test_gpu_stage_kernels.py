"""The optional stages' kernels at the edges of their tiles and dispatches: the spatial Flatfield's
32- and 16-row tiles, radii one to thirty-one that differ between the axes, sizes that do not fill
a tile; Filter2D inside the plan behind every front (fused FP32, fused two-sided with several plane
groups, 16-bit, stand-alone time DFT) and at the lengths of its combined row pass.  FP32 bar of the
path: relative L2 <= 1e-5 against FP64 (16-bit time DFT: its own bar of 1e-3)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from oracle import stages as OS
from tests.conftest import rel_l2
from tests.test_gpu_stages import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 1, 7), (3, 33, 70), (2, 16, 64), (3, 37, 129), (9, 512, 300), (40, 100, 260)])
@pytest.mark.parametrize("sy,sx", [(0.3, 0.3), (1.0, 10.3), (10.3, 0.4), (3.0, 3.3), (8.9, 9.6)])
def test_flatfield_tiles(gpu, shape, sy, sx):
    if OS.flatfield_uses_fft(shape[1], shape[2], sy, sx):
        pytest.fail("the case is meant for the spatial form")
    rng = np.random.default_rng(shape[1] + int(10 * sx))
    x = (rng.standard_normal(shape) + 2.0).astype(np.float32)
    out = _run("Flatfield", {"sigma_y": sy, "sigma_x": sx}, torch.from_numpy(x).cuda())
    assert rel_l2(out, OS.flatfield(x, sy, sx)) < 1e-5


@pytest.mark.parametrize("H,W,T,kb,ke,kw,tol", [
    (48, 512, 32, 6, 13, {}, 1e-5), (256, 768, 64, 3, 15, {}, 1e-5), (16, 1024, 64, 2, 16, {"both_sidebands": True}, 1e-5),
    (32, 512, 64, 3, 9, {"precision": "fp16"}, 1e-3), (24, 96, 64, 1, 30, {}, 1e-5), (128, 32, 36, 3, 9, {}, 1e-5),
    (16, 2048, 32, 3, 9, {}, 1e-5), (2048, 16, 32, 3, 9, {}, 1e-5), (8, 4, 32, 3, 9, {}, 1e-5)])
def test_filter2d_in_the_plan(gpu, H, W, T, kb, ke, kw, tol):
    from holoflow_amd import hfx

    filt = (1, max(2, min(H, W) // 3), 1, 2)
    p = O.PathParams(H, W, T, T // 4, kb, ke, "fresnel", 852e-9, 12e-6, 12e-6, 0.3, fftshift=True, filt=filt,
                     both_sidebands=kw.get("both_sidebands", False))
    g = torch.Generator(device="cuda").manual_seed(H + W)
    ring = torch.randint(0, 4096, (T + 6, H, W), dtype=torch.int16, device="cuda", generator=g)
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, T // 4, kb, ke, "fresnel", p.lambda_m, p.dx_m, p.dy_m, p.z_m,
                                           fftshift=True, filt=filt, **kw))
    out = plan.moments(ring, 9)
    ref = O.doppler_moments(ring.cpu().numpy().view(np.uint16)[(9 + np.arange(T)) % (T + 6)], p, "f64")
    assert max(rel_l2(out[i].cpu().numpy(), ref[i]) for i in range(3)) < tol
    batch = plan.moments_batch(ring, 9, 3)
    assert torch.equal(batch[0], out)
