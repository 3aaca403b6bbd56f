"""The spatial Flatfield at NaN and infinities, which reach exactly the pixels whose blur contains them,
and inside batches whose windows take several launches."""
import numpy as np
import pytest
import torch

from oracle import stages as OS
from tests.test_gpu_stages import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 40, 200), (40, 100, 260)])     # 16-row and 32-row tiles
@pytest.mark.parametrize("sy,sx", [(1.0, 1.0), (3.0, 0.3), (8.9, 10.3)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_what_is_not_finite_stays_in_its_neighbourhood(gpu, shape, sy, sx, bad):
    assert not OS.flatfield_uses_fft(shape[1], shape[2], sy, sx)
    g = torch.Generator().manual_seed(shape[2])
    x = torch.randn(shape, generator=g) + 2.0
    clean = torch.from_numpy(np.asarray(_run("Flatfield", {"sigma_y": sy, "sigma_x": sx}, x.cuda())))
    assert bool(torch.isfinite(clean).all())
    y, c = 17, 63
    z = x.clone()
    z[0, y, c] = bad
    got = torch.from_numpy(np.asarray(_run("Flatfield", {"sigma_y": sy, "sigma_x": sx}, z.cuda())))
    ry, rx = int(np.ceil(3 * sy)), int(np.ceil(3 * sx))
    hit = torch.zeros(shape, dtype=torch.bool)
    hit[0, max(0, y - ry):y + ry + 1, max(0, c - rx):c + rx + 1] = True
    assert not bool(torch.isfinite(got[hit]).any())
    assert torch.equal(got[~hit], clean[~hit])


@pytest.mark.parametrize("H,W,T,n,sigma", [(64, 96, 64, 70, 2.0), (128, 128, 32, 35, 1.0), (256, 256, 64, 7, 3.0),
                                            (64, 512, 32, 40, 9.0), (512, 512, 64, 3, 3.0), (64, 64, 32, 34, 12.0)])
@pytest.mark.parametrize("prop", ["fresnel", "asm"])
def test_flatfield_in_batches_of_several_launches(gpu, H, W, T, n, sigma, prop):
    """More windows than one launch takes (at most 32), both forms of the Flatfield (12.0: the Fourier
    one), images apart in the output."""
    import ctypes as C

    from holoflow_amd import hfx
    from holoflow_amd._lib import check, lib

    S = T // 4
    F = T + 2 * S + 1
    g = torch.Generator(device="cuda").manual_seed(H + n)
    ring = torch.randint(0, 4096, (F, H, W), dtype=torch.int16, device="cuda", generator=g)
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, S, 6, 13, prop, z_m=0.2, fftshift=True, flatfield=(sigma, sigma)))
    ref = [plan.moments(ring, (3 + w * S) % F) for w in range(n)]
    per = ref[0].numel()
    out = torch.full((n, per + 7), -5.0, device="cuda")
    check(lib().hfx_moments_batch(plan._h, C.c_void_p(ring.data_ptr()), F, 3, n, per + 7, C.c_void_p(out.data_ptr()),
                                  C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    for w in range(n):
        assert torch.equal(out[w, :per].view_as(ref[w]), ref[w]), w
    assert bool((out[:, per:] == -5.0).all())
