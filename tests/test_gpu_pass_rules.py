"""The launch rules of the column and row passes at the edges of their ranges: 1024-row columns with a
transfer function in blocks of four waves and of eight, moment rows with the planes of a row over
several waves and one wave per row, 2048-row moment columns."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


def _case(H, W, T, kb, ke, prop, frames=0, **kw):
    from holoflow_amd import hfx

    F = T + frames + 3
    g = torch.Generator(device="cuda").manual_seed(H + W + ke)
    ring = torch.randint(0, 4096, (F, H, W), dtype=torch.int16, device="cuda", generator=g)
    p = O.PathParams(H, W, T, T // 4, kb, ke, prop, 852e-9, 12e-6, 12e-6, 0.4, fftshift=True, split_bin=kw.get("split_bin", 0))
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, T // 4, kb, ke, prop, p.lambda_m, p.dx_m, p.dy_m, p.z_m, fftshift=True, **kw))
    return ring, p, plan


def _check(ring, p, plan, first):
    out = plan.moments(ring, first)
    win = ring.cpu().numpy().view(np.uint16)[(first + np.arange(p.window)) % ring.shape[0]]
    ref = O.doppler_moments(win, p, "f64")
    # the FP32 bar of the path: relative L2 against FP64
    assert max(rel_l2(out[i].cpu().numpy(), ref[i]) for i in range(out.shape[0])) < 1e-5
    return out


# blocks of four waves: W / 4 x planes
@pytest.mark.parametrize("W,planes", [(4, 1), (8, 5), (128, 8), (128, 9), (512, 4), (512, 5), (768, 4), (256, 13)])
def test_transfer_function_columns_of_1024_rows(gpu, W, planes):
    _check(*_case(1024, W, 64, 6, 6 + planes, "asm"), 5)


@pytest.mark.parametrize("H,W,planes", [(2048, 16, 5), (2048, 24, 9)])
@pytest.mark.parametrize("split", [0, 8])
def test_moment_columns_of_2048_rows(gpu, H, W, planes, split):
    ring, p, plan = _case(H, W, 64, 6, 6 + planes, "fresnel", split_bin=split)
    assert _check(ring, p, plan, 4).shape[0] == (5 if split else 3)


# items (W / 8 x planes) around five per CU, where the blocks start to stay
@pytest.mark.parametrize("W,planes", [(1024, 9), (1024, 10), (1024, 11), (512, 21)])
def test_transfer_function_columns_of_2048_rows(gpu, W, planes):
    ring, p, plan = _case(2048, W, 64, 1, 1 + planes, "asm", frames=16)
    out = _check(ring, p, plan, 2)
    assert torch.equal(plan.moments_batch(ring, 2, 2)[0], out)


# a batch of windows has rows enough for one wave each: the sums must be those of a single window
@pytest.mark.parametrize("H,W", [(512, 256), (512, 768), (768, 512), (768, 768)])
@pytest.mark.parametrize("planes", [1, 2, 3, 4, 5, 7, 8])
def test_moment_rows_do_not_depend_on_the_launch(gpu, H, W, planes):
    for split in (0, 7) if planes > 1 else (0,):
        ring, p, plan = _case(H, W, 32, 6, 6 + planes, "asm", frames=16, split_bin=split)
        F = ring.shape[0]
        batch = plan.moments_batch(ring, 2, 3)
        for w in range(3):
            assert torch.equal(batch[w], plan.moments(ring, (2 + 8 * w) % F)), (split, w)


# 512-point rows at T = 64: four consumer waves from 1024 rows on, eight below; the folded and the
# interleaved DFT, one band and two
@pytest.mark.parametrize("H", [768, 1024, 2048])
@pytest.mark.parametrize("kb,ke,both", [(8, 15, False), (8, 17, False), (8, 24, False), (8, 23, True)])
def test_front_of_512_point_rows(gpu, H, kb, ke, both):
    from holoflow_amd import hfx

    g = torch.Generator(device="cuda").manual_seed(H + ke)
    ring = torch.randint(0, 4096, (64 + 35, H, 512), dtype=torch.int16, device="cuda", generator=g)
    p = O.PathParams(H, 512, 64, 16, kb, ke, "fresnel", 852e-9, 12e-6, 12e-6, 0.4, fftshift=True, both_sidebands=both)
    plan = hfx.MomentPlan(hfx.MomentConfig(H, 512, 64, 16, kb, ke, "fresnel", p.lambda_m, p.dx_m, p.dy_m, p.z_m, fftshift=True,
                                           both_sidebands=both, batch_windows=2))
    out = _check(ring, p, plan, 5)
    batch = plan.moments_batch(ring, 5, 2)
    assert torch.equal(batch[0], out) and torch.equal(batch[1], plan.moments(ring, 21))


# 768- and 1024-point rows at T = 32: frames of 1024 rows and more take a form of their own
@pytest.mark.parametrize("H", [768, 1024, 2048])
@pytest.mark.parametrize("W", [768, 1024])
@pytest.mark.parametrize("kb,ke", [(1, 10), (1, 17)])
def test_front_of_short_windows(gpu, H, W, kb, ke):
    ring, p, plan = _case(H, W, 32, kb, ke, "fresnel", frames=8, batch_windows=2)
    out = _check(ring, p, plan, 5)
    batch = plan.moments_batch(ring, 5, 2)
    assert torch.equal(batch[0], out) and torch.equal(batch[1], plan.moments(ring, 13))
