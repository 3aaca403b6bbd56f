"""Plane workspaces of a plan by its batch_windows: one window per launch holds one window's planes per
lane, a count holds that many, and the windows of a batch are the same whatever the count."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# fused front (blocked planes only); stand-alone time DFT and padding (natural planes as well);
# two-sided planes in several groups; 16-bit front
@pytest.mark.parametrize("H,W,T,kb,ke,kw,nat", [
    (64, 512, 64, 11, 26, {}, False), (128, 128, 32, 6, 13, dict(prop="asm"), True),
    (48, 64, 32, 5, 14, dict(prop="asm", pad=(64, 96)), True), (64, 1024, 64, 3, 14, dict(both_sidebands=True), False),
    (64, 768, 64, 3, 9, dict(precision="fp16_split"), False)])
@pytest.mark.parametrize("lanes", [1, 2])
def test_workspace_follows_batch_windows(gpu, H, W, T, kb, ke, kw, nat, lanes):
    from holoflow_amd import hfx

    S = T // 4
    F = T + 5 * S + 1
    g = torch.Generator(device="cuda").manual_seed(H + W)
    ring = torch.randint(0, 4096, (F, H, W), dtype=torch.int16, device="cuda", generator=g)
    plans = {n: hfx.MomentPlan(hfx.MomentConfig(H, W, T, S, kb, ke, z_m=0.2, fftshift=True, batch_windows=n, batch_lanes=lanes,
                                                **kw)) for n in (0, 1, 2, 3)}
    oh, ow = plans[1].out_shape[1:]
    per = plans[1].n_planes * 8 * (oh * ow + (H * W if nat else 0)) * lanes  # one window's planes
    held = {n: p.workspace_bytes for n, p in plans.items()}
    assert held[2] - held[1] == per and held[3] - held[1] == 2 * per
    windows = min(32, (64 << 20) // (plans[1].n_planes * 8 * max(oh * ow, H * W)))
    assert windows > 3 and held[0] - held[1] == (windows - 1) * per
    ref = [plans[1].moments(ring, (F - 3 + w * S) % F) for w in range(7)]
    for n, p in plans.items():
        out = p.moments_batch(ring, F - 3, 7)
        for w in range(7):
            assert torch.equal(out[w], ref[w]), (n, w)


def test_default_is_the_librarys_choice(gpu):
    from holoflow_amd import hfx

    size = lambda **kw: hfx.MomentPlan(hfx.MomentConfig(128, 128, 32, 8, 6, 13, **kw)).workspace_bytes  # noqa: E731
    assert size() == size(batch_windows=0) > size(batch_windows=4) > size(batch_windows=1) == size(batch_windows=-1)
