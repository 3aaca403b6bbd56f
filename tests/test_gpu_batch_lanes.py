"""Batches whose windows take several launches on two streams, and several windows of fronts whose
planes take several LDS groups: each window must equal its own hfx_moments result bit for bit.  How
many windows share a launch is read off the workspaces, so that every case has the groups it means."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ring(H, W, F):
    g = torch.Generator(device="cuda").manual_seed(H + W + F)
    return torch.randint(0, 4096, (F, H, W), dtype=torch.int16, device="cuda", generator=g)


def _plans(H, W, T, kb, ke, **kw):
    """(two-lane plan, one-lane plan, windows per launch)"""
    from holoflow_amd import hfx

    two, one = (hfx.MomentPlan(hfx.MomentConfig(H, W, T, T // 4, kb, ke, z_m=0.3, fftshift=True, batch_lanes=n, **kw))
                for n in (2, 1))
    assert (two.batch_lanes, one.batch_lanes) == (2, 1)
    sets = (two.workspace_bytes - one.workspace_bytes) / (two.n_planes * H * W * 8)
    nat = W not in (512, 768, 1024) or ke - kb > 16   # natural planes as well
    return two, one, round(sets / (2 if nat else 1))


CASES = [
    (64, 512, 64, 11, 26, {}),                               # pipelined front
    (64, 1024, 64, 11, 26, dict(prop="asm")),
    (64, 512, 64, 11, 26, dict(precision="fp16_split")),     # 16-bit front
    (96, 1024, 32, 3, 9, dict(precision="bf16", prop="asm")),
    (128, 128, 32, 6, 13, dict(prop="asm")),                 # stand-alone time DFT
    (64, 2048, 64, 11, 26, {}),
    (64, 512, 64, 11, 26, dict(batch_windows=2)),
    (64, 512, 64, 11, 26, dict(batch_windows=1)),
]


@pytest.mark.parametrize("H,W,T,kb,ke,kw", CASES)
def test_two_lanes_with_several_groups(gpu, H, W, T, kb, ke, kw):
    two, one, per = _plans(H, W, T, kb, ke, **kw)
    S, F = T // 4, T + 3 * (T // 4) + 1
    n = 2 * per + max(1, per // 2)          # three groups or more, not of one size
    assert n > 2 * per >= 2
    ring = _ring(H, W, F)
    ref = one.moments_batch(ring, F - 5, n)
    for w in (0, 1, per, n - 1):
        assert torch.equal(ref[w], one.moments(ring, (F - 5 + w * S) % F)), w
    for _ in range(3):
        assert torch.equal(two.moments_batch(ring, F - 5, n), ref)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = two.moments_batch(ring, F - 5, n)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("H,W,T,kb,ke,kw", CASES)
def test_two_lanes_under_capture(gpu, H, W, T, kb, ke, kw):
    """The fork to the plan's stream and the join become graph edges; every replay, with eager work of
    the same plan between, equals the eager batch."""
    two, one, per = _plans(H, W, T, kb, ke, **kw)
    S, F = T // 4, T + 3 * (T // 4) + 1
    n = 2 * per + 1
    ring = _ring(H, W, F)
    ref = one.moments_batch(ring, 3, n)
    out = torch.empty_like(ref)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        two.moments_batch(ring, 3, n, out)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        two.moments_batch(ring, 3, n, out)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
        assert torch.equal(two.moments(ring, (3 + S) % F), ref[1])


@pytest.mark.parametrize("H,W,T,kb,ke,prec", [
    (64, 1024, 64, 3, 14, "fp32"), (64, 1024, 48, 3, 14, "fp32"), (64, 1024, 64, 3, 14, "bf16"),   # 22 planes, two groups
    (96, 768, 128, 2, 14, "fp32"), (96, 768, 32, 0, 11, "fp32"), (24, 1024, 32, 1, 16, "fp32")])
@pytest.mark.parametrize("prop", ["fresnel", "asm"])
def test_windows_of_two_sided_fronts_with_several_groups(gpu, H, W, T, kb, ke, prec, prop):
    from holoflow_amd import hfx

    S, F, n = T // 4, T + 3 * (T // 4) + 1, 12
    cfg = lambda lanes: hfx.MomentConfig(H, W, T, S, kb, ke, prop, z_m=0.3, fftshift=True, both_sidebands=True,  # noqa: E731
                                         precision=prec, batch_lanes=lanes)
    plan = hfx.MomentPlan(cfg(2))
    per = (plan.workspace_bytes - hfx.MomentPlan(cfg(1)).workspace_bytes) // (plan.n_planes * H * W * 8)
    assert per >= 2 and per * H > 256        # more rows per launch than CUs: a block walks into the next window
    assert plan.n_planes > (20 if W == 768 else 15)
    ring = _ring(H, W, F)
    batch = plan.moments_batch(ring, F - 7, n)
    for w in range(n):
        assert torch.equal(batch[w], plan.moments(ring, (F - 7 + w * S) % F)), w


@pytest.mark.parametrize("H,W,T,kb,ke,kw", [
    (48, 512, 32, 6, 13, {}), (16, 1024, 64, 2, 16, {"both_sidebands": True}), (32, 512, 64, 3, 9, {"precision": "fp16"}),
    (24, 96, 64, 1, 30, {}), (128, 32, 36, 3, 9, {}), (16, 2048, 32, 3, 9, {})])
def test_every_window_of_a_batch_with_filter2d(gpu, H, W, T, kb, ke, kw):
    from holoflow_amd import hfx

    S, F = T // 4, T + 6
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, S, kb, ke, z_m=0.3, fftshift=True,
                                           filt=(1, max(2, min(H, W) // 3), 1, 2), **kw))
    ring = _ring(H, W, F)
    batch = plan.moments_batch(ring, 9 % F, 37)
    for w in range(37):
        assert torch.equal(batch[w], plan.moments(ring, (9 + w * S) % F)), w
