"""hfx_moments_batch puts several small windows into one launch of every kernel: each window must
equal its own hfx_moments result bit for bit, for every front (stand-alone interleaved and folded
time DFT, fused FP32 and 16-bit), both propagations and the optional stages, with window counts
that do not divide into the launches, windows that wrap around the ring's end, and images that lie
apart in the output."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,T,kb,ke,n,kw", [
    (64, 64, 32, 6, 13, 37, {}),                                       # interleaved DFT, 32 + 5 -> 19 + 18
    (24, 96, 64, 1, 30, 70, dict(prop="asm", split_bin=9)),            # folded DFT, three groups
    (4, 24, 36, 3, 9, 33, {}),                                         # ragged tile, ragged window length
    (32, 512, 32, 6, 13, 40, dict(prop="asm")),                        # pipelined front, fewer rows than CUs
    (48, 512, 48, 6, 18, 9, {}),                                       # fused front, not pipelined
    (64, 768, 64, 3, 9, 11, dict(precision="fp16_split")),             # 16-bit fused front
    (16, 512, 64, 2, 16, 13, dict(both_sidebands=True, precision="bf16")),  # several LDS groups of planes
    (48, 64, 32, 5, 14, 21, dict(prop="asm", pad=(64, 96), filt=(4, 20, 2, 6))),
    (64, 96, 64, 11, 26, 18, dict(filt=(3, 20, 2, 4), flatfield=(2.0, 1.5))),
    (256, 256, 64, 11, 26, 5, dict(prop="asm")),                       # two windows per launch
])
def test_small_windows_of_a_batch_equal_single_windows(gpu, H, W, T, kb, ke, n, kw):
    from holoflow_amd import hfx
    from holoflow_amd._lib import check, lib

    S = T // 4 + 1
    F = T + 3 * S + 2
    g = torch.Generator(device="cuda").manual_seed(H + W + n)
    ring = torch.randint(0, 4096, (F, H, W), dtype=torch.int16, device="cuda", generator=g)
    plan = hfx.MomentPlan(hfx.MomentConfig(H, W, T, S, kb, ke, z_m=0.2, fftshift=True, **kw))
    first = F - 3
    ref = [plan.moments(ring, (first + w * S) % F) for w in range(n)]
    per = ref[0].numel()
    out = torch.full((n, per + 5), -1.0, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for _ in range(2):
        check(lib().hfx_moments_batch(plan._h, C.c_void_p(ring.data_ptr()), F, first, n, per + 5,
                                      C.c_void_p(out.data_ptr()), C.c_void_p(stream)))
    for w in range(n):
        assert torch.equal(out[w, :per].view_as(ref[w]), ref[w]), f"window {w}"
    assert bool((out[:, per:] == -1.0).all())
