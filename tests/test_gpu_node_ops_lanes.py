"""Node kernels whose split over lanes depends on the sizes, at the edges of those rules: data movement
bit-exact, sums within the rounding of their terms."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.complex64])
@pytest.mark.parametrize("shape,axes", [((5000, 8), (1,)), ((300, 2), (0, 1)), ((70000, 4, 4), (1, 2)), ((70000, 3, 3), (1, 2)),
                                        ((9, 5, 7), (1, 2)), ((65, 64), (0, 1)), ((3, 258), (0, 1)), ((100003,), (0,)),
                                        ((2, 2, 2), (1, 2)), ((1, 2, 12), (1, 2)), ((300000, 4), (1,)), ((4096, 16, 2), (1,))])
def test_fftshift_of_narrow_rows_and_small_images(gpu, dtype, shape, axes):
    from holoflow_amd import hfx

    n = 1
    for s in shape:
        n *= s
    x = torch.arange(n, device="cuda").to(dtype).reshape(shape)
    ref = torch.roll(x, [-(shape[a] // 2) for a in axes], axes)
    assert torch.equal(hfx.fftshift(x, axes), ref)


@pytest.mark.parametrize("planes,npix", [(1, 131072), (2, 131072), (3, 131074), (15, 262144), (16, 1000), (33, 1 << 20)])
@pytest.mark.parametrize("weighted", [False, True])
def test_mean_of_complex_planes(gpu, planes, npix, weighted):
    """Two planes in flight, eight, one pixel per lane; NaN and infinities stay in their pixels."""
    from holoflow_amd import hfx

    g = torch.Generator(device="cuda").manual_seed(planes)
    x = torch.randn((planes, npix), dtype=torch.complex64, device="cuda", generator=g)
    x[planes // 2, 5] = complex(float("nan"), 1.0)
    x[planes - 1, 9] = complex(float("inf"), 1.0)
    w = torch.rand(planes, device="cuda", generator=g) + 0.5 if weighted else None
    got = hfx.weighted_mean(x, w)
    a = x.to(torch.complex128).abs()
    ref = (a if w is None else w.double()[:, None] * a).mean(0)
    assert torch.isnan(got[5]) and torch.isinf(got[9])
    fine = torch.isfinite(ref)
    assert bool(torch.isfinite(got[fine]).all()) and int((~fine).sum()) == 2
    # each |x| within 2 ulp, the product and each of `planes` additions of positive terms within half
    assert bool(((got[fine] - ref[fine]).abs() <= (planes + 4) * 2.0**-23 * ref[fine]).all())
