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
