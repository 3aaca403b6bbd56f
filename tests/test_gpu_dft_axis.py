"""The time-transform node (hfx_dft_axis) on the matrix cores: every input type, lengths around the
folding's edges (1, 2, odd, even, more pairs than a batch of steps, the table's limit and past it),
bin ranges around the 16-bin tiles and their passes, inner sizes that are and are not multiples of
the four columns of a lane, and misaligned tensors, against an FP64 DFT.  FP32 bar: 1e-5 (sums of up
to 4096 FP32 products with twiddles rounded once)."""
import numpy as np
import pytest
import torch

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


def _input(kind, shape, seed):
    g = torch.Generator().manual_seed(seed)
    if kind == "u16":
        return torch.randint(0, 1 << 16, shape, generator=g, dtype=torch.int32).to(torch.uint16)
    if kind == "f32":
        return torch.randn(shape, generator=g)
    return torch.complex(torch.randn(shape, generator=g), torch.randn(shape, generator=g))


@pytest.mark.parametrize("kind", ["u16", "f32", "cf32"])
@pytest.mark.parametrize("outer,n,inner,kb,ke", [
    (1, 1, 5, 0, 1), (2, 2, 4, 0, 2), (3, 3, 64, 0, 3), (1, 8, 257, 1, 6), (2, 9, 100, 0, 9), (1, 33, 68, 2, 18),
    (1, 34, 1, 0, 34), (5, 64, 1, 0, 33), (2, 64, 260, 0, 33), (1, 100, 36, 17, 66), (1, 127, 12, 0, 127),
    (1, 128, 64, 0, 65), (1, 1000, 8, 490, 510), (1, 4096, 4, 2040, 2060), (1, 4100, 4, 3, 9)])
def test_dft_axis_vs_fp64(gpu, kind, outer, n, inner, kb, ke):
    from holoflow_amd import hfx

    x = _input(kind, (outer, n, inner), n + inner)
    wide = x.to(torch.complex128 if kind == "cf32" else torch.float64) if kind != "u16" else \
        torch.from_numpy(x.numpy().astype(np.float64))
    ref = torch.fft.fft(wide, dim=1)[:, kb:ke].numpy() * 0.5
    got = hfx.dft_axis(x.cuda(), 1, kb, ke, scale=0.5).cpu().numpy()
    assert rel_l2(got, ref) < 1e-5


def test_dft_axis_misaligned_input(gpu):
    from holoflow_amd import hfx

    buf = torch.randn(40 * 64 + 1, device="cuda")
    x = buf[1:].view(40, 64)  # contiguous, 4 bytes off a 16-byte boundary
    assert x.data_ptr() % 16 == 4
    ref = torch.fft.fft(x.double(), dim=0)[:21].cpu().numpy()
    assert rel_l2(hfx.dft_axis(x, 0, 0, 21).cpu().numpy(), ref) < 1e-5


@pytest.mark.parametrize("kind", ["f32", "cf32"])
@pytest.mark.parametrize("n,j", [(12, 0), (12, 6), (13, 5), (64, 63)])
def test_dft_axis_infinite_sample_stays_in_its_column(gpu, kind, n, j):
    from holoflow_amd import hfx

    x = _input(kind, (n, 70), n)
    ref = hfx.dft_axis(x.cuda(), 0).cpu()
    bad = x.clone()
    bad[j, 17] = float("inf")
    got = hfx.dft_axis(bad.cuda(), 0).cpu()
    keep = torch.arange(70) != 17
    assert torch.equal(torch.view_as_real(got[:, keep]), torch.view_as_real(ref[:, keep]))
    assert not torch.isfinite(torch.view_as_real(got[:, 17])).all(dim=-1).any()


@pytest.mark.parametrize("kind", ["f32", "cf32"])
@pytest.mark.parametrize("n", [9, 12, 13, 33, 64, 127])
def test_dft_axis_samples_near_the_largest_float(gpu, kind, n):
    """Two samples of a folded pair whose sum or difference is beyond the float range, in results that
    are not: each product and sum rounds by half an ulp of at most sqrt(2) |x|, as does each twiddle."""
    from holoflow_amd import hfx

    big = 3.0e38
    x = torch.zeros((n, 6), dtype=torch.complex64 if kind == "cf32" else torch.float32)
    for c, (p, q, a, b) in enumerate([(1, n - 1, 1, 1), (1, n - 1, 1, -1), (2, n - 2, -1, -1), (n // 2, n - n // 2, 1, 1),
                                      (4, n - 4, 1, 1), (4, n - 4, -1, 1)]):
        x[p, c], x[q, c] = a * big, b * big
        if kind == "cf32":
            x[p, c] *= 1j
    got = hfx.dft_axis(x.cuda(), 0, scale=0.25).cpu().to(torch.complex128)
    ref = torch.fft.fft(x.to(torch.complex128), dim=0) * 0.25
    assert bool(torch.isfinite(torch.view_as_real(got)).all())
    assert bool(((got - ref).abs() <= 6 * 2.0**-23 * 0.25 * 2 * big).all())
