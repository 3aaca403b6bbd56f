"""The element-wise node kernels take several elements per lane where size and alignment allow: each
against torch at the edges of those rules (tails, buffers a few elements off, rows whose halves
allow 16-, 8-, 4-byte or no wide copies, planes around the groups of eight).  Data movement and
integer results are bit-exact; means are FP32 sums of at most 33 planes, held to 1e-6 of FP64."""
import ctypes as C

import pytest
import torch

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.uint8, torch.int16, torch.float32, torch.complex64])
@pytest.mark.parametrize("shape,axes", [((64, 64), (0, 1)), ((3, 50, 30), (1, 2)), ((7, 12), (1,)), ((7, 12), (0,)),
                                        ((5, 6, 7), (0, 1, 2)), ((4, 6, 10), (0, 2)), ((2, 3, 16, 8), (1, 2)),
                                        ((1, 9), (0, 1)), ((130,), (0,)), ((2, 1024, 3), (1,)), ((6, 4, 8), ())])
def test_fftshift_forms(gpu, dtype, shape, axes):
    from holoflow_amd import hfx

    n = 1
    for s in shape:
        n *= s
    x = torch.arange(n, device="cuda").remainder(251).to(dtype).reshape(shape)
    ref = x
    for ax in axes:
        ref = torch.roll(ref, -(shape[ax] // 2), ax)
    assert torch.equal(hfx.fftshift(x, axes), ref)


def test_fftshift_misaligned(gpu):
    from holoflow_amd import hfx

    buf = torch.arange(64 * 64 + 1, device="cuda", dtype=torch.float32)
    x = buf[1:].view(64, 64)
    assert torch.equal(hfx.fftshift(x, (0, 1)), torch.roll(x, (-32, -32), (0, 1)))


@pytest.mark.parametrize("planes", [1, 7, 8, 9, 33])
@pytest.mark.parametrize("npix,off", [(1 << 18, 0), (1 << 18, 1), ((1 << 18) + 2, 0), (1000, 0)])
@pytest.mark.parametrize("cplx", [False, True])
def test_weighted_mean_forms(gpu, planes, npix, off, cplx):
    from holoflow_amd import hfx

    g = torch.Generator(device="cuda").manual_seed(planes + npix)
    dt = torch.complex64 if cplx else torch.float32
    x = torch.randn(planes * npix + off, dtype=dt, device="cuda", generator=g)[off:].view(planes, npix)
    w = torch.rand(planes, device="cuda", generator=g)
    a = x.to(torch.complex128 if cplx else torch.float64).abs()
    assert rel_l2(hfx.weighted_mean(x, absval=True).cpu(), a.mean(0).cpu()) < 1e-6
    assert rel_l2(hfx.weighted_mean(x, w, absval=True).cpu(), (w.double()[:, None] * a).mean(0).cpu()) < 1e-6
    assert rel_l2(hfx.weighted_mean(x, w, power2=True).cpu(), (w.double()[:, None] * a * a).mean(0).cpu()) < 1e-6


_DT = {torch.uint16: 1, torch.float32: 2, torch.complex64: 3, torch.uint8: 4}


def _convert(x, out, strategy):
    from holoflow_amd._lib import check, lib

    n = x.numel()
    scratch = torch.empty(int(lib().hfx_convert_scratch_bytes(n)), dtype=torch.uint8, device="cuda")
    check(lib().hfx_convert(C.c_void_p(x.data_ptr()), _DT[x.dtype], C.c_void_p(out.data_ptr()), _DT[out.dtype], strategy,
                            n, C.c_void_p(scratch.data_ptr()), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return out


@pytest.mark.parametrize("n", [1, 3, 4095, 4096, 4097, 12291])
@pytest.mark.parametrize("off", [0, 1])
def test_convert_forms(gpu, n, off):
    g = torch.Generator(device="cuda").manual_seed(n)
    ints = torch.randint(0, 65536, (n + off,), device="cuda", generator=g)
    for src in (ints.to(torch.uint16)[off:], ints.remainder(256).to(torch.uint8)[off:]):
        ref = src.to(torch.int32).float()
        guard = torch.full((n + 8,), -7.0, device="cuda")
        assert torch.equal(_convert(src, guard[4:4 + n], 0), ref)
        assert bool((guard[:4] == -7).all()) and bool((guard[4 + n:] == -7).all())
        z = _convert(src, torch.empty(n, dtype=torch.complex64, device="cuda"), 0)
        assert torch.equal(z.real, ref) and bool((z.imag == 0).all())
    f = torch.randn(n + off, device="cuda", generator=g)[off:]
    assert torch.equal(_convert(f, torch.empty(n, dtype=torch.complex64, device="cuda"), 0).real, f)
    z = torch.randn(n + off, dtype=torch.complex64, device="cuda", generator=g)[off:]
    assert rel_l2(_convert(z, torch.empty(n, device="cuda"), 2).cpu(), z.to(torch.complex128).abs().cpu()) < 1e-6
    assert rel_l2(_convert(z, torch.empty(n, device="cuda"), 3).cpu(), z.to(torch.complex128).angle().cpu()) < 1e-6
    if n > 1:
        lo, hi = f.min(), f.max()
        for dt, top in ((torch.uint8, 255.0), (torch.uint16, 65535.0)):
            got = _convert(f, torch.empty(n, dtype=dt, device="cuda"), 1).to(torch.int32)
            scale = torch.tensor(top, device="cuda") / (hi - lo)
            ref = ((f - lo) * scale + 0.5).to(torch.int32).clamp(0, int(top))
            assert int((got - ref).abs().max()) <= 1  # the product and sum may contract to one rounding
