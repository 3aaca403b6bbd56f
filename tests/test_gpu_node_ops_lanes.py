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


@pytest.mark.parametrize("n", [1, 2, 3, 511, 512, 513, 1023, 1025, 4095, (1 << 21) - 1, 1 << 21, (1 << 21) + 1027])
@pytest.mark.parametrize("src", [torch.uint8, torch.uint16, torch.float32])
def test_conversion_tails(gpu, n, src):
    from holoflow_amd._lib import DTYPE_CF32, DTYPE_F32, DTYPE_U16, check, lib
    import ctypes as C

    host = torch.arange(n, dtype=torch.int64) * 7 % (255 if src == torch.uint8 else 65521)
    x = host.to(torch.int32).to(src).cuda() if src != torch.float32 else (host - 9.5).float().cuda()
    if src == torch.float32 and n > 2:
        x[0], x[n // 2], x[n - 1] = float("nan"), -0.0, float("inf")
    want = x.cpu().float() if src == torch.float32 else host.float()
    for dt, out in ((DTYPE_F32, torch.full((n + 1,), -3.0, device="cuda")),
                    (DTYPE_CF32, torch.full((n + 1,), -3.0, dtype=torch.complex64, device="cuda"))):
        if src == torch.float32 and dt == DTYPE_F32:
            continue
        code = {torch.uint8: 4, torch.uint16: DTYPE_U16, torch.float32: DTYPE_F32}[src]
        check(lib().hfx_convert(C.c_void_p(x.data_ptr()), code, C.c_void_p(out.data_ptr()), dt, 0, n, None,
                                C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        got = out.cpu()
        re = got.real if got.is_complex() else got
        assert torch.equal(re[:n].contiguous().view(torch.int32), want.view(torch.int32)) and float(re[n]) == -3.0
        if got.is_complex():
            assert not bool(got.imag.any())


@pytest.mark.parametrize("n", [1, 3, 513, 4095, 1 << 21, (1 << 21) + 1025])
@pytest.mark.parametrize("off", [0, 1])
def test_modulus_and_argument_tails(gpu, n, off):
    from holoflow_amd._lib import DTYPE_CF32, DTYPE_F32, check, lib
    import ctypes as C

    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n + off, dtype=torch.complex64, device="cuda", generator=g)[off:]
    out = torch.empty(n, device="cuda")
    d = x.to(torch.complex128)
    for strategy, ref in ((2, d.abs()), (3, d.angle())):
        check(lib().hfx_convert(C.c_void_p(x.data_ptr()), DTYPE_CF32, C.c_void_p(out.data_ptr()), DTYPE_F32, strategy, n,
                                None, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        # hypotf and atan2f are within a few ulp
        assert bool(((out - ref).abs() <= 8 * 2.0**-24 * ref.abs() + 1e-30).all())


@pytest.mark.parametrize("kind", ["u16", "f32", "cf32"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 12, 13])
@pytest.mark.parametrize("outer,inner", [(1, 4099), (3, 64), (70, 1), (5, 33), (1, 300 * 3)])
def test_dft_of_few_points_and_odd_columns(gpu, kind, n, outer, inner):
    """The direct sums up to eight points and the matrix form beyond, with columns that are and are not
    adjacent per lane."""
    from holoflow_amd import hfx

    g = torch.Generator().manual_seed(n + inner)
    if kind == "u16":
        x = torch.randint(0, 1 << 16, (outer, n, inner), generator=g, dtype=torch.int32)
        wide, x = x.double(), x.to(torch.uint16)
    else:
        x = torch.randn((outer, n, inner), generator=g, dtype=torch.float32 if kind == "f32" else torch.complex64)
        wide = x.to(torch.complex128)
    for kb, ke in ((0, n), (n - 1, n), (0, n // 2 + 1)):
        ref = torch.fft.fft(wide, dim=1)[:, kb:ke]
        got = hfx.dft_axis(x.cuda(), 1, kb, ke).cpu()
        # n products with twiddles rounded once, summed in FP32
        bound = (n + 2) * 2.0**-23 * wide.abs().sum(1, keepdim=True) * 2**0.5
        assert bool(((got - ref).abs() <= bound).all())
