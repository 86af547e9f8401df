"""GPU parity of conv1d / corr by the FFT method (mxr_conv1d_fft; MatX
MATX_C_METHOD_FFT, include/matx/transforms/conv.h:51-172, corr.h:60-67)
against the FP64 direct convolution of the oracle (pinned to MatX's ConvCorr
KATs and numpy.convolve in tests/test_oracle.py).  corr(x, f) is checked as
conv1d(x, reverse(conj(f))).  Relative L2 <= 1e-5.

Covers the fused path (n + L - 1 <= 16384: real and complex, even and odd
filters, filters longer than the signal, strided batch views) and the long
path (overlap-save correlation plus the fused head), including the size of
MatX's CorrelationConvolutionLargeTest (n = 8*122880 + 2*32768, L = 209).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

RTOL = 1e-5


def rel(a, b):
    a = np.asarray(a, dtype=np.complex128)
    b = np.asarray(b, dtype=np.complex128)
    return float(np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300))


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def sig(rng, shape, cplx):
    x = rng.standard_normal(shape)
    if cplx:
        x = x + 1j * rng.standard_normal(shape)
        return x.astype(np.complex64)
    return x.astype(np.float32)


def dev(a):
    return torch.as_tensor(np.ascontiguousarray(a)).cuda()


@pytest.fixture(scope="module")
def mx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import matx_amd
    matx_amd.lib()
    return matx_amd


def modes(N, L):
    return ("full", "same", "valid") if N >= L else ("full", "same")


@pytest.mark.parametrize("rows,N,L,xc,fc", [
    ((3,), 256, 16, True, True),       # ConvCorr.cu sizes (even and odd filters)
    ((3,), 256, 15, True, False),
    ((2, 2), 128, 8, False, False),    # real in, real filter: real output
    ((4,), 128, 7, False, True),
    ((2,), 16, 256, True, True),       # filter longer than the signal
    ((5,), 1000, 1, True, True),
    ((2,), 5000, 3000, True, True),
    ((1,), 10000, 6385, False, False),  # n + L - 1 = 16384
])
def test_conv1d_corr_fft_fused(mx, orc, rows, N, L, xc, fc):
    rng = np.random.default_rng(N + L)
    x = sig(rng, rows + (N,), xc)
    f = sig(rng, (L,), fc)
    fr = np.conj(f[::-1])
    for mode in modes(N, L):
        got = host(mx.conv1d(dev(x), dev(f), mode, method="fft"))
        ref = orc.conv1d(x, f, mode)
        if not (xc or fc):
            assert got.dtype == np.float32
            ref = ref.real
        assert rel(got, ref) < RTOL, mode
        got = host(mx.corr(dev(x), dev(f), mode, method="fft"))
        ref = orc.conv1d(x, fr, mode)
        assert rel(got, ref.real if not (xc or fc) else ref) < RTOL, mode
        if L <= 4096:  # the direct method's filter limit
            got = host(mx.corr(dev(x), dev(f), mode, method="direct"))
            assert rel(got, ref.real if not (xc or fc) else ref) < RTOL, mode


def test_conv1d_fft_strided_views(mx, orc):
    """A permuted input view (the transform axis strided) and an output view
    into a wider buffer."""
    rng = np.random.default_rng(5)
    x = sig(rng, (3, 300, 4), True)
    f = sig(rng, (33,), True)
    xd = dev(x).permute(0, 2, 1)              # [3, 4, 300], axis stride 4
    buf = torch.zeros((3, 4, 400), dtype=torch.complex64, device="cuda")
    out = buf[:, :, 10:10 + 300]
    mx.conv1d(xd, dev(f), "same", method="fft", out=out)
    ref = orc.conv1d(np.moveaxis(x, 1, 2), f, "same")
    assert rel(host(out), ref) < RTOL
    assert float(buf[:, :, :10].abs().max()) == 0.0


@pytest.mark.parametrize("N,L", [(8 * 122880 + 2 * 32768, 209), (100000, 4096), (40000, 3)])
def test_conv1d_corr_fft_long(mx, orc, N, L):
    """Rows past the fused kernel: overlap-save correlation blocks for the
    outputs at FULL index >= L-1, the fused kernel on x[0, L-1) before."""
    rng = np.random.default_rng(N % 1000 + L)
    x = sig(rng, (N,), True)
    f = sig(rng, (L,), True)
    fr = np.conj(f[::-1])
    xd, fd = dev(x), dev(f)
    for mode in ("full", "same", "valid"):
        assert rel(host(mx.conv1d(xd, fd, mode, method="fft")), orc.conv1d(x, f, mode)) < RTOL, mode
        assert rel(host(mx.corr(xd, fd, mode, method="fft")), orc.conv1d(x, fr, mode)) < RTOL, mode


def test_conv1d_fft_long_batched(mx, orc):
    rng = np.random.default_rng(9)
    x = sig(rng, (3, 20000), True)
    f = sig(rng, (500,), True)
    got = host(mx.conv1d(dev(x), dev(f), "same", method="fft"))
    assert rel(got, orc.conv1d(x, f, "same")) < RTOL


def test_conv1d_fft_errors(mx):
    x = torch.zeros((20000,), dtype=torch.float32, device="cuda")
    f = torch.zeros((9,), dtype=torch.float32, device="cuda")
    with pytest.raises(Exception, match="c64"):
        mx.conv1d(x, f, "full", method="fft")   # long rows need complex operands
    with pytest.raises(Exception, match="VALID"):
        mx.conv1d(f, x[:100], "valid", method="fft",
                  out=torch.empty((0,), dtype=torch.float32, device="cuda"))
    with pytest.raises(ValueError):
        mx.conv1d(f, f, "full", method="winograd")


@pytest.mark.parametrize("n", [2, 16, 32, 64, 256, 512, 1024, 2048, 4096, 3, 7, 100, 129, 300, 700, 1025])
@pytest.mark.parametrize("cols", [1, 15, 33])
def test_fft_axes_direct(mx, n, cols):
    """Transforms along a contiguous and along a strided axis, batches that do
    not fill a workgroup, inputs shorter and longer than the transform, both
    directions, real in and out, in place, against numpy in FP64."""
    rng = np.random.default_rng(100 * n + cols)
    for extent in {n, max(1, n - n // 3), n + 5}:
        x = sig(rng, (2, extent, cols), True)
        xt = np.ascontiguousarray(x.transpose(0, 2, 1))
        r = sig(rng, (2, extent, cols), False)
        ref, inv = np.fft.fft(x.astype(complex), n, axis=1), np.fft.ifft(x.astype(complex), n, axis=1)
        assert rel(host(mx.fft(dev(x), n, 1)), ref) < RTOL
        assert rel(host(mx.ifft(dev(x), n, 1)), inv) < RTOL
        assert rel(host(mx.fft(dev(xt), n)), ref.transpose(0, 2, 1)) < RTOL
        assert rel(host(mx.ifft(dev(xt), n)), inv.transpose(0, 2, 1)) < RTOL
        rr = np.fft.rfft(r.astype(float), n, axis=1)
        assert rel(host(mx.rfft(dev(r), n, 1)), rr) < RTOL
        assert rel(host(mx.rfft(dev(np.ascontiguousarray(r.transpose(0, 2, 1))), n)), rr.transpose(0, 2, 1)) < RTOL
        h = sig(rng, (2, n // 2 + 1, cols), True)
        back = np.fft.irfft(h.astype(complex), n, axis=1)
        assert rel(host(mx.irfft(dev(h), n, 1)), back) < RTOL
    y = dev(x := sig(rng, (3, n, cols), True))
    mx.fft(y, n, 1, out=y)
    assert rel(host(y), np.fft.fft(x.astype(complex), axis=1)) < RTOL


@pytest.mark.parametrize("n,cols", [(24, 33), (30, 300), (45, 15), (60, 1), (96, 33), (100, 70), (135, 15),
                                    (225, 33), (360, 15), (1000, 33), (1000, 1200), (1152, 15), (1500, 33),
                                    (2187, 3), (3000, 15), (3125, 3), (4500, 9), (5184, 2), (7200, 3)])
def test_fft_mixed_radix(mx, n, cols):
    """Sizes without large primes: every radix as a first, a middle and a last
    pass, odd first radices and padded even ones, batches that do not fill a
    workgroup and those that make it larger; the largest row a workgroup
    holds."""
    test_fft_axes_direct(mx, n, cols)


@pytest.mark.parametrize("mode", ["full", "same", "valid"])
@pytest.mark.parametrize("L", [2, 17, 210, 1300, 4001])
def test_conv1d_long_rows_from_first_lag(mx, mode, L):
    """Long rows start at the mode's first lag: outputs that reach before the
    row, convolution and correlation, each block size, a filter that is part
    of the signal, against numpy in FP64."""
    rng = np.random.default_rng(L)
    N = 20011
    x, f = sig(rng, (2, N), True), sig(rng, (L,), True)
    xd = dev(x)
    X = np.fft.fft(x.astype(complex), 32768)
    s0, num = {"full": (0, N + L - 1), "same": ((L - 1) // 2, N), "valid": (L - 1, N - L + 1)}[mode]
    for corr in (False, True):
        h = np.conj(f[::-1]) if corr else f
        ref = np.fft.ifft(X * np.fft.fft(h.astype(complex), 32768))[:, s0:s0 + num]
        got = (mx.corr if corr else mx.conv1d)(xd, dev(f), mode, method="fft")
        assert rel(host(got), ref) < RTOL
    part = xd[1, 5:5 + L]
    ref = np.fft.ifft(X * np.fft.fft(x[1, 5:5 + L].astype(complex), 32768))[:, s0:s0 + num]
    assert rel(host(mx.conv1d(xd, part, mode, method="fft")), ref) < RTOL


@pytest.mark.parametrize("n,L", [(1024, 1), (1024, 100), (1024, 1024), (2048, 300), (16384, 100), (16384, 300)])
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("conj", [True, False])
def test_fft_conv_waveform_beside_blocks(mx, n, L, rows, conj):
    """Small calls whose workgroups transform the waveform beside one or three
    blocks: rows that do not fill a workgroup, wrapping blocks, both forms."""
    rng = np.random.default_rng(n + L + rows)
    S = n - n // 5
    x, w = sig(rng, (rows, S), True), sig(rng, (L,), True)
    W = np.fft.fft(w.astype(complex), n)
    ref = np.fft.ifft(np.fft.fft(x.astype(complex), n) * (np.conj(W) if conj else W))
    assert rel(host(mx.fft_conv(dev(x), dev(w), n, conj=conj)), ref) < RTOL


@pytest.mark.parametrize("S,L,n", [(9000, 1000, 16384), (20000, 900, 32768), (30000, 3000, 32768), (1500, 200, 2048)])
def test_pulse_compress_in_place_rows(mx, S, L, n):
    """In place: a row's blocks one after another in one workgroup, bit for bit
    (same block size) or closely (another one) the out-of-place result."""
    rng = np.random.default_rng(S)
    x = dev(sig(rng, (3, n), True))
    w = dev(sig(rng, (L,), True))
    y = mx.pulse_compress(x[:, :S], w, n=n)
    buf = x.clone()
    out = buf[:, :S - L + 1]
    mx.pulse_compress(buf[:, :S], w, n=n, out=out)
    assert rel(host(out), host(y)) < 1e-6
    assert np.array_equal(host(buf[:, S:]), host(x[:, S:]))


@pytest.mark.parametrize("n", [32, 64, 128, 256, 512, 1024, 2048, 4096, 8192, 16384, 65536, 100, 29, 509, 2039])
def test_fft_large_magnitudes(mx, n):
    """Samples of 1e31: every intermediate of a transform is at most n times
    that, far from the largest float, so nothing overflows on the way (both
    directions, contiguous and strided, chirp-z and mixed radix too)."""
    rng = np.random.default_rng(n)
    x = (1e31 * (sig(rng, (3, n), True))).astype(np.complex64)
    xs = np.ascontiguousarray(np.repeat(x[:, :, None], 5, axis=2))
    for ref, f in ((np.fft.fft(x.astype(complex)), mx.fft), (np.fft.ifft(x.astype(complex)), mx.ifft)):
        assert rel(host(f(dev(x), n)) / 1e31, ref / 1e31) < RTOL
        assert rel(host(f(dev(xs), n, 1)) / 1e31, np.repeat(ref[:, :, None], 5, axis=2) / 1e31) < RTOL


@pytest.mark.parametrize("N,L", [(20, 5), (300, 33), (3000, 500), (9000, 700), (20011, 210), (20011, 1300), (20011, 4001)])
def test_conv_large_magnitudes(mx, N, L):
    """The same for convolutions (one workgroup a row, overlap-save blocks) and
    matched filters: signals of 1e31 under unit filters."""
    rng = np.random.default_rng(N + L)
    x, f = (1e31 * sig(rng, (2, N), True)).astype(np.complex64), sig(rng, (L,), True)
    n = max(1024, 1 << (N + L - 1).bit_length())   # fft_conv's smallest transform
    X = np.fft.fft(x.astype(complex) / 1e31, n)
    full = np.fft.ifft(X * np.fft.fft(f.astype(complex), n))[:, :N + L - 1]
    assert rel(host(mx.conv1d(dev(x), dev(f), "full", method="fft")) / 1e31, full) < RTOL
    lags = np.fft.ifft(X * np.conj(np.fft.fft(f.astype(complex), n)))
    assert rel(host(mx.fft_conv(dev(x), dev(f), n)) / 1e31, lags) < RTOL
    buf = dev(x)
    R = N - L + 1
    mx.pulse_compress(buf, dev(f), n, window=False, normalize=False, out=buf[:, :R])
    assert rel(host(buf[:, :R]) / 1e31, lags[:, :R]) < RTOL


@pytest.mark.parametrize("n", [7, 11, 29, 59, 101, 251, 509, 1021, 2039, 4093, 8191])
@pytest.mark.parametrize("cols", [1, 15])
def test_fft_chirp_z_lengths(mx, n, cols):
    """Primes, one for every convolution length of the chirp-z kernels (16 to
    16384 points): contiguous and strided, both directions, real in and out."""
    test_fft_axes_direct(mx, n, cols)


@pytest.mark.parametrize("L", [700, 3000])   # blocks of 4096 and 8192 points
@pytest.mark.parametrize("over", [0, 1])
def test_conv1d_longest_rows(mx, L, over):
    """FULL outputs of rows that just fit a period of 2^27 samples, the largest
    of the block kernels' 32-bit byte offsets, and of rows one longer (general
    addressing): the first blocks start before the row, the last end past it.
    Noise at either end of the row, zeros between."""
    rng = np.random.default_rng(L)
    N, K = (1 << 27) - L + 1 + over, 5000
    a, b, f = sig(rng, (K,), True), sig(rng, (K,), True), sig(rng, (L,), True)
    x = torch.zeros((1, N), dtype=torch.complex64, device="cuda")
    x[0, :K], x[0, N - K:] = dev(a), dev(b)
    y = mx.conv1d(x, dev(f), "full", method="fft")
    f64 = lambda u: np.fft.fft(u.astype(complex), 16384)  # noqa: E731
    lo, hi = (np.fft.ifft(f64(u) * f64(f))[:K + L - 1] for u in (a, b))
    assert rel(host(y[0, :K + L - 1]), lo) < RTOL
    assert rel(host(y[0, N - K:]), hi) < RTOL
    assert not y[0, K + L + 16384:N - K - 16384].any()


def test_conv1d_long_rows_error(mx):
    """Rows of 1048576 samples through 4096-point blocks lose no accuracy to
    2048-point ones, which erred by 2.12e-7 here: a radix-16 block of twice the
    points has 12 / 11 = 1.09 times the levels, so 1.1 times that is allowed."""
    rng = np.random.default_rng(209)
    N, L = 1048576, 209
    x, f = sig(rng, (4, N), True), sig(rng, (L,), True)
    n = 1 << 21
    ref = np.fft.ifft(np.fft.fft(x.astype(complex), n) * np.fft.fft(f.astype(complex), n))[:, (L - 1) // 2:(L - 1) // 2 + N]
    assert rel(host(mx.conv1d(dev(x), dev(f), "same", method="fft")), ref) < 1.1 * 2.12e-7
