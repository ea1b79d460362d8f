"""Overlap-save segments of correlation and convolution: kernels at the edges of
the segment lengths (1, 256 / 257, 512, 1025, 2049, 16384 taps), signals of a
part of a segment, of whole segments and one value more, enough segments for
the reference's spectrum to be computed once instead of in every segment,
decimations that divide nothing, exceed a segment or leave one output.

Against float64 (scipy's FFT convolution), rel-L2 <= 1.5e-6: the linear
convolution of a segment is three FP32 transforms of at most 14 levels, each
adding about 2^-24 per level that grows with the square root,
sqrt(3) * 2 * sqrt(14) * 6e-8 = 7.8e-7; up to twice that as the bar, as the
valid outputs are half a segment's energy.  The unbiased divisors are checked
exactly: the biased outputs divided by them in float32."""
import numpy as np
import pytest
from scipy.signal import fftconvolve

pytestmark = pytest.mark.gpu

REL_L2 = 1.5e-6


def cg(rng, n):
    return (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def divisor(support, p, m, n):
    k = np.arange(p)
    d = np.full(p, m, dtype=np.float32)
    if support == "full":
        d = np.where(k < m - 1, k + 1, np.where(k >= n, n + m - 1 - k, d))
    elif support == "same":
        d = np.where(k < m // 2, k + (m + 1) // 2, np.where(k >= n - m // 2, n - 1 + (m + 1) // 2 - k, d))
    return d.astype(np.float32)


@pytest.mark.parametrize("m,n", [(1, 1), (1, 600), (17, 17), (16, 497), (16, 498), (256, 3001), (257, 3001),
                                 (512, 9000), (513, 2048), (1025, 5000), (2049, 30000), (16384, 20000),
                                 (5, 530001), (300, 800001)])
def test_correlation_segments(ovx, m, n):
    import torch
    rng = np.random.default_rng(m * 7 + n)
    ref, x = cg(rng, m), cg(rng, n)
    rd, xd = torch.from_numpy(ref).cuda(), torch.from_numpy(x).cuda()
    c = fftconvolve(ref[::-1].astype(np.complex128), x.conj().astype(np.complex128))
    for support in ("full", "same", "min"):
        shift = {"full": m - 1, "same": m // 2, "min": 0}[support]
        plan = ovx.Correlation(support, m, n)
        p = plan.output_size
        biased = plan("biased", rd, xd).cpu().numpy()
        assert rel(biased, c[m - 1 - shift: m - 1 - shift + p]) < REL_L2, (support, m, n)
        unbiased = plan("unbiased", rd, xd).cpu().numpy()
        d = divisor(support, p, m, n)
        assert np.array_equal(unbiased.real, biased.real / d) and np.array_equal(unbiased.imag, biased.imag / d)


@pytest.mark.parametrize("m,n,d", [(1, 700, 1), (9, 5000, 3), (129, 40007, 4), (129, 40007, 7), (257, 9001, 600),
                                   (64, 100000, 32768), (64, 100000, 33000), (64, 100000, 99999), (64, 1000, 5000),
                                   (1000, 30011, 2), (33, 700001, 5)])
def test_convolution_segments_and_decimation(ovx, m, n, d):
    import torch
    rng = np.random.default_rng(m + n + d)
    h, x = cg(rng, m), cg(rng, n)
    xd = torch.from_numpy(x).cuda()
    c = fftconvolve(h.astype(np.complex128), x.astype(np.complex128))
    for support in ("full", "same", "min"):
        plan = ovx.Convolution(h, "nonsym", support, n, d)
        off = {"full": 0, "same": m // 2, "min": m - 1}[support]
        want = c[off::d][: plan.output_size]
        out = torch.full((plan.output_size + 3,), 7.0, dtype=torch.complex64, device="cuda")
        plan(xd, out=out[: plan.output_size])
        got = out.cpu().numpy()
        # one value has no other to average its rounding with: the bar is the
        # error of the record's, not of itself
        scale = np.linalg.norm(want) if want.size > 8 else np.sqrt(want.size) * np.sqrt(np.mean(np.abs(c) ** 2)) * 4
        assert np.linalg.norm(got[: want.size] - want) / scale < REL_L2, (support, m, n, d)
        assert np.all(got[want.size:] == 7.0)


@pytest.mark.parametrize("support,m,n", [("same", 200, 800), ("min", 150, 1000), ("full", 300, 900), ("min", 1024, 9000),
                                         ("same", 17, 300), ("same", 2000, 16384)])
def test_result_over_the_operands(ovx, support, m, n):
    """A result that is stored over the signal, and one over the reference: in
    one segment and in several, whose stores meet each other's samples."""
    import torch
    rng = np.random.default_rng(m * 3 + n)
    ref, x = cg(rng, m), cg(rng, n)
    rd, xd = torch.from_numpy(ref).cuda(), torch.from_numpy(x).cuda()
    shift = {"full": m - 1, "same": m // 2, "min": 0}[support]
    corr = ovx.Correlation(support, m, n)
    conv = ovx.Convolution(ref, "nonsym", support, n, 1)
    p = corr.output_size
    c = fftconvolve(ref[::-1].astype(np.complex128), x.conj().astype(np.complex128))[m - 1 - shift:][:p]
    for operand, at in ((xd, 0), (rd, 0), (rd, p - m // 2)):
        buf = torch.zeros(2 * (n + m), dtype=torch.complex64, device="cuda")
        # the operand begins `at` values into the result
        over = buf[at: at + operand.numel()]
        over.copy_(operand)
        out = buf[:p]
        corr("biased", over if operand is rd else rd, over if operand is xd else xd, out=out)
        assert rel(out.cpu().numpy(), c) < REL_L2, (support, m, n, at)
    q = conv.output_size
    c = fftconvolve(ref.astype(np.complex128), x.astype(np.complex128))
    off = {"full": 0, "same": m // 2, "min": m - 1}[support]
    buf = torch.zeros(2 * (n + m), dtype=torch.complex64, device="cuda")
    buf[:n].copy_(xd)
    conv(buf[:n], out=buf[:q])
    assert rel(buf[:q].cpu().numpy(), c[off: off + q]) < REL_L2, (support, m, n)
