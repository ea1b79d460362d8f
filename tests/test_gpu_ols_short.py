"""Correlation and convolution with short kernels, whose segments share a wave:
kernels at the edges of the segment lengths (17 / 18, 33 / 34), outputs that fill
one segment, a wave of four and a second one, or miss each by one, decimation, the
unbiased divisors; and the error that the short segments keep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rel-L2: 7 radix-2 levels in each of three transforms, sqrt(2 * 3 * 7) * 6e-8 = 3.9e-7
REL_L2 = 5e-7


def cg(rng, n):
    return (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)


def full(a, b):
    """Convolution of two signals in 64 bits."""
    size = a.size + b.size - 1
    return np.fft.ifft(np.fft.fft(a.astype(np.complex128), size) * np.fft.fft(b.astype(np.complex128), size))


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("m,length", [(1, 64), (2, 64), (16, 64), (17, 64), (18, 128), (32, 128), (33, 128)])
@pytest.mark.parametrize("segments", [1, 4, 5])
@pytest.mark.parametrize("more", [-1, 0, 1])
def test_segments_that_share_a_wave(ovx, m, length, segments, more):
    import torch
    n = segments * (length - (m - 1)) + more - (m - 1)
    if n < m:
        pytest.skip("a kernel longer than its signal")
    rng = np.random.default_rng(1000 * m + 10 * segments + more)
    ref, x = cg(rng, m), cg(rng, n)
    rd, xd = torch.from_numpy(ref).cuda(), torch.from_numpy(x).cuda()
    c = full(ref[::-1], x.conj())
    for support, at in (("full", 0), ("same", m - 1 - m // 2), ("min", m - 1)):
        plan = ovx.Correlation(support, m, n)
        p = plan.output_size
        got = plan("biased", rd, xd).cpu().numpy()
        assert rel(got, c[at:at + p]) < REL_L2, support
        divisor = full(np.ones(m, np.complex64), np.ones(n, np.complex64)).real[at:at + p].round()
        if support != "same":
            assert rel(plan("unbiased", rd, xd).cpu().numpy(), c[at:at + p] / divisor) < REL_L2, support
    c = full(ref, x)
    for d in (1, 3, 7):
        got = ovx.Convolution(ref, "nonsym", "full", n, d)(xd).cpu().numpy()
        assert rel(got, c[::d]) < REL_L2, d


@pytest.mark.parametrize("m,n", [(8, 700000), (33, 1100000)])
def test_reference_in_many_segments(ovx, m, n):
    import torch
    rng = np.random.default_rng(m)
    ref, x = cg(rng, m), cg(rng, n)
    got = ovx.Correlation("full", m, n)("biased", torch.from_numpy(ref).cuda(), torch.from_numpy(x).cuda())
    assert rel(got.cpu().numpy(), full(ref[::-1], x.conj())) < REL_L2


@pytest.mark.parametrize("m,bound", [(1, 1.55e-7), (8, 1.55e-7), (17, 1.55e-7), (18, 1.62e-7), (33, 1.65e-7)])
def test_error_of_short_kernels(ovx, m, bound):
    """The error grows with the root of a transform's levels: 1.70e-7 in segments
    of 512 points, 1.39e-7 in 64 and 1.50e-7 in 128; the bounds lie between."""
    import torch
    errors = []
    for seed in range(4):
        rng = np.random.default_rng(seed)
        ref, x = cg(rng, m), cg(rng, 100000)
        rd, xd = torch.from_numpy(ref).cuda(), torch.from_numpy(x).cuda()
        errors.append(rel(ovx.Correlation("full", m, x.size)("biased", rd, xd).cpu().numpy(), full(ref[::-1], x.conj())))
        errors.append(rel(ovx.Convolution(ref, "nonsym", "full", x.size, 1)(xd).cpu().numpy(), full(ref, x)))
    assert np.mean(errors) < bound
