"""Every register-Stockham configuration (radices of 2, 3, 5 and 9 and their
products, few and many values per thread) at every compiled length: one line,
a few, and more than two lines per CU with a partly empty last workgroup, both
directions and fastconv against one spectrum and one per line, against FP64.

Tolerance: rel-L2 <= 1e-6: at most 15 radix-2 levels a transform, each adding a
relative error of about 2^-24 that grows with the square root of their number,
2 * sqrt(15) * 6e-8 = 4.6e-7 for a transform and sqrt(2) of it for the two of a
fastconv."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL_L2 = 1e-6

LENGTHS = sorted([1 << k for k in range(1, 15)] + [3 << k for k in range(0, 13)] + [5 << k for k in range(0, 12)]
                 + [9 << k for k in range(0, 11)])


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n", LENGTHS)
def test_every_row_configuration(ovx, n):
    import torch
    rng = np.random.default_rng(n)
    for rows in (1, 7, 517) if n <= 2560 else (1, 7):
        x = (rng.standard_normal((rows, n)) + 1j * rng.standard_normal((rows, n))).astype(np.complex64)
        w = (rng.standard_normal((rows, n)) + 1j * rng.standard_normal((rows, n))).astype(np.complex64)
        xd, wd = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
        x64, w64 = x.astype(np.complex128), w.astype(np.complex128)
        f64 = np.fft.fft(x64)
        # the default (by the number of lines) and every variant
        for v in [None] + list(range(ovx.variants(n))):
            fwd = ovx.Fftm(rows, n, variant=v)
            inv = ovx.Fftm(rows, n, direction=ovx.FFT_INV, scale=1.0 / n, variant=v)
            fc = ovx.Fastconv(rows, n, variant=v)
            assert rel(fwd(xd).cpu().numpy(), f64) < REL_L2, (n, rows, v)
            assert rel(inv(xd).cpu().numpy(), np.fft.ifft(x64)) < REL_L2, (n, rows, v)
            assert rel(fc(xd, wd[0].contiguous()).cpu().numpy(), np.fft.ifft(f64 * w64[0])) < REL_L2, (n, rows, v)
            if rows > 1:
                assert rel(fc(xd, wd).cpu().numpy(), np.fft.ifft(f64 * w64)) < REL_L2, (n, rows, v)
