"""Rows of 2 MB on both sides of the counts at which the passes of a call stay on
one XCD (eight rows, ten for a fastconv's middle pass): transforms and fastconv,
in place and not, interleaved and split, every row against 64 bits.

Tolerance: rel-L2 1e-6 (18 radix-2 levels a transform, two transforms:
sqrt(2) * 2 * sqrt(18) * 6e-8 = 7.2e-7)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 262144


@pytest.mark.parametrize("rows", [7, 8, 9, 10, 11])
def test_rows_of_two_megabytes(ovx, rows):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, N, dtype=torch.complex64, device="cuda", generator=gen)
    w = torch.randn(N, dtype=torch.complex64, device="cuda", generator=gen)
    f64 = np.fft.fft(x.cpu().numpy().astype(np.complex128))
    c64 = np.fft.ifft(f64 * w.cpu().numpy())

    def check(got, want):
        for a, b in zip(got.cpu().numpy(), want):
            assert np.linalg.norm(a - b) < 1e-6 * np.linalg.norm(b)

    fwd = ovx.Fftm(rows, N, ovx.ROW, ovx.FFT_FWD, 1.0)
    y = fwd(x)
    check(y, f64)
    here = x.clone()
    fwd(here, out=here)
    assert torch.equal(here, y)
    check(ovx.Fftm(rows, N, ovx.ROW, ovx.FFT_INV, 1.0 / N)(y), x.cpu().numpy())
    fc = ovx.Fastconv(rows, N)
    y = fc(x, w)
    check(y, c64)
    here = x.clone()
    fc(here, w, out=here)
    assert torch.equal(here, y)
    check(fc.with_replica(x, ovx.Replica(N, w.cpu().numpy(), is_spectrum=True)), c64)
    xr, xi, wr, wi = (t.contiguous() for t in (x.real, x.imag, w.real, w.imag))
    yr, yi = torch.empty_like(xr), torch.empty_like(xi)
    p = [ctypes.c_void_p(t.data_ptr()) for t in (xr, xi, wr, wi, yr, yi)]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert ovx._lib.lib().ovx_fastconv_split_exec(fc._h, p[0], p[1], N, p[2], p[3], 0, p[4], p[5], N, rows, stream) == 0
    assert torch.equal(torch.complex(yr, yi), y)
