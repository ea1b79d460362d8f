"""The rules that choose ordinary or non-temporal access by the amount of work:
16384-point fastconv rows at counts on both sides of each boundary (part of
the chip, the chip filled, a remainder of every kind), and four-step fastconvs
below 64 MB, from there on, and from 96 MB on.  One call of many rows gives, bit
for bit, what calls of few rows give, and sampled rows agree with FP64.

Tolerance: rel-L2 <= 1e-6: 20 radix-2 levels a transform at most, each adding
about 2^-24 that grows with the square root, sqrt(2) * 2 * sqrt(20) * 6e-8 =
8e-7 for a fastconv's two."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL_L2 = 1e-6


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,rows,few", [
    (16384, 223, 64), (16384, 224, 64), (16384, 256, 64), (16384, 257, 64), (16384, 479, 100), (16384, 480, 100),
    (65536, 127, 32), (65536, 128, 32), (65536, 191, 32), (65536, 192, 32), (1 << 20, 8, 2), (1 << 20, 12, 2)])
def test_many_rows_as_few(ovx, n, rows, few):
    import torch
    from openvsip_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(n + rows)
    x = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    w = torch.randn(n, dtype=torch.complex64, device="cuda", generator=gen)
    rep = ovx.Replica(n, w.cpu().numpy(), is_spectrum=True)
    fc = ovx.Fastconv(rows, n)
    y = fc.with_replica(x, rep, out=torch.empty_like(x))
    small = [ovx.Fastconv(min(few, rows - r), n).with_replica(x[r:r + few], rep, out=torch.empty_like(x[r:r + few]))
             for r in range(0, rows, few)]
    assert torch.equal(y, torch.cat(small))
    some = [0, rows // 2, rows - 1]
    y64 = np.fft.ifft(np.fft.fft(x[some].cpu().numpy().astype(np.complex128)) * w.cpu().numpy().astype(np.complex128))
    assert rel(y[some].cpu().numpy(), y64) < REL_L2

    def ptr(t):
        return ctypes.c_void_p(t.data_ptr())

    xr, xi, wr, wi = x.real.contiguous(), x.imag.contiguous(), w.real.contiguous(), w.imag.contiguous()
    yr, yi = torch.empty_like(xr), torch.empty_like(xi)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert _lib.lib().ovx_fastconv_split_exec(fc._h, ptr(xr), ptr(xi), n, ptr(wr), ptr(wi), 0, ptr(yr), ptr(yi), n,
                                              rows, stream) == 0
    assert rel(yr[some].cpu().numpy() + 1j * yi[some].cpu().numpy(), y64) < REL_L2
    fc.with_replica(x, rep, out=x)  # in place
    assert torch.equal(x, y)
