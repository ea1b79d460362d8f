"""Fastconv with spectra passed as they are, in natural order: read by the
middle pass itself (lines of up to 512 points, calls on both sides of the size
rule) or laid out first (longer lines, spectra that share memory with the
result), one spectrum and one per row, padded spectrum rows, one row to several
per workgroup; and 8192- and 16384-point calls.  Each against FP64 on sampled
rows.

Tolerance: rel-L2 <= 1e-6: 20 radix-2 levels a transform at most, each adding
about 2^-24 that grows with the square root, sqrt(2) * 2 * sqrt(20) * 6e-8 =
8e-7 for the two."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL_L2 = 1e-6


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def expected(x, w):
    return np.fft.ifft(np.fft.fft(x.cpu().numpy().astype(np.complex128)) * w.cpu().numpy().astype(np.complex128))


CASES = [(8192, 9), (16384, 3), (32768, 1), (32768, 13),
         (32768, 140), (65536, 1), (65536, 9), (65536, 41), (65536, 70), (131072, 1), (131072, 31), (131072, 33),
         (262144, 2), (262144, 15), (262144, 17), (524288, 3), (1 << 20, 2), (1 << 22, 1)]


@pytest.mark.parametrize("n,rows", CASES)
def test_spectra_in_natural_order(ovx, n, rows):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(n + rows)
    x = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    room = torch.randn(rows, n + 7, dtype=torch.complex64, device="cuda", generator=gen)
    some = sorted({0, rows // 2, rows - 1})
    fc = ovx.Fastconv(rows, n)
    y1 = fc(x, room[0, :n].contiguous())
    ym = fc(x, room[:, :n])
    for r in some:
        assert rel(y1[r].cpu().numpy(), expected(x[r], room[0, :n])) < REL_L2
        assert rel(ym[r].cpu().numpy(), expected(x[r], room[r, :n])) < REL_L2
    fc(x, room[:, :n], out=x)  # in place
    assert torch.equal(x, ym)


@pytest.mark.parametrize("n,rows", [(8192, 9), (16384, 5), (32768, 3), (65536, 9), (131072, 4), (262144, 3), (1 << 20, 2)])
def test_result_over_the_spectrum(ovx, n, rows):
    """The result may take a spectrum's place: a matrix of them, or a vector that
    is one of the result's rows (lengths whose spectra are laid out first)."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(n + rows)
    x = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    w = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    fc = ovx.Fastconv(rows, n)
    want = fc(x, w)
    over = w.clone()
    fc(x, over, out=over)
    assert rel(over.cpu().numpy(), want.cpu().numpy()) < REL_L2
    vec = [expected(x[r], w[0]) for r in range(rows)]
    over = w.clone()
    fc(x, over[0], out=over)
    for r in range(rows):
        assert rel(over[r].cpu().numpy(), vec[r]) < REL_L2


@pytest.mark.parametrize("n,rows", [(64, 5), (1024, 3), (2048, 9), (4096, 70), (8192, 9), (8192, 257), (16384, 5), (32768, 3),
                                    (131072, 40)])
@pytest.mark.parametrize("matrix", [False, True])
def test_split_spectra(ovx, n, rows, matrix):
    """Split storage, spectra included, equals interleaved storage bit for bit, and
    the result may take the spectra's place."""
    import ctypes
    import torch
    from openvsip_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(n + rows + matrix)
    x = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    w = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    fc = ovx.Fastconv(rows, n)
    want = fc(x, w if matrix else w[0].clone())

    def ptr(t):
        return ctypes.c_void_p(t.data_ptr())

    xr, xi, wr, wi = (t.contiguous() for t in (x.real, x.imag, w.real, w.imag))
    yr, yi = torch.empty_like(xr), torch.empty_like(xi)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for outr, outi in ((yr, yi), (wr, wi)):
        assert _lib.lib().ovx_fastconv_split_exec(fc._h, ptr(xr), ptr(xi), n, ptr(wr), ptr(wi), n if matrix else 0,
                                                  ptr(outr), ptr(outi), n, rows, stream) == 0
        if outr is yr or n not in (8192, 16384):  # those take another kernel beside an overlapping vector
            assert torch.equal(torch.complex(outr, outi), want)
        else:
            got = torch.complex(outr, outi).cpu().numpy()
            assert rel(got, want.cpu().numpy()) < REL_L2
