"""The four-step middle pass over several rows per workgroup, and the column
pass's placement of rows: every line length (128 to 2048), one row and a few,
row counts that are no multiple of eight, that fill two and four rows per
workgroup with the last one partly empty, padded rows, in place, one spectrum
and one per row, both directions of the plain transform; sampled rows against
FP64.

Tolerance: rel-L2 <= 1e-6: 22 radix-2 levels a transform at most, each adding
about 2^-24 that grows with the square root, sqrt(2) * 2 * sqrt(22) * 6e-8 =
8e-7 for a fastconv's two."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL_L2 = 1e-6

# n, rows: 16 (32768) and 32 (65536) line groups a row need 2048 / 16 and 64
# rows for two rows per workgroup, four times that for four
CASES = [(32768, 1), (32768, 131), (32768, 517), (65536, 9), (65536, 67), (65536, 259), (131072, 35), (262144, 17),
         (524288, 9), (1 << 20, 5), (1 << 20, 17), (1 << 21, 3), (1 << 22, 2), (1 << 22, 9)]
# up to 32 MB of rows of at most 1 MB: worked on one XCD from pass to pass, one
# and two rows per workgroup, the last pair incomplete, fewer than eight rows,
# rows left over from eights
CASES += [(32768, 5), (32768, 96), (32768, 121), (65536, 41), (65536, 56), (65536, 64), (65536, 65), (131072, 7),
          (131072, 31)]


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,rows", CASES)
def test_four_step_rows(ovx, n, rows):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(n + rows)
    pad = 5 if rows * n < 1 << 25 else 0
    room = torch.randn(rows, n + pad, dtype=torch.complex64, device="cuda", generator=gen)
    x = room[:, :n]
    some = sorted({0, 1, rows // 2, max(rows - 2, 0), rows - 1} & set(range(rows)))
    x64 = x[some].cpu().numpy().astype(np.complex128)
    f64 = np.fft.fft(x64)
    w = torch.randn(n, dtype=torch.complex64, device="cuda", generator=gen)
    w64 = w.cpu().numpy().astype(np.complex128)
    fc = ovx.Fastconv(rows, n)
    y = fc(x, w, out=torch.empty_like(room)[:, :n])
    assert rel(y[some].cpu().numpy(), np.fft.ifft(f64 * w64)) < REL_L2
    fwd = ovx.Fftm(rows, n)(x, out=torch.empty_like(room)[:, :n])
    assert rel(fwd[some].cpu().numpy(), f64) < REL_L2
    inv = ovx.Fftm(rows, n, direction=ovx.FFT_INV, scale=1.0 / n)(x, out=torch.empty_like(room)[:, :n])
    assert rel(inv[some].cpu().numpy(), np.fft.ifft(x64)) < REL_L2
    if rows > 1 and rows * n <= 1 << 25:
        wm = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
        ym = fc(x, wm)
        assert rel(ym[some].cpu().numpy(), np.fft.ifft(f64 * wm[some].cpu().numpy().astype(np.complex128))) < REL_L2
    rep = ovx.Replica(n, w.cpu().numpy(), is_spectrum=True)
    fc.with_replica(x, rep, out=x)  # in place
    assert torch.equal(x, y)


@pytest.mark.parametrize("rows,n,pad", [(1, 65536, 1), (3, 65536, 33), (9, 16 * 2048, 8), (9, 131072, 5),
                                        (24, 131072, 33), (13, 1 << 20, 24), (50, 262144, 33)])
def test_rows_off_the_cache_lines(ovx, rows, n, pad):
    """Rows of other strides and bases than whole 128-byte lines are stored by
    other launches: the arithmetic of a line is the same, so the same bits."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(rows * n + pad)
    x = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=g)
    w = torch.randn(n, dtype=torch.complex64, device="cuda", generator=g)
    xo, yo = (torch.full((rows * (n + pad) + 1,), 7.0, dtype=torch.complex64, device="cuda") for _ in range(2))
    xp, yp = (t[1:].view(rows, n + pad) for t in (xo, yo))
    xp[:, :n].copy_(x)
    plans = [ovx.Fftm(rows, n, ovx.ROW, d, 0.5) for d in (ovx.FFT_FWD, ovx.FFT_INV)]
    calls = [lambda a, b, p=p: p(a, out=b) for p in plans]
    fc = ovx.Fastconv(rows, n)
    calls.append(lambda a, b: fc(a, w, out=b))
    for call in calls:
        want = call(x, torch.empty_like(x))
        call(xp[:, :n], yp[:, :n])
        assert torch.equal(yp[:, :n], want)
        assert bool((yp[:, n:] == 7.0).all()) and bool(yo[0] == 7.0)
