"""Real transforms longer than one workgroup's LDS: the passes that split and
join the half-length transform, one pair a thread and four, row counts that are
no multiple of eight, both directions, interleaved and (through the complex half)
a round trip.  FP64 on sampled rows.

Tolerance: rel-L2 <= 1e-6: 17 radix-2 levels and the pair step, each adding about
2^-24 that grows with the square root, 2 * sqrt(18) * 6e-8 = 5e-7; a round trip
sqrt(2) times that."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL_L2 = 1e-6


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,rows", [(65536, 1), (65536, 9), (65536, 31), (65536, 33), (65536, 130), (131072, 15),
                                    (131072, 17), (131072, 66), (524288, 3), (524288, 5)])
def test_long_real_rows(ovx, n, rows):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(n + rows)
    x = torch.randn(rows, n, device="cuda", generator=gen)
    some = sorted({0, rows // 2, rows - 1})
    f = ovx.FftmReal(rows, n)(x)
    assert rel(f[some].cpu().numpy(), np.fft.rfft(x[some].cpu().numpy().astype(np.float64))) < REL_L2
    y = ovx.FftmReal(rows, n, ovx.ROW, ovx.FFT_INV, 1.0 / n)(f)
    assert rel(y.cpu().numpy(), x.cpu().numpy()) < REL_L2
