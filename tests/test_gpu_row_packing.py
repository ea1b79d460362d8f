"""Row transforms and fastconv whose workgroups hold one line, a wave of them and
as many as they ever do (more than 1024 full workgroups, or 256 for one-thread
lines: up to 78 and 86 KB of LDS at 36 and 40 points), each with a last workgroup
that is not full; every line against 64 bits.

Tolerance: rel-L2 1e-6 (8 radix-2 levels a transform at most here, sqrt(2 * 2 * 8) *
6e-8 = 3.4e-7)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (length, lines of the fullest workgroup, workgroups that are to be full)
LENGTHS = [(2, 256, 1024), (8, 256, 1024), (16, 64, 1024), (36, 256, 256), (40, 256, 256), (72, 21, 1024),
           (128, 8, 1024), (160, 16, 1024), (288, 10, 1024)]


@pytest.mark.parametrize("n,most,groups", LENGTHS)
@pytest.mark.parametrize("how", ["one", "some", "full"])
def test_lines_in_a_workgroup(ovx, n, most, groups, how):
    import torch
    rows = {"one": 1, "some": 77, "full": groups * most + 1}[how]
    gen = torch.Generator(device="cuda").manual_seed(n + rows)
    x = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    w = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    x64 = x.cpu().numpy().astype(np.complex128)
    f = np.fft.fft(x64)

    def check(got, want):
        got = got.cpu().numpy()
        assert np.linalg.norm(got - want) < 1e-6 * np.linalg.norm(want)
        assert np.linalg.norm(got[-1] - want[-1]) < 2e-6 * np.linalg.norm(want[-1])

    check(ovx.Fftm(rows, n, ovx.ROW, ovx.FFT_FWD, 1.0)(x), f)
    check(ovx.Fastconv(rows, n)(x, w), np.fft.ifft(f * w.cpu().numpy()))
    real = torch.view_as_real(x).reshape(rows, 2 * n)
    check(ovx.FftmReal(rows, 2 * n, ovx.ROW, ovx.FFT_FWD)(real), np.fft.rfft(x64.view(np.float64)))
