"""One-pass real <-> complex rows (half-length line in registers, the pair
pass on one LDS exchange): the smallest and largest lines, odd half lengths
(no middle value), lines of part of a wavefront, of one and of several, row
counts that leave a workgroup's last lines empty, padded strides on both
sides, interleaved and split, against the FP64 oracle.

Tolerance: rel-L2 <= 1e-6.  Each of the log2(n) <= 15 levels of an FP32
transform adds a relative error of at most a few 2^-24 = 6e-8 that grows with
the square root of their number: sqrt(15) * 2 * 6e-8 = 4.6e-7, twice that as
the bar."""
import ctypes

import numpy as np
import pytest

import oracle as o

pytestmark = pytest.mark.gpu

REL_L2 = 1e-6

# half lengths: 2, 3, 5, 9 (one thread a line), 64 and 48 (part of a wave), 1024
# and 1536 (one wave), 2304, 8192, 16384 (several)
CASES = [(4, 5), (6, 3), (10, 4), (18, 1), (96, 33), (128, 70), (2048, 9), (3072, 7), (4608, 3), (16384, 5),
         (32768, 2)]


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _stream():
    import torch
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("pad", [0, 6])
@pytest.mark.parametrize("n,rows", CASES)
def test_real_rows_both_ways(ovx, n, rows, pad):
    import torch
    from openvsip_amd import _lib
    rng = np.random.default_rng(n + rows + pad)
    h = n // 2
    x = rng.standard_normal((rows, n + pad)).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    y = torch.full((rows, h + 1 + pad), 7.0, dtype=torch.complex64, device="cuda")
    fwd = ovx.FftmReal(rows, n, scale=0.5)
    fwd(xd[:, :n], out=y[:, : h + 1])
    want = 0.5 * o.rfftm64(x[:, :n])
    got = y.cpu().numpy()
    assert o.rel_l2(got[:, : h + 1], want) < REL_L2
    assert np.all(got[:, h + 1:] == 7.0)

    re, im = (torch.full((rows, h + 1 + pad), 7.0, device="cuda") for _ in range(2))
    _lib.check(_lib.lib().ovx_fftm_r2c_split(fwd._h, _p(xd), n + pad, 1, _p(re), _p(im), h + 1 + pad, 1, rows, n,
                                             _stream()))
    assert torch.equal(torch.complex(re, im)[:, : h + 1], y[:, : h + 1])
    assert bool((re[:, h + 1:] == 7).all()) and bool((im[:, h + 1:] == 7).all())

    inv = ovx.FftmReal(rows, n, direction=ovx.FFT_INV, scale=1.0 / n)
    back = torch.full((rows, n + pad), 7.0, device="cuda")
    inv(y[:, : h + 1], out=back[:, :n])
    assert o.rel_l2(back.cpu().numpy()[:, :n], o.irfftm64(got[:, : h + 1], n, scale=1.0 / n)) < REL_L2
    assert bool((back[:, n:] == 7).all())
    b2 = torch.full((rows, n + pad), 7.0, device="cuda")
    _lib.check(_lib.lib().ovx_fftm_c2r_split(inv._h, _p(re), _p(im), h + 1 + pad, 1, _p(b2), n + pad, 1, rows, n,
                                             _stream()))
    assert torch.equal(b2, back)
