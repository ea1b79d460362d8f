"""Spectra whose rows lie between the result's rows (the halves of one wide
matrix): they share no memory, so the call copies nothing and takes no buffer of
the plan's, and gives what it gives with the spectra elsewhere."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rows", [(64, 70), (2048, 5), (3072, 3), (8192, 4), (16384, 3)])
@pytest.mark.parametrize("split", [False, True])
def test_no_copy_for_spectra_beside_the_result(ovx, n, rows, split):
    import torch
    lib = ovx._lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(n)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    dtype = torch.float32 if split else torch.complex64

    def p(t):
        return ctypes.c_void_p(t.data_ptr())

    def call(fc, x, w, y):
        if split:
            return lib.ovx_fastconv_split_exec(fc._h, p(x[0]), p(x[1]), x[0].stride(0), p(w[0]), p(w[1]),
                                               w[0].stride(0), p(y[0]), p(y[1]), y[0].stride(0), rows, stream)
        return lib.ovx_fastconv_exec(fc._h, p(x[0]), x[0].stride(0), p(w[0]), w[0].stride(0), p(y[0]),
                                     y[0].stride(0), rows, stream)

    parts = 2 if split else 1
    wide = torch.randn(rows, 2 * parts * n, dtype=dtype, device="cuda", generator=gen)
    x = [torch.randn(rows, n, dtype=dtype, device="cuda", generator=gen) for _ in range(parts)]
    w = [wide[:, 2 * k * n:(2 * k + 1) * n] for k in range(parts)]
    y = [wide[:, (2 * k + 1) * n:(2 * k + 2) * n] for k in range(parts)]
    apart_w, apart_y = [t.contiguous() for t in w], [torch.empty_like(t) for t in x]
    fc = ovx.Fastconv(rows, n)
    assert call(fc, x, apart_w, apart_y) == 0
    before = lib.ovx_plan_device_bytes(fc._h)
    assert call(fc, x, w, y) == 0
    assert lib.ovx_plan_device_bytes(fc._h) == before
    for a, b, ww, copy in zip(y, apart_y, w, apart_w):
        assert torch.equal(a, b) and torch.equal(ww, copy)
