"""The fastconv without allocation where the spectra share memory with the
result, each row's with another row's result: up to the lent scratch it copies
them first and equals the allocating call, beyond it is refused and writes
nothing."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

VALUES = (4 << 20) // 8  # OVX_NOALLOC_SCRATCH_BYTES


@pytest.mark.parametrize("n,rows", [(2048, 256), (2048, 257), (8192, 64), (8192, 65), (16384, 33), (64, 8193)])
def test_spectra_over_other_rows_results(ovx, n, rows):
    import torch
    lib = ovx._lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(n + rows)
    x = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    room = torch.randn(rows + 1, n, dtype=torch.complex64, device="cuda", generator=gen)
    other = room.clone()
    kept = room.clone()
    fc = ovx.Fastconv(rows, n)
    want = fc(x, other[1:], out=other[:-1])
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    st = lib.ovx_fastconv_exec_noalloc(fc._h, ctypes.c_void_p(x.data_ptr()), n, ctypes.c_void_p(room[1:].data_ptr()),
                                       n, ctypes.c_void_p(room.data_ptr()), n, rows, stream)
    torch.cuda.synchronize()
    if rows * n <= VALUES:
        assert st == 0 and torch.equal(room[:-1], want)
    else:
        with pytest.raises(RuntimeError):
            ovx._lib.check(st)
        assert torch.equal(room, kept)
    apart = fc(x, kept[1:].clone())
    assert torch.equal(want, apart)
