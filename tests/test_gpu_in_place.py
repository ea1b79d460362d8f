"""Transforms in place on both sides of the sizes at which their loads (rows) or
stores (four-step) change between ordinary and non-temporal ones, both
directions: the same floats as out of place."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rows", [(64, 100), (192, 300), (256, 300), (1024, 3840), (1024, 3841), (6144, 640), (6144, 641), (8192, 20),
                                    (2048, 7679), (2048, 7680), (16384, 959), (16384, 960), (65536, 39),
                                    (65536, 40), (131072, 64), (131072, 65), (262144, 10), (1 << 20, 3), (1 << 21, 4)])
@pytest.mark.parametrize("inverse", [False, True])
def test_in_place_equals_out_of_place(ovx, n, rows, inverse):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(n + rows)
    x = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    plan = ovx.Fftm(rows, n, ovx.ROW, ovx.FFT_INV if inverse else ovx.FFT_FWD, 1.0 / n if inverse else 1.0)
    want = plan(x)
    plan(x, out=x)
    assert torch.equal(x, want)
