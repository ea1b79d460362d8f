"""Calls of one plan on two streams that keep a copy in the plan's buffers: a
convolution or correlation in place over several segments, a correlation whose
reference's spectrum is a launch of its own.  The second call waits for the first
stream's work, and the results are those of calls one after the other.  A
fastconv that would copy its spectra is refused meanwhile."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

N = 800  # two or three segments


def asleep(stream):
    """Keeps the stream at work for some milliseconds."""
    import torch
    with torch.cuda.stream(stream):
        torch.cuda._sleep(20_000_000)


@pytest.mark.parametrize("kind", ["conv", "corr", "corr_reference"])
def test_second_stream_waits(ovx, kind):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(3)
    m = 101 if kind == "corr_reference" else 201
    xs = [torch.randn(N, dtype=torch.complex64, device="cuda", generator=gen) for _ in range(2)]
    refs = [torch.randn(m, dtype=torch.complex64, device="cuda", generator=gen) for _ in range(2)]
    plan = (ovx.Convolution(refs[0].cpu().numpy(), "nonsym", "same", N) if kind == "conv"
            else ovx.Correlation("same", m, N))

    def operands(i):
        """Signal, reference and result: the result over the signal or around the reference."""
        x = xs[i].clone()
        if kind != "corr_reference":
            return x, refs[i], x
        out = torch.zeros_like(x)
        out[50:50 + m] = refs[i]
        return x, out[50:50 + m], out

    def call(x, ref, out):
        plan(x, out=out) if kind == "conv" else plan("biased", ref, x, out=out)

    alone = [operands(i) for i in range(2)]
    for a in alone:
        call(*a)
        torch.cuda.synchronize()
    together = [operands(i) for i in range(2)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    with torch.cuda.stream(streams[0]):
        call(*together[0])
    asleep(streams[0])
    with torch.cuda.stream(streams[1]):
        call(*together[1])
    second = torch.cuda.Event()
    second.record(streams[1])
    early = second.query()
    assert not early or streams[0].query()
    torch.cuda.synchronize()
    for (_, _, a), (_, _, b) in zip(alone, together):
        assert torch.equal(a, b)


def test_fastconv_copy_refused_meanwhile(ovx):
    import torch
    n, rows = 2048, 4
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen)
    room = torch.randn(rows + 1, n, dtype=torch.complex64, device="cuda", generator=gen)
    plan = ovx.Fastconv(rows, n)
    want = plan(x, room[1:].clone())
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]

    def call(w, y, stream):
        return ovx._lib.lib().ovx_fastconv_exec(
            plan._h, ctypes.c_void_p(x.data_ptr()), n, ctypes.c_void_p(w.data_ptr()), n,
            ctypes.c_void_p(y.data_ptr()), n, rows, ctypes.c_void_p(stream.cuda_stream))

    other = room.clone()
    torch.cuda.synchronize()
    assert call(room[1:], room[:-1], streams[0]) == 0
    asleep(streams[0])
    refused = call(other[1:], other[:-1], streams[1])
    assert refused or streams[0].query()
    torch.cuda.synchronize()
    assert torch.equal(room[:-1], want)
