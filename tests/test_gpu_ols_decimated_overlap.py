"""A decimating convolution whose few results are stored over its signal, where
the signal is longer than a segment can be but what the results need is not: each
result lies over samples that another segment reads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,d,at", [(4000, 19000, 10000, 12000), (4000, 19000, 10000, 1000), (3000, 17000, 6500, 7000)])
def test_results_over_a_longer_signal(ovx, m, n, d, at):
    import torch
    rng = np.random.default_rng(m + at)
    taps, x = [(rng.standard_normal(k) + 1j * rng.standard_normal(k)).astype(np.complex64) for k in (m, n)]
    plan = ovx.Convolution(taps, "nonsym", "min", n, d)
    assert n > 16384 and (plan.output_size - 1) * d + m <= 16384
    x64, t64 = x.astype(np.complex128), taps.astype(np.complex128)
    want = np.array([np.dot(t64[::-1], x64[k * d:k * d + m]) for k in range(plan.output_size)])
    signal = torch.from_numpy(x).cuda()
    plan(signal, out=signal[at:at + plan.output_size])
    got = signal[at:at + plan.output_size].cpu().numpy()
    # rel-L2: 14 radix-2 levels a transform, three transforms, over a result
    # whose length is a small part of the segment's: sqrt(2 * 3 * 14) * 6e-8 times
    # sqrt(16384 / 4000) at most
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 2e-6
