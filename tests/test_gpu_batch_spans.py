"""Batches and server batches of many small jobs: more spans in a queue than a
wave reads at once (64, 128 and beyond), four-step jobs whose rows leave every
remainder of eight and of the middle pass's rows per tile, jobs of one row.
Each job's result equals its standalone call bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHORT = [512, 1024, 2048, 3072, 4096, 6144, 8192, 12288, 16384]
LONG = [65536, 131072, 262144]


def job_list(count, long_every):
    rng = np.random.default_rng(count)
    return [(LONG[i // long_every % 3] if i % long_every == 0 else SHORT[int(rng.integers(len(SHORT)))],
             1 + i % 19) for i in range(count)]


@pytest.mark.parametrize("count,long_every", [(1, 2), (64, 70), (65, 9), (129, 2), (300, 40)])
def test_many_jobs(ovx, count, long_every):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(count)
    jobs = job_list(count, long_every)
    reps = {n: ovx.Replica(n, np.random.default_rng(n).standard_normal(2 * n).astype(np.float32).view(np.complex64))
            for n, _ in jobs}
    xs = [torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen) for n, rows in jobs]
    ys = [torch.zeros_like(x) for x in xs]
    batch = ovx.Batch()
    for (n, _), x, y in zip(jobs, xs, ys):
        batch.add(x, reps[n], y)
    batch.commit()
    batch()
    torch.cuda.synchronize()
    alone = [torch.zeros_like(x) for x in xs]
    for (n, rows), x, y in zip(jobs, xs, alone):
        b = ovx.Batch()
        b.add(x, reps[n], y)
        b.commit()
        b()
    torch.cuda.synchronize()
    for job, a, b in zip(jobs, ys, alone):
        assert torch.equal(a, b), job
    # every job against FP64 on its last row (rel-L2: 18 radix-2 levels a transform
    # at most, sqrt(2) * 2 * sqrt(18) * 6e-8 = 7.2e-7)
    for (n, _), x, y in list(zip(jobs, xs, ys))[::7]:
        w = np.random.default_rng(n).standard_normal(2 * n).astype(np.float32).view(np.complex64).astype(np.complex128)
        want = np.fft.ifft(np.fft.fft(x[-1].cpu().numpy().astype(np.complex128)) * np.fft.fft(w))
        got = y[-1].cpu().numpy()
        assert np.linalg.norm(got - want) / np.linalg.norm(want) < 1e-6


@pytest.mark.parametrize("count", [5, 70, 200])
def test_server_many_requests(ovx, count):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(count)
    jobs = job_list(count, 6)
    reps = {n: ovx.Replica(n, np.random.default_rng(n).standard_normal(2 * n).astype(np.float32).view(np.complex64))
            for n, _ in jobs}
    xs = [torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen) for n, rows in jobs]
    ys = [torch.zeros_like(x) for x in xs]
    # every fourth request is a forward transform; the long ones among them use
    # the server's workspace
    req = [ovx.fftm_request(x, y) if i % 4 == 0 else ovx.fastconv_request(x, reps[n], y)
           for i, ((n, _), x, y) in enumerate(zip(jobs, xs, ys))]
    torch.cuda.synchronize()
    ovx.Server(workspace_mb=512).run_trace(req)
    plain = [torch.zeros_like(x) for x in xs]
    req = [ovx.fftm_request(x, y) if i % 4 == 0 else ovx.fastconv_request(x, reps[n], y)
           for i, ((n, _), x, y) in enumerate(zip(jobs, xs, plain))]
    torch.cuda.synchronize()
    ovx.Server(workspace_mb=512, plain=True).run_trace(req)
    for job, a, b in zip(jobs, ys, plain):
        assert torch.equal(a, b), job
