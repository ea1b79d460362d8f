"""A job's result in a batch is bitwise that of a plan made for it without a
variant: at every length whose default configurations have tiles, on both sides
of the row counts at which the default changes (1024 points: 256 rows, 2048:
1024), with jobs of several lengths in one batch."""
import pytest

pytestmark = pytest.mark.gpu

JOBS = [(256, 1), (256, 700), (512, 3), (512, 2500), (1024, 1), (1024, 64), (1024, 256), (1024, 257), (1024, 1000),
        (2048, 2), (2048, 300), (2048, 1024), (2048, 1025), (3072, 5), (4096, 37), (8192, 9), (8192, 300), (16384, 3),
        (65536, 2), (131072, 3)]


@pytest.mark.parametrize("mixed", [False, True])
def test_job_equals_its_default_plan(ovx, mixed):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(7)
    xs = [torch.randn(rows, n, dtype=torch.complex64, device="cuda", generator=gen) for n, rows in JOBS]
    spectra = {n: torch.randn(n, dtype=torch.complex64, device="cuda", generator=gen) for n, _ in JOBS}
    reps = {n: ovx.Replica(n, w.cpu().numpy(), is_spectrum=True) for n, w in spectra.items()}
    ys = [torch.zeros_like(x) for x in xs]
    batches = []
    for (n, _), x, y in zip(JOBS, xs, ys):
        if not mixed or not batches:
            batches.append(ovx.Batch())
        batches[-1].add(x, reps[n], y)
    for b in batches:
        b.commit()
        b()
    torch.cuda.synchronize()
    variants = [v for b in batches for v in b.job_variants()]
    for (n, rows), x, y, v in zip(JOBS, xs, ys, variants):
        tuned = ovx.tuned_variant(n, rows) >= 0 or (n in (2048, 4096) and v == 0)
        plan = ovx.Fastconv(rows, n, variant=v) if tuned else ovx.Fastconv(rows, n)
        alone = plan.with_replica(x, reps[n])
        assert torch.equal(alone, y), (n, rows, v)
