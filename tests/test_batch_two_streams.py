"""Large batches run their window sizes on two streams (from five sizes, 32768
tiles, and 128 a request): every request bitwise as run alone, run three times in a row
(both descriptor blocks, and one again) and followed, with no wait, by a batch
that overwrites the inputs; and inside a graph capture, with a large batch on
another stream of the same context meanwhile."""
import pytest

import occastft_amd as ostft

pytestmark = pytest.mark.gpu
# a tile of 256 threads is 32, 16, 8, 4, 2 or 1 frames, at 75% overlap always 2048 samples apart
EXPS = (8, 9, 10, 11, 12, 13)
TILE_HOP = 2048


@pytest.fixture(scope="module")
def runner():
    import torch  # ahead of the engine library, which then shares its HIP runtime

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    r = ostft.Runner(0)
    yield r
    r.close()


def _batch(exps, seed, tiles=33000):
    """Requests of `exps` with outputs bound, `tiles` tiles in all."""
    import torch

    gen = torch.Generator("cuda").manual_seed(seed)
    opts = ["--hanning_window --remove_dc --power_return", "--blackman_window --half_spectrum_return"]
    jobs = []
    for i, exp in enumerate(exps):
        n = (tiles // len(exps) + 1) * TILE_HOP + 13 * i
        p = ostft.parse_options(opts[i % 2], exp, 0.75)
        x = torch.randn(n, device="cuda", generator=gen)
        jobs.append((x, p, torch.zeros(ostft.geometry(p, n)["out_floats"], device="cuda")))
    assert sum((ostft.geometry(p, x.numel())["frames"] << p.exp) // (4 * TILE_HOP) for x, p, _ in jobs) >= 32768
    return jobs


@pytest.mark.parametrize("persistent", [False, True])
def test_every_request_as_alone(runner, persistent):
    import torch

    jobs = _batch(EXPS * 2, 1)
    want = [runner.run_device(x, p).clone() for x, p, _ in jobs]
    # outputs of the batch behind: the inputs of this one
    y = torch.randn(1 << 23, device="cuda")
    over = [(y, ostft.parse_options("--power_return", 8, 0.0), x) for x, _, _ in jobs]
    over_want = runner.run_device(*over[0][:2]).clone()
    runner.run_batch_device([(y, p, None) for _, p, _ in over])  # its tables become resident
    if persistent:
        for exp in EXPS:
            runner.batch_config(exp, blocks_per_cu=2)
    torch.cuda.synchronize()
    try:
        for _ in range(3):
            runner.run_batch_device(jobs)
        runner.run_batch_device(over)
    finally:
        for exp in EXPS:
            runner.batch_config(exp, blocks_per_cu=-1)
    torch.cuda.synchronize()
    for (x, p, out), w in zip(jobs, want):
        assert torch.equal(out, w), p.exp
        assert torch.equal(x[: over_want.numel()], over_want)


def test_captured_beside_another_streams_batch(runner):
    """The side stream of a batch under capture is not the one that a batch on
    another stream forks meanwhile; the next capture takes it over."""
    import torch

    captured, eager = _batch(EXPS, 2), _batch(EXPS[::-1] * 2, 3)
    runner.batch_config(use_graphs=0)  # a batch of many sizes may be captured
    want = [runner.run_device(x, p).clone() for x, p, _ in eager]
    for jobs in (captured, eager):
        runner.run_batch_device(jobs)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    graphs = []
    for _ in range(2):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], capture_error_mode="relaxed"):
            runner.run_batch_device(captured)
            runner.run_batch_device(eager, stream=other)
            runner.run_batch_device(captured)
        other.synchronize()
        for (_, p, out), w in zip(eager, want):
            assert torch.equal(out, w), p.exp
            out.zero_()
    for rep in range(4):
        for i, (x, _, out) in enumerate(captured):
            x.normal_(generator=torch.Generator("cuda").manual_seed(10 * rep + i))
            out.zero_()
        graphs[rep % 2].replay()
        torch.cuda.synchronize()
        for x, p, out in captured:
            assert torch.equal(out, runner.run_device(x, p)), (rep, p.exp)
        assert all(int(out.count_nonzero()) == 0 for _, _, out in eager)
    runner.batch_config(use_graphs=1)
