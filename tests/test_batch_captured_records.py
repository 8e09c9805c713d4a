"""A captured batch of one or two window sizes keeps request records of its own:
its replays follow new inputs whatever batches ran in between, also larger ones
(for which the ordinary records and descriptor blocks are allocated anew), and
write nothing but their own outputs.  Beyond the bound on kept records a
captured batch is a launch per request.  Every result is compared, bitwise,
with the request run alone."""
import pytest

import occastft_amd as ostft

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def runner():
    import torch  # ahead of the engine library, which then shares its HIP runtime

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    r = ostft.Runner(0)
    yield r
    r.close()


def _jobs(runner, sizes, seed):
    """Requests with outputs bound, run once (tables become resident)."""
    import torch

    gen = torch.Generator("cuda").manual_seed(seed)
    opts = ["--power_return", "--hanning_window --remove_dc", "--half_spectrum_return --blackman_window"]
    jobs = []
    for i, (exp, n) in enumerate(sizes):
        p = ostft.parse_options(opts[i % 3], exp, 0.5)
        x = torch.randn(n, device="cuda", generator=gen)
        jobs.append((x, p, torch.zeros(max(ostft.geometry(p, n)["out_floats"], 4), device="cuda")))
    runner.run_batch_device(jobs)
    return jobs


def _check(runner, jobs):
    import torch

    for x, p, out in jobs:
        want = runner.run_device(x, p)
        assert torch.equal(out[: want.numel()], want), (p.exp, x.numel())


@pytest.mark.parametrize("persistent", [False, True])
@pytest.mark.parametrize("sizes", [[(10, 30_000), (10, 1), (10, 77_777)], [(8, 50_001), (12, 90_000), (8, 300)]])
def test_replays_do_not_depend_on_later_batches(sizes, persistent):
    import torch

    torch.zeros(1, device="cuda")
    with ostft.Runner(0) as r:
        if persistent:
            for exp in {e for e, _ in sizes}:
                r.batch_config(exp, blocks_per_cu=2)
        jobs = _jobs(r, sizes, 1)
        others = [_jobs(r, [(8, 2000)], 2), _jobs(r, [(e, 40_000 + 7 * i) for i, e in enumerate([8, 10, 12] * 20)], 3),
                  _jobs(r, [(9, 3000)] * 600, 4)]
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            r.run_batch_device(jobs)
        for rep in range(4):
            # more records and longer tile tables than any batch before
            others.append(_jobs(r, [(6, 30_000 * (rep + 1))] * (700 * (rep + 1)) if rep < 2 else [(7, 999)], 10 + rep))
            for other in others:
                r.run_batch_device(other)
            for other in others:
                for _, _, out in other:
                    out.fill_(-7.0)
            for x, _, out in jobs:
                x.normal_(generator=torch.Generator("cuda").manual_seed(100 + rep))
                out.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            _check(r, jobs)
            assert all(bool((out == -7.0).all()) for other in others for _, _, out in other)
            others[-1:] = []


def test_captured_batches_beyond_the_kept_records(runner):
    """300 batches in one graph: the last ones are launches per request."""
    import torch

    batches = [_jobs(runner, [(7, 500 + i), (11, 5000 + 3 * i)], i) for i in range(300)]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for jobs in batches:
            runner.run_batch_device(jobs)
    for rep in range(2):
        for jobs in batches:
            for x, _, out in jobs:
                x.normal_(generator=torch.Generator("cuda").manual_seed(rep))
                out.zero_()
        g.replay()
        torch.cuda.synchronize()
        for jobs in batches:
            _check(runner, jobs)


def test_ordinary_batches_go_on_after_a_capture(runner):
    """The two blocks of ordinary batches are not part of the graph."""
    import torch

    captured = _jobs(runner, [(9, 10_000), (13, 60_000)], 5)
    jobs = _jobs(runner, [(10, 20_000), (11, 30_000), (12, 40_000)], 6)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        runner.run_batch_device(captured)
    for rep in range(3):  # both blocks, and one again
        for x, _, out in jobs:
            x.normal_(generator=torch.Generator("cuda").manual_seed(rep))
            out.zero_()
        g.replay()
        runner.run_batch_device(jobs)
        torch.cuda.synchronize()
        _check(runner, jobs)
