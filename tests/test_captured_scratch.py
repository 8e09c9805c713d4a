"""Captured requests of the two-pass windows keep a scratch buffer of their own:
replays are right after later calls have outgrown the context's buffer, and
beside calls on other streams, during the capture and after it.  Beyond the
scratch budget a graph uses the context's buffer, which is then not freed.
Every result bitwise that of the request run alone."""
import pytest

import occastft_amd as ostft

pytestmark = pytest.mark.gpu
OPTS = "--hanning_window --remove_dc --power_return"


def _request(r, exp, frames, seed):
    """frames - 1 hops of 75% overlap and a window: bound, and run once."""
    import torch

    n = 1 << exp
    p = ostft.parse_options(OPTS, exp, 0.75)
    x = torch.randn((frames - 4) * (n // 4) + n // 8, device="cuda", generator=torch.Generator("cuda").manual_seed(seed))
    assert ostft.geometry(p, x.numel())["frames"] == frames - 3
    out = torch.zeros(ostft.geometry(p, x.numel())["out_floats"], device="cuda")
    r.run_device(x, p, out=out)
    return x, p, out


def _replay(r, g, requests, seed):
    import torch

    for i, (x, _, out) in enumerate(requests):
        x.normal_(generator=torch.Generator("cuda").manual_seed(seed + i))
        out.zero_()
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    got = [out.clone() for _, _, out in requests]
    for (x, p, _), y in zip(requests, got):
        assert torch.equal(y, r.run_device(x, p)), p.exp


@pytest.mark.parametrize("exp,frames", [(16, 8), (16, 40), (17, 20), (17, 700), (20, 90)])
def test_replays_after_the_contexts_scratch_was_outgrown(exp, frames):
    import torch

    torch.zeros(1, device="cuda")
    with ostft.Runner(0) as r:
        requests = [_request(r, exp, frames, 1), _request(r, exp, frames - 1, 2)]
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for x, p, out in requests:
                r.run_device(x, p, out=out)
        for rep in range(3):
            _request(r, 18, 100 * (rep + 1), 9)  # grows the context's buffer
            if rep == 1:
                before = r.scratch_budget()
                r.scratch_budget(1)  # and gives it back
                r.scratch_budget(before)
            _replay(r, g, requests, 10 * rep)


def test_beside_another_stream():
    """A long request under capture, long requests on another stream meanwhile,
    and replays on one stream while the other runs requests."""
    import torch

    torch.zeros(1, device="cuda")
    with ostft.Runner(0) as r:
        requests = [_request(r, 17, 700, 3), _request(r, 16, 30, 4)]
        x, p, out = _request(r, 18, 300, 5)
        want = out.clone()
        s, other = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s, capture_error_mode="relaxed"):
            r.run_device(*requests[0][:2], out=requests[0][2])
            r.run_device(x, p, out=out, stream=other)
            r.run_device(*requests[1][:2], out=requests[1][2])
        other.synchronize()
        assert torch.equal(out, want)
        alone = [r.run_device(a, b).clone() for a, b, _ in requests]
        for rep in range(4):
            out.zero_()
            for _, _, o in requests:
                o.zero_()
            torch.cuda.synchronize()
            for _ in range(3):
                with torch.cuda.stream(s):
                    g.replay()
                r.run_device(x, p, out=out, stream=other)
            torch.cuda.synchronize()
            assert torch.equal(out, want), rep
            assert all(torch.equal(o, a) for (_, _, o), a in zip(requests, alone)), rep


def test_beyond_the_budget():
    """Captures in turn until the budget is used up, and two more: each graph's
    replays are right, also after the context's buffer was outgrown."""
    import torch

    torch.zeros(1, device="cuda")
    with ostft.Runner(0) as r:
        requests = [_request(r, 17, 20, 6), _request(r, 16, 20, 7)]  # 17 frames: 8.5 MiB and 4.25 MiB
        r.scratch_budget(20 << 20)
        torch.cuda.synchronize()
        graphs = []
        for _ in range(4):
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1]):
                for x, p, out in requests:
                    r.run_device(x, p, out=out)
        for rep in range(2):
            for i, g in enumerate(graphs):
                _replay(r, g, requests, 100 * rep + 10 * i)
            r.scratch_budget(1 << 30)
            _request(r, 18, 200, 8)
