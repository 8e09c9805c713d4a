"""Window 2^16 through two passes (requests of few frames) against the one
kernel that longer requests take, at the edges of the rule, of the workgroup
sizes and of the signal: bitwise, since both do the same arithmetic.  A scratch
budget of one frame keeps a request in the one kernel.  The larger windows'
smallest workgroups against the larger ones likewise."""
import numpy as np
import pytest

import occastft_amd as ostft

pytestmark = pytest.mark.gpu
LAYOUTS = ["", "--magnitude_return", "--half_complex_return", "--power_return", "--half_spectrum_return"]


@pytest.fixture(scope="module")
def runner():
    import torch

    torch.zeros(1, device="cuda")
    with ostft.Runner(0) as r:
        yield r


def _signal(n, offset):
    import torch

    x = np.random.default_rng(n + offset).standard_normal(n + offset).astype(np.float32) + 0.3
    return torch.from_numpy(x).cuda()[offset:]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("L,ov,offset", [(5, 0.0, 0), (65535, 0.5, 3), (1 << 16, 0.0, 0), (300_001, 0.33, 1),
                                         (16 << 16, 0.0, 1), (20 << 16, 0.0, 0), (21 << 16, 0.25, 2),
                                         (55 << 16, 0.0, 0), (56 << 16, 0.0, 3),
                                         (127 << 16, 0.0, 0), (128 << 16, 0.0, 0)])
def test_passes_equal_the_one_kernel(runner, layout, L, ov, offset):
    import torch

    x = _signal(L, offset)
    for opts in ("--blackman_window --remove_dc", "--hanning_window", "--remove_dc", ""):
        p = ostft.parse_options(f"{opts} {layout}", 16, ov)
        got = runner.run_device(x, p).clone()
        before = runner.scratch_budget()
        try:
            runner.scratch_budget(1 << 18)  # one frame
            want = runner.run_device(x, p)
        finally:
            runner.scratch_budget(before)
        assert torch.equal(got, want), opts


def test_every_form_gives_the_same_frames(runner):
    import torch

    x = _signal(7 << 16, 0)
    p = ostft.parse_options("--hanning_window --remove_dc --power_return", 16, 0.5)
    want = runner.run_device(x, p)
    one = runner.run_strided_device(x.view(1, -1), p)
    two = runner.run_strided_device(torch.stack([x, x]), p)  # one launch of the one kernel
    (job,) = runner.run_batch_device([(x, p, None)])
    for got in (one[0], two[0], two[1], job):
        assert torch.equal(got[: want.numel()], want)


def test_captured_call_takes_the_one_kernel():
    """A context that has run only a long request at 2^16 holds neither the
    scratch nor the tables of the two passes: a short one is captured all the
    same, and its replays follow new inputs and eager work between."""
    import torch

    torch.zeros(1, device="cuda")
    with ostft.Runner(0) as r:
        p = ostft.parse_options("--hanning_window --power_return", 16, 0.5)
        r.run_device(_signal(100 << 16, 0), p)
        x = torch.zeros(5 << 16, device="cuda")
        out = torch.zeros(ostft.geometry(p, x.numel())["out_floats"], device="cuda")
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            r.run_device(x, p, out=out)
        for rep in range(3):
            x.normal_(generator=torch.Generator("cuda").manual_seed(rep))
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            got = out.clone()
            assert torch.equal(got, r.run_device(x, p)), rep


@pytest.mark.parametrize("exp,frames", [(17, 10), (18, 5), (19, 2)])
def test_smallest_workgroups_equal_larger_ones(runner, exp, frames):
    """`frames` frames are the most that take 128 threads; the same signal with
    more behind it takes 256, and its first frames are the same bits."""
    import torch

    n = 1 << exp
    x = _signal(2 * frames * n, 0)
    p = ostft.parse_options("--blackman_window --remove_dc", exp, 0.0)
    long = runner.run_device(x, p).clone()
    # overlap 0: a request has one frame more than its signal fills
    short = runner.run_device(x[: (frames - 1) * n].contiguous(), p)
    assert torch.equal(short[: (frames - 1) * n], long[: (frames - 1) * n])
