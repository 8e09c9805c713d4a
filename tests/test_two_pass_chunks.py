"""Windows 2^17..2^20: requests of more than 2304 workgroups a pass (4096 for most
layouts at 2^20), whose chunks of
frames run two at a time on two streams, and chunks of any scratch budget.

A frame's result does not depend on its chunk, so every frame of a long request
equals, bit for bit, the same frame requested alone (test_two_pass_tiles.py
holds those against FP64), and the whole result is the same under every budget:
one frame, a few, just below two chunks of 64 MiB, and chunks that do not divide
the request.  Requests queued alternately on two streams, long ones (with their
side stream) and short ones, take turns on the one scratch buffer."""
import pytest

import occastft_amd as ostft

pytestmark = pytest.mark.gpu
LAYOUTS = ["", "--magnitude_return", "--half_complex_return", "--power_return", "--half_spectrum_return"]
MiB = 1 << 20


@pytest.fixture(scope="module")
def runner():
    import torch  # ahead of the engine library, which then shares its HIP runtime

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    r = ostft.Runner(0)
    yield r
    r.close()


def _signal(exp, frames, seed):
    """75% overlap: `frames` frames, the last four cut by the signal's end or beyond it."""
    import torch

    hop = 1 << (exp - 2)
    return torch.randn((frames - 1) * hop + 333, device="cuda", generator=torch.Generator("cuda").manual_seed(seed))


def _run(runner, x, p):
    """The result, and that nothing is written past it."""
    import torch

    n = ostft.geometry(p, x.numel())["out_floats"]
    out = torch.full((n + 4,), float("nan"), device="cuda")
    runner.run_device(x, p, out=out)
    assert bool(out[n:].isnan().all()) and not bool(out[:n].isnan().any())
    return out[:n]


@pytest.mark.parametrize("exp,frames", [(17, 1161), (18, 581), (19, 301), (20, 151)])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_long_request_equals_its_frames_alone(runner, exp, frames, layout):
    import torch

    n, hop = 1 << exp, 1 << (exp - 2)
    x = _signal(exp, frames, frames)
    p = ostft.parse_options(f"--blackman_window --remove_dc {layout}", exp, 0.75)
    g = ostft.geometry(p, x.numel())
    assert g["frames"] == frames
    count = g["compute_frames"]  # complex half: half the frames, the last one cut in its middle
    assert (count << (exp - 1)) > 2304 * 16384
    per = g["out_floats"] // frames if layout != "--half_complex_return" else 2 * n
    y = _run(runner, x, p)
    picks = {0, 1, 127, 128, 129, count // 2, count // 2 + 1, *range(count - 6, count)}
    for f in sorted(f for f in picks if 0 <= f < count):
        alone = runner.run_device(torch.nn.functional.pad(x[f * hop: f * hop + n], (0, max(0, f * hop + n - x.numel()))), p)
        want = alone[: min(per, y.numel() - f * per)]
        assert torch.equal(y[f * per: f * per + want.numel()], want), f


@pytest.mark.parametrize("exp,frames,layout", [(17, 1161, "--half_complex_return"), (17, 700, "--power_return"),
                                               (18, 300, ""), (19, 150, "--half_complex_return"),
                                               (20, 137, "--half_spectrum_return")])
def test_every_budget_gives_the_same(runner, exp, frames, layout):
    import torch

    x = _signal(exp, frames, exp)
    p = ostft.parse_options(f"--hanning_window --remove_dc {layout}", exp, 0.75)
    frame = 8 << (exp - 1)
    before = runner.scratch_budget()
    want = _run(runner, x, p)
    try:
        for budget in (1, frame, 3 * frame + 1, 37 * MiB, 128 * MiB - 1, 128 * MiB, 144 * MiB):
            assert runner.scratch_budget(budget) == budget
            assert torch.equal(_run(runner, x, p), want), budget
    finally:
        runner.scratch_budget(before)


@pytest.mark.parametrize("budget", [1 << 30, 128 * MiB - 1, 16 * MiB])
def test_requests_on_two_streams_take_turns(runner, budget):
    import torch

    sizes = [(17, 700), (18, 20), (18, 320), (16, 30), (20, 80), (17, 5), (19, 150)]
    work = []
    for i, (exp, frames) in enumerate(sizes):
        p = ostft.parse_options("--hanning_window --remove_dc --power_return", exp, 0.75)
        x = _signal(exp, frames, i)
        work.append((x, p, runner.run_device(x, p).clone()))
    before = runner.scratch_budget()
    outs = [[torch.zeros_like(w) for _, _, w in work] for _ in range(3)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    try:
        runner.scratch_budget(budget)
        for k, row in enumerate(outs):  # each request on the one stream and then on the other
            for i, ((x, p, _), out) in enumerate(zip(work, row)):
                runner.run_device(x, p, out=out, stream=streams[(i + k) % 2])
        torch.cuda.synchronize()
    finally:
        runner.scratch_budget(before)
    for row in outs:
        for (_, p, want), out in zip(work, row):
            assert torch.equal(out, want), p.exp


def test_one_frame_in_the_one_kernel_and_in_passes(runner):
    """Window 2^16: a set of two signals runs in the one kernel always, a request
    of one frame in two passes."""
    import torch

    for layout in LAYOUTS:
        for n in (5, 65535, 1 << 15):
            p = ostft.parse_options(f"--blackman_window --remove_dc {layout}", 16, 0.0)
            x = torch.randn(2, n, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
            assert ostft.geometry(p, n)["compute_frames"] == 1
            two = runner.run_strided_device(x, p)
            for i in range(2):
                one = runner.run_device(x[i].contiguous(), p)
                assert torch.equal(one, two[i][: one.numel()]), (layout, n)
