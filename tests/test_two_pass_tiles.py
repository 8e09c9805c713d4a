"""Windows 2^17..2^20: the two-pass path's workgroup sizes and chunks.

A short request runs in workgroups of 256 threads, a long one in workgroups of
512 and in chunks of frames; a frame's arithmetic is the same in all of them,
so every frame of a long request equals, bit for bit, the same frame requested
alone.  The frames alone are held against the FP64 pipeline, cut by the
signal's end at an odd sample, with an odd hop and a misaligned input.

Bar: per-frame relative L2 error <= 1e-6.  A float32 transform of 2^19 points
rounds about 3 times a radix-2 level, 2^-24 rms each at most: sqrt(3 * 20) *
6e-8 = 4.6e-7, twice that for the squares of the power layout.
"""
import numpy as np
import pytest

from conftest import frame_errors

import occastft_amd as ostft

import pyoracle as po

pytestmark = pytest.mark.gpu

LAYOUTS = {"": po.OUT_COMPAT_POWER, "--magnitude_return": po.OUT_MAGNITUDE,
           "--half_complex_return": po.OUT_HALF_COMPLEX, "--power_return": po.OUT_POWER,
           "--half_spectrum_return": po.OUT_HALF_SPECTRUM}


@pytest.fixture(scope="module")
def runner():
    import torch  # ahead of the engine library, which then shares its HIP runtime

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    r = ostft.Runner(0)
    yield r
    r.close()


def _per(layout, n):
    return {"--power_return": n // 2 + 1, "--half_spectrum_return": n + 2}.get(layout, n)


@pytest.mark.parametrize("exp", [17, 18, 19, 20])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_short_request_against_fp64(runner, exp, layout):
    import torch

    n = 1 << exp
    L, ov, offset = n + n // 3 + 1, 0.33, exp % 4
    x = np.random.default_rng(exp).standard_normal(L).astype(np.float32)
    xd = torch.zeros(L + 4, device="cuda")
    xd[offset: offset + L] = torch.from_numpy(x)
    for opts in ("--blackman_window --remove_dc --exact_window", ""):
        p = ostft.parse_options(f"{opts} {layout}", exp, ov)
        g = ostft.geometry(p, L)
        out = torch.full((g["out_floats"] + 4,), float("nan"), device="cuda")
        runner.run_device(xd[offset: offset + L], p, out=out)
        y = out.cpu().numpy()
        assert np.isnan(y[g["out_floats"]:]).all()  # nothing written past the result
        t = po.stft64(x, exp, g["hop"], g["frames"], po.WINDOWS["blackman"] if opts else 0, 0.0, bool(opts),
                      LAYOUTS[layout])
        mx, _, zabs = frame_errors(y[: g["out_floats"]], t[: g["out_floats"]], _per(layout, n))
        assert mx <= 1e-6 and zabs <= 1e-6, (exp, layout, opts, mx, zabs)


@pytest.mark.parametrize("exp,frames", [(17, 50), (17, 300), (18, 25), (19, 13), (20, 7), (20, 37)])
def test_long_request_equals_its_frames_alone(runner, exp, frames):
    import torch

    n = 1 << exp
    hop = n // 4
    x = torch.randn((frames - 1) * hop + n, device="cuda", generator=torch.Generator("cuda").manual_seed(frames))
    layouts = list(LAYOUTS) if frames < 30 else ["--power_return"]
    for layout in layouts:
        p = ostft.parse_options(f"--hanning_window --remove_dc {layout}", exp, 0.75)
        per = _per(layout, n) * (2 if layout == "--half_complex_return" else 1)
        y = runner.run_device(x, p)
        count = frames // 2 if layout == "--half_complex_return" else frames
        for f in sorted({0, 1, count // 3, count // 2, count - 2, count - 1}):
            alone = runner.run_device(x[f * hop: f * hop + n].contiguous(), p)
            assert torch.equal(y[f * per: (f + 1) * per], alone[:per]), (exp, layout, f)


def test_captured_long_request_replays(runner):
    """Two chunks at a time fork to a side stream and join again: also inside a
    captured graph, whose replays follow new inputs and eager work between."""
    import torch

    exp, frames = 17, 620  # 2480 workgroups a pass
    n = 1 << exp
    x = torch.zeros((frames - 1) * (n // 4) + n, device="cuda")
    p = ostft.parse_options("--hanning_window --power_return", exp, 0.75)
    out = torch.empty(ostft.geometry(p, x.numel())["out_floats"], device="cuda")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        runner.run_device(x, p, out=out)  # tables and scratch become resident
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        runner.run_device(x, p, out=out)
    with torch.cuda.stream(s):
        for rep in range(3):
            x.normal_(generator=torch.Generator("cuda").manual_seed(rep))
            out.zero_()
            g.replay()
            got = out.clone()
            want = runner.run_device(x, p)
            s.synchronize()
            assert torch.equal(got, want), rep
