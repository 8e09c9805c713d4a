"""ostft_run_device_noalloc at window 2^16, requests of few frames: through the
two passes where an earlier call left scratch and tables for them, through the
one kernel else and under capture.  Bitwise ostft_run_device's result in every
form, no device memory taken, and right on two streams at once."""
import ctypes

import pytest

import occastft_amd as ostft
from occastft_amd import _native as N

pytestmark = pytest.mark.gpu
LAYOUTS = ["", "--half_complex_return", "--power_return"]


def _noalloc(r, x, p, out, stream=None):
    import torch

    s = (stream or torch.cuda.current_stream()).cuda_stream
    rc = N.lib().ostft_run_device_noalloc(r._h, ctypes.byref(p), x.data_ptr(), x.numel(), out.data_ptr(), out.numel(), s)
    assert rc == N.OK, r.last_error


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("prepared", ["same request", "fewer frames", "long request only", "budget of one frame"])
def test_equals_run_device(layout, prepared):
    import torch

    x = torch.randn((20 << 16) + 77, device="cuda")
    p = ostft.parse_options(f"--hanning_window --remove_dc {layout}", 16, 0.25)
    with ostft.Runner(0) as other:
        want = other.run_device(x, p)
    with ostft.Runner(0) as r:
        if prepared == "long request only":
            r.run_device(torch.zeros(100 << 16, device="cuda"), p)
        else:
            r.run_device(x if prepared == "same request" else x[: 2 << 16], p)
        if prepared == "budget of one frame":
            r.scratch_budget(1 << 18)
        out = torch.full((want.numel() + 4,), float("nan"), device="cuda")
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        _noalloc(r, x, p, out)
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] >= free - (2 << 20)  # a kernel's first launch loads its code
        assert torch.equal(out[: want.numel()], want)
        assert bool(out[want.numel():].isnan().all())


def test_two_streams_and_capture():
    import torch

    torch.zeros(1, device="cuda")
    p = ostft.parse_options("--blackman_window --power_return", 16, 0.5)
    with ostft.Runner(0) as r:
        xs = [torch.randn((12 + i) << 16, device="cuda") for i in range(4)]
        want = [r.run_device(x, p).clone() for x in xs]
        outs = [torch.zeros_like(w) for w in want]
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        torch.cuda.synchronize()
        for _ in range(5):
            for i in range(4):
                _noalloc(r, xs[i], p, outs[i], streams[i % 2])
        torch.cuda.synchronize()
        assert all(torch.equal(o, w) for o, w in zip(outs, want))
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for i in range(4):
                _noalloc(r, xs[i], p, outs[i])
        for rep in range(3):
            for o in outs:
                o.zero_()
            g.replay()
            r.run_device(xs[0], p)
            torch.cuda.synchronize()
            assert all(torch.equal(o, w) for o, w in zip(outs, want)), rep
