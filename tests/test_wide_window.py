"""Window 2^16: one workgroup per frame, the transform in its registers
(fused_wide.hip).  Every frame against the FP64 pipeline at the edges of what
the kernel distinguishes: frames inside the signal, cut by its end (at an even
and an odd sample) and past it, odd hops and misaligned inputs, every layout,
and several signals in a launch.

Bar: per-frame relative L2 error <= 1e-6.  A float32 transform of 2^15 points
rounds about 3 times a radix-2 level, 2^-24 rms each at most: sqrt(3 * 16) *
6e-8 = 4.1e-7, twice that for the squares of the power layout.
"""
import numpy as np
import pytest

from conftest import frame_errors

import occastft_amd as ostft

import pyoracle as po

pytestmark = pytest.mark.gpu

N_ = 1 << 16
LAYOUTS = {"": (po.OUT_COMPAT_POWER, N_), "--magnitude_return": (po.OUT_MAGNITUDE, N_),
           "--half_complex_return": (po.OUT_HALF_COMPLEX, N_), "--power_return": (po.OUT_POWER, N_ // 2 + 1),
           "--half_spectrum_return": (po.OUT_HALF_SPECTRUM, N_ + 2)}


@pytest.fixture(scope="module")
def runner():
    import torch  # ahead of the engine library, which then shares its HIP runtime

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    r = ostft.Runner(0)
    yield r
    r.close()


def _check(runner, L, ov, layout, opts, offset, seed):
    import torch

    mode, per = LAYOUTS[layout]
    x = np.random.default_rng(seed).standard_normal(L).astype(np.float32)
    xd = torch.zeros(L + 4, device="cuda")
    xd[offset: offset + L] = torch.from_numpy(x)
    p = ostft.parse_options(f"{opts} {layout} --exact_window", 16, ov)
    g = ostft.geometry(p, L)
    out = torch.full((g["out_floats"] + 4,), float("nan"), device="cuda")
    runner.run_device(xd[offset: offset + L], p, out=out)
    y = out.cpu().numpy()
    assert np.isnan(y[g["out_floats"]:]).all()  # nothing written past the result
    window = po.WINDOWS["blackman"] if "--blackman_window" in opts else 0
    t = po.stft64(x, 16, g["hop"], g["frames"], window, 0.0, "--remove_dc" in opts, mode)
    mx, _, zabs = frame_errors(y[: g["out_floats"]], t[: g["out_floats"]], per)
    assert mx <= 1e-6 and zabs <= 1e-6, (L, ov, layout, opts, offset, mx, zabs)


@pytest.mark.parametrize("layout", list(LAYOUTS))
@pytest.mark.parametrize("L,ov,offset", [(2 * N_, 0.0, 0), (3 * N_ + 4097, 0.33, 1), (N_ - 1, 0.5, 3), (5, 0.0, 0)])
def test_frames_at_the_signals_end(runner, layout, L, ov, offset):
    for opts in ("--blackman_window --remove_dc", "--remove_dc", ""):
        _check(runner, L, ov, layout, opts, offset, L + offset)


def test_strided_batch_and_noalloc_forms_equal_one_request(runner):
    import ctypes

    import torch

    from occastft_amd import _native as N

    L, count = 2 * N_ + 77, 3
    x = torch.randn(count, L, device="cuda", generator=torch.Generator("cuda").manual_seed(9))
    p = ostft.parse_options("--hanning_window --remove_dc --half_spectrum_return", 16, 0.5)
    one = [runner.run_device(x[i].contiguous(), p).cpu() for i in range(count)]
    strided = runner.run_strided_device(x, p).cpu()
    batch = runner.run_batch_device([(x[i].contiguous(), p, None) for i in range(count)])
    out = torch.empty_like(one[0], device="cuda")
    for i in range(count):
        assert torch.equal(one[i], strided[i]) and torch.equal(one[i], batch[i].cpu())
        rc = N.lib().ostft_run_device_noalloc(runner._h, ctypes.byref(p), ctypes.c_void_p(x[i].data_ptr()), L,
                                              ctypes.c_void_p(out.data_ptr()), out.numel(),
                                              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == N.OK and torch.equal(one[i], out.cpu())
