"""Error of the large windows against FP64 on noise, power layout.

Bar: the relative error over all values of the form these kernels replaced (two
passes of radix 16 in LDS, twiddles with at most three chained roundings), which
it had measured for the same requests with 12 seeds, alike to the third digit:
2.57e-7 at 2^16, 2.64e-7, 2.77e-7, 2.84e-7 and 3.05e-7 at 2^17..2^20.  A second
step's twiddle as the product of two rounded factors gave 2.82e-7, 2.90e-7 and
2.97e-7 at 2^17..2^19."""
import math

import pytest

import occastft_amd as ostft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exp,bar", [(16, 2.57e-7), (17, 2.64e-7), (18, 2.77e-7), (19, 2.84e-7), (20, 3.05e-7)])
def test_no_further_from_fp64_than_before(exp, bar):
    import torch

    n, hop, size = 1 << exp, 1 << (exp - 1), 1 << 23
    x = torch.randn(size, device="cuda", generator=torch.Generator("cuda").manual_seed(exp))
    with ostft.Runner(0) as r:
        p = ostft.parse_options("--blackman_window --remove_dc --exact_window --power_return", exp, 0.5)
        y = r.run_device(x, p).view(-1, n // 2 + 1).double()
    k = torch.arange(n, dtype=torch.float64, device="cuda") * (2 * math.pi / n)
    window = 0.42 - 0.5 * torch.cos(k) + 0.08 * torch.cos(2 * k)
    frames = torch.nn.functional.pad(x, (0, n)).double().unfold(0, n, hop)[: y.shape[0]] * window
    z = torch.fft.rfft(frames - frames.mean(dim=1, keepdim=True))
    want = z.real.square() + z.imag.square()
    assert ((y - want).norm() / want.norm()).item() <= bar
