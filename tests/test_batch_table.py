"""The tile table that the batch's fill kernel writes: one request of many tiles
(its entries split over several workgroups), many requests of one tile each,
and sizes of every class in one batch, against each request run alone, bitwise
(the same kernels; a wrong table entry runs another request's frames)."""
import numpy as np
import pytest

import occastft_amd as ostft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [(6, 40_000_000)],                                    # 625001 frames: thousands of tiles, in parts
    [(8, 100)] * 700,                                     # one tile each
    [(e, 5000 * (e - 5) + 7) for e in range(6, 16)] * 3,  # every class
    [(12, 1 << 20), (7, 1), (12, 0), (16, 1 << 18)],      # an empty signal, a window outside the classes
])
def test_batch_equals_requests_alone(sizes):
    import torch

    rng = np.random.default_rng(len(sizes))
    opts = ["--power_return", "--hanning_window --remove_dc", "--half_spectrum_return"]
    with ostft.Runner(0) as r:
        jobs = []
        for i, (exp, n) in enumerate(sizes):
            x = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda()
            jobs.append((x, ostft.parse_options(opts[i % 3], exp, 0.0 if exp == 6 else 0.5), None))
        for _ in range(3):  # both descriptor blocks, and one again
            outs = r.run_batch_device(jobs)
        for i in range(0, len(jobs), max(1, len(jobs) // 40)):
            assert torch.equal(outs[i], r.run_device(jobs[i][0], jobs[i][1])), sizes[i]
