"""ostft_batch_out_floats: each job's output size as ostft_get_geometry gives
it, 0 where the geometry is refused.  No GPU needed."""
import ctypes

import numpy as np

import occastft_amd as ostft
from occastft_amd import _native as N


def test_sizes_of_a_mixed_batch():
    rng = np.random.default_rng(1)
    layouts = ["", "--half_complex_return", "--magnitude_return", "--power_return", "--half_spectrum_return"]
    params, sizes = [], []
    for i in range(40):
        params.append(ostft.parse_options(layouts[i % 5], int(rng.integers(6, 21)), float(rng.choice([0.0, 0.33, 0.75]))))
        sizes.append(int(rng.integers(0, 1 << 22)))
    params += [ostft.make_params(5, 0.0), ostft.make_params(10, 1.0), ostft.make_params(10, 0.5, output=9)]  # refused
    sizes += [1000] * 3
    jobs = (N.Job * len(params))()
    for j, p, n in zip(jobs, params, sizes):
        j.params, j.full_size = p, n
    got = (ctypes.c_uint64 * len(params))()
    assert N.lib().ostft_batch_out_floats(jobs, len(params), got) == N.OK
    want = [ostft.geometry(p, n)["out_floats"] for p, n in zip(params[:40], sizes)] + [0, 0, 0]
    assert list(got) == want
    assert N.lib().ostft_batch_out_floats(None, 0, None) == N.OK
    assert N.lib().ostft_batch_out_floats(None, 2, got) == N.ERR_INVALID_ARG
