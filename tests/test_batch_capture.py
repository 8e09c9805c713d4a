"""A captured batch would replay from request records that later batches have
rewritten: with three or more window sizes it is refused, before anything is
launched, and the capture and the context go on."""
import numpy as np
import pytest

import occastft_amd as ostft

pytestmark = pytest.mark.gpu


def test_batch_of_three_sizes_is_not_captured():
    import torch

    x = torch.from_numpy(np.random.default_rng(0).standard_normal(50_000).astype(np.float32)).cuda()
    with ostft.Runner(0) as r:
        jobs = [(x, ostft.parse_options("--power_return", e, 0.5), None) for e in (7, 9, 11)]
        outs = [o.clone() for o in r.run_batch_device(jobs)]  # tables become resident
        bound = [(x, p, torch.zeros_like(o)) for (_, p, _), o in zip(jobs, outs)]
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        g = torch.cuda.CUDAGraph()
        y = torch.zeros_like(x)
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=s):
            with pytest.raises(ostft.STFTError, match="captured"):
                r.run_batch_device(bound)
            y.copy_(x)
        for _ in range(2):
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, x)
            assert all(int(o.count_nonzero()) == 0 for _, _, o in bound)
        r.run_batch_device(bound)
        assert all(torch.equal(b, o) for (_, _, b), o in zip(bound, outs))
