"""A batch of three or more window sizes on a capturing stream: taken with
use_graphs off, refused again once it is on."""
import pytest

import occastft_amd as ostft

pytestmark = pytest.mark.gpu


def test_many_sizes_are_captured_with_use_graphs_off():
    import torch

    torch.zeros(1, device="cuda")
    with ostft.Runner(0) as r:
        jobs = []
        for i, exp in enumerate(list(range(6, 16)) * 2):
            p = ostft.parse_options("--hanning_window --remove_dc --power_return", exp, 0.5)
            x = torch.zeros(9000 * (exp - 4) + i, device="cuda")
            jobs.append((x, p, torch.zeros(ostft.geometry(p, x.numel())["out_floats"], device="cuda")))
        r.run_batch_device(jobs)
        r.batch_config(use_graphs=0)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            r.run_batch_device(jobs)
        r.batch_config(use_graphs=1)
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            with pytest.raises(ostft.STFTError, match="captured"):
                r.run_batch_device(jobs)
            jobs[0][2].zero_()
        for rep in range(3):
            for i, (x, _, out) in enumerate(jobs):
                x.normal_(generator=torch.Generator("cuda").manual_seed(100 * rep + i))
                out.fill_(-1.0)
            g.replay()
            got = [out.clone() for _, _, out in jobs]
            for (x, p, _), y in zip(jobs, got):
                assert torch.equal(y, r.run_device(x, p)), (rep, p.exp)
            eager = r.run_batch_device(jobs)
            assert all(torch.equal(a, b) for a, b in zip(eager, got))
