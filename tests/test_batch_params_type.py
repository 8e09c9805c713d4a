"""Runner.run_batch_device takes Params and nothing that merely has, or makes,
as many bytes.  No GPU needed: the inputs' checks come first and are met by a
stand-in."""
import ctypes
import types

import pytest

import occastft_amd as ostft
from occastft_amd import _native as N

GOOD = ostft.make_params(10, 0.5)


@pytest.mark.parametrize("bad", [bytes(GOOD), ctypes.sizeof(N.Params), [0] * ctypes.sizeof(N.Params), N.Geometry(), None],
                         ids=["bytes", "int", "list", "another structure", "None"])
def test_other_types_are_refused(bad):
    torch = pytest.importorskip("torch")
    x = types.SimpleNamespace(dtype=torch.float32, is_cuda=True, is_contiguous=lambda: True, data_ptr=lambda: 16,
                              numel=lambda: 64, device=torch.device("cpu"))
    r = ostft.Runner.__new__(ostft.Runner)  # no context: nothing may be run
    with pytest.raises(TypeError):
        r.run_batch_device([(x, GOOD, None), (x, bad, None)])
