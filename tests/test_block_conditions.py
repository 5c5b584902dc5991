"""Which calls the MLP block's single node takes (on the CPU)."""
import pytest
import torch

from bitsparse_amd import layers
from bitsparse_amd.bitsparse import TensorBuffer

E4M3 = torch.float8_e4m3fn


@pytest.mark.parametrize("dtype", [torch.bfloat16, E4M3])
def test_tracing_is_asked_first(monkeypatch, dtype):
    """Under a tracer nothing that it cannot follow (addresses above all) is
    looked at: the separate nodes are taken at once."""
    monkeypatch.setattr(layers, "_plain", lambda t: True)
    x = torch.ones((16, 16), dtype=torch.bfloat16)
    buf = TensorBuffer(512, device="cpu", dtype=dtype)
    args = (x, x, x, x[0], x[0], buf, False, dtype)
    assert layers._block_ok(*args)
    monkeypatch.setattr(torch.compiler, "is_compiling", lambda: True)

    def refuse(*a):
        raise AssertionError("looked at while tracing")
    for name in ("data_ptr", "is_contiguous", "dim"):
        monkeypatch.setattr(torch.Tensor, name, refuse)
    assert not layers._block_ok(*args)
