"""The TensorBuffer's cursor as the native calls are given it (on the CPU: the
native module is replaced by one that records its arguments)."""
import copy
import pickle
import types

import pytest
import torch

from bitsparse_amd import layers
from bitsparse_amd.bitsparse import TensorBuffer
from bitsparse_amd.src import functions as F

E4M3 = torch.float8_e4m3fn
BLOCK_OK = layers._block_ok


@pytest.fixture
def calls(monkeypatch):
    """What the native entry points were called with: (offset, in_place)."""
    seen = []
    meta = torch.zeros(1, dtype=torch.int64)

    def compress(dense, vals, offset, in_place, *rest):
        seen.append((offset, in_place))
        return meta, meta, meta, offset if in_place else meta, None, None

    def block_forward(x, W1, b1, W2, b2, vals, offset, err, in_place, *rest):
        seen.append((offset, in_place))
        return x.new_zeros((x.shape[0], W2.shape[0])), meta, meta, meta, offset if in_place else meta, None
    stub = types.SimpleNamespace(compress=compress, block_forward=block_forward)
    monkeypatch.setattr(F, "native", lambda: stub)
    monkeypatch.setattr(layers, "native", lambda: stub)
    monkeypatch.setattr(F.ops, "require_device", lambda *a: None)
    monkeypatch.setattr(layers, "_block_ok", lambda *a: True)
    return seen


def _use(what, buf):
    x = torch.ones((8, 8), dtype=torch.bfloat16)
    if what == "compress":
        F.dense_to_tilesparse(x, None, buf)
    elif what == "quantize":
        F.quantize_and_compress(x, buf)
    else:
        layers.FFNRelu.apply(x, x, x, sparse_data=buf)


@pytest.mark.parametrize("what", ["compress", "quantize", "block"])
def test_in_place_cursor_chosen_after_a_reset(calls, what):
    """An in-place call always comes with the cursor tensor it advances."""
    buf = TensorBuffer(128, device="cpu", dtype=E4M3 if what == "quantize" else torch.bfloat16)
    buf.reset_buffer()
    _use(what, buf)
    assert calls[-1][0] is None and calls[-1][1] is False        # 0, no tensor needed
    buf.reset_buffer()
    buf.inplace_offset = True
    _use(what, buf)
    offset, in_place = calls[-1]
    assert in_place is True and offset is buf.offset and int(offset) == 0


def test_buffers_of_earlier_files(calls):
    """A TensorBuffer saved when the cursor was a plain attribute loads with
    its cursor, and one copied or saved now keeps it, reset or not."""
    buf = TensorBuffer(128, device="cpu")
    state = dict(buf.__dict__)
    state["offset"] = state.pop("_offset") + 5
    old = TensorBuffer.__new__(TensorBuffer)
    pickled = pickle.dumps(buf)
    if hasattr(old, "__setstate__"):
        old.__setstate__(state)
    else:
        old.__dict__.update(state)
    _use("compress", old)
    offset, in_place = calls[-1]
    assert int(offset) == 5 and in_place is False
    for again in (pickle.loads(pickled), copy.deepcopy(buf)):
        assert int(again.offset) == 0 and again.offset is not buf.offset
    buf.reset_buffer()
    assert pickle.loads(pickle.dumps(buf))._offset is None


@pytest.mark.parametrize("what", ["compress", "quantize", "block"])
@pytest.mark.parametrize("hook", ["cursor", "advance", "offset"])
def test_buffers_with_a_cursor_of_their_own(calls, monkeypatch, what, hook):
    """A subclass that takes over the cursor's protocol is asked through it:
    the native calls, which go past it, are for the plain buffer."""
    used = []

    class Own(TensorBuffer):
        pass
    if hook == "offset":
        def get(self):
            used.append(hook)
            return TensorBuffer.offset.fget(self)
        Own.offset = property(get, TensorBuffer.offset.fset)
    else:
        def method(self, *a):
            used.append(hook)
            return getattr(TensorBuffer, hook)(self, *a)
        setattr(Own, hook, method)
    for op in ("compress_into", "amax_into_workspace"):
        monkeypatch.setattr(F.ops, op, lambda *a, **k: 1)
    buf = Own(128, device="cpu", dtype=E4M3 if what == "quantize" else torch.bfloat16)
    if what == "block":
        monkeypatch.setattr(layers, "_plain", lambda t: True)
        x = torch.ones((16, 16), dtype=torch.bfloat16)
        args = (None, None), (False, torch.bfloat16)
        assert BLOCK_OK(x, x, x, *args[0], TensorBuffer(512, device="cpu"), *args[1])
        assert not BLOCK_OK(x, x, x, *args[0], buf, *args[1])
        return
    _use(what, buf)
    assert used and not calls


def test_plain_subclass_keeps_the_native_calls(calls):
    class Plain(TensorBuffer):
        pass
    _use("compress", Plain(128, device="cpu"))
    assert calls
