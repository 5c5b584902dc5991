"""The MLP block's single node and its activation / gradient kernels against
the separate steps they stand for, bit for bit (column sums: fp32 order)."""
import contextlib
import itertools
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn


def _z(shape, seed, special, dev):
    g = torch.Generator().manual_seed(seed)
    z = torch.randn(shape, generator=g).to(torch.bfloat16)
    b = (0.5 * torch.randn(shape[1], generator=g)).to(torch.bfloat16)
    # -0, +Inf, -Inf, largest finite, a value whose square overflows, denormals; NaNs of either
    # sign and any payload
    values = {"inf": (-32768, 0x7f80, -128, 0x7f7f, 0x5f80, 1, 0x0080),
              "nan": (-1, -64, 0x7fff, 0x7f81, -127, 0x7fc0, -32768)}.get(special, ())
    f = z.view(torch.int16).view(-1)
    for i, v in enumerate(values):
        f[(i * 977 + 13) % f.numel()] = v
    return z.to(dev), b.to(dev)


def _same(a, b, what):
    assert a.shape == b.shape and torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what


def _buffer(n, dev, store):
    """A TensorBuffer with room for n values: store is a value type and _packed or not."""
    from bitsparse_amd.bitsparse import TensorBuffer
    fp8, pack = store.startswith("e4m3"), store.endswith("packed")
    size = (n * (7 if fp8 else 15) + 7) // 8 + 16 if pack else n * (1 if fp8 else 2)
    return TensorBuffer(size, device=dev, dtype=E4M3 if fp8 else torch.bfloat16, pack_sbit=pack)


def _activate(z, bias, buf, square, k=1.0):
    """The native activation step: (operand, its scale, bitmask, prefix, start, scale)."""
    from bitsparse_amd._lib import native
    offset, in_place = buf.native_cursor()
    operand, oscale, bitmask, prefix, start, buf.offset, scale = native().activate(
        z, bias, buf.vals, offset, buf.err_flags, in_place, buf.pack_sbit, buf.dtype == E4M3, square, k)
    return operand, oscale, bitmask, prefix, start, scale


def _separate_activation(z, bias, buf, square, k=1.0):
    """The same by the layers' separate steps."""
    from bitsparse_amd.fp8 import to_fp8
    from bitsparse_amd.src import functions as F
    z = z + bias if bias is not None else z.clone()
    if buf.dtype == E4M3:
        operand, oscale, sp = F.relu_quantize_and_compress(z, buf, buf.pack_sbit)
        if square:
            operand, oscale = to_fp8(z.square().mul_(k))
    else:
        operand, sp = F.relu_and_compress(z, buf, buf.pack_sbit)
        oscale = None
        if square:
            operand = operand.square().mul_(k)
    return operand, oscale, sp.bitmask, sp.prefix, sp.vals_offset, sp.scale


def _same_step(want, got, bufs):
    for a, b, name in zip(want, got, ("operand", "operand scale", "bitmask", "prefix", "start", "scale")):
        assert (a is None) == (b is None), name
        if a is not None:
            _same(a.reshape(1) if a.numel() == 1 else a, b.reshape(1) if b.numel() == 1 else b, name)
    _same(bufs[0].vals, bufs[1].vals, "values")
    _same(bufs[0].offset, bufs[1].offset, "cursor")


STORES = ["bf16", "e4m3", "bf16_packed", "e4m3_packed"]


# one tile, short last tile rows and columns, a row of several workgroups
@pytest.mark.parametrize("shape", [(1, 8), (64, 64), (65, 72), (80, 1416), (304, 528), (1000, 1024)])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("special", [None, "inf", "nan"])
def test_activation_step(dev, shape, bias, square, store, special):
    z, b = _z(shape, 3, special, dev)
    bufs = [_buffer(z.numel(), dev, store) for _ in range(2)]
    b = b if bias else None
    want = _separate_activation(z, b, bufs[0], square)
    _same_step(want, _activate(z, b, bufs[1], square), bufs)


@pytest.mark.parametrize("value", [2.0e25, 3.0e-25, float("inf"), float("nan"), -float("nan"), None])
@pytest.mark.parametrize("k", [1.0, 0.37, -2.0, 0.0])
@pytest.mark.parametrize("store", STORES)
def test_codes_of_the_square(dev, value, k, store):
    """h = k r^2 over the whole range of scales: a square past
    bf16's range (an infinite scale), all squares underflowing, Inf, NaN of
    either sign, an all-negative pre-activation; k of either sign and 0."""
    z, _ = _z((70, 136), 4, None, dev)
    if value is None:
        z = -z.abs()
    elif value == 3.0e-25:
        z = z * value
    else:
        z[3, 5] = value
    bufs = [_buffer(z.numel(), dev, store) for _ in range(2)]
    want = _separate_activation(z, None, bufs[0], True, k)
    _same_step(want, _activate(z, None, bufs[1], True, k), bufs)


# (over z without a bias, where a recount sees the relu of z; the square of a
# z written over is waited for instead)
@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("bias,square", [(True, True), (True, False), (False, False), (False, True)])
def test_activation_step_lookback_fallback(dev, store, bias, square, monkeypatch):
    """With no patience a unit that finds a predecessor unpublished counts it
    from the dense input, where the bias has to be added too (and rows past the matrix, whose
    bias alone may be positive, count nothing)."""
    from bitsparse_amd import _lib
    z, b = _z((8008, 4096), 12, None, dev)         # 1000 units: some meet an unpublished predecessor
    b = b.abs() if bias else None
    ws = _lib.workspace_for(z.device)
    outs, bufs, counted = [], [], []
    for patience in (None, "0"):
        if patience is not None:
            monkeypatch.setenv("BITSPARSE_LOOKBACK_PATIENCE", patience)
        bufs.append(_buffer(z.numel(), dev, store))
        before = ws.fallback_count()
        outs.append(_activate(z.clone(), b, bufs[-1], square))
        counted.append(ws.fallback_count() - before)
    in_place = square and not bias and not store.startswith("e4m3")
    assert counted[0] == 0 and (counted[1] > 0) == (not in_place), counted
    _same_step(*outs, bufs)
    assert not bufs[1].overflowed()


@pytest.mark.parametrize("shape", [(1, 8), (64, 64), (65, 72), (80, 1416), (1000, 1024), (4100, 192)])
@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("zeros", [0.0, 0.5, 1.0])
def test_gradient_step(dev, shape, store, square, zeros):
    """The activation's gradient with every set of what rides on it: the
    gradient and its codes bit for bit, the bias gradient to its rounding."""
    from bitsparse_amd._lib import native
    from bitsparse_amd.src import functions as F
    from bitsparse_amd.src import hip_operators as H
    z, _ = _z(shape, 6, None, dev)
    z = z.abs() + 1 if zeros == 0.0 else (-z.abs() if zeros == 1.0 else z)
    fp8, pack = store.startswith("e4m3"), store.endswith("packed")
    if fp8:
        sp = F.quantize_and_compress(z.relu(), None, pack)[2]
    else:
        sp = F.dense_to_tilesparse(z.relu(), None, None, pack)
    g0 = torch.randn(shape, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).to(dev)
    want = g0.clone()
    (H.relu2_grad_sparse_ if square else H.mask_with_bitmask_)(want, sp)
    wq, wscale = H.quantize_e4m3fn(want, H.amax_into_workspace(want))
    w64 = want.double().sum(0)
    bound = shape[0] * 2.0 ** -24 * want.double().abs().sum(0) + 2.0 ** -8 * w64.abs() + 1e-30
    # transposed codes: rows in whole groups of 4
    for bias, rows, cols in itertools.product((False, True), (False, fp8), (False, fp8 and shape[0] % 4 == 0)):
        g, held = g0.clone(), [sp.vals, sp.bitmask, sp.prefix, sp.vals_offset, sp.scale]
        sums, q, qt, scale, scale_t = native().act_grad(g, held, pack, fp8, square, 1.0, bias, rows, cols)
        assert held == []
        _same(want, g, "gradient")
        assert (sums is not None, q is not None, qt is not None) == (bias, rows, cols)
        if bias:
            assert ((sums.double() - w64).abs() <= bound).all()
        for codes, s, t in ((q, scale, wq), (qt, scale_t, wq.view(torch.uint8).t().contiguous())):
            if codes is not None:
                _same(wscale.reshape(1), s.reshape(1), "scale")
                _same(t.view(torch.uint8), codes.view(torch.uint8), "codes")


# ---------------------------------------------------------------------------
# the whole block against the separate nodes
# ---------------------------------------------------------------------------
NAMES = ("x", "W1", "W2", "b1", "b2")


def _operands(dev, T, D, Hn, O, biases=("b1", "b2"), seed=11):
    """(operands by name, gradient of y)"""
    g = torch.Generator().manual_seed(seed)

    def r(*s, mul=0.1):
        return (mul * torch.randn(s, generator=g)).to(torch.bfloat16).to(dev)
    p = dict(x=r(T, D, mul=1.0), W1=r(Hn, D), W2=r(O, Hn), b1=r(Hn), b2=r(O))
    dY = r(T, O, mul=1.0)
    return {k: v if k in biases or k[0] != "b" else None for k, v in p.items()}, dY


def _block(p, store, square, block, buf=None):
    """y of the layer on operands p, as one node or by the separate ones."""
    from bitsparse_amd import layers
    layer, kw = (layers.FFNRelu2, "storage_dtype") if square else (layers.FFNRelu, "dtype")
    buf = buf or _buffer(p["x"].shape[:-1].numel() * p["W1"].shape[0], p["x"].device, store)
    with pytest.MonkeyPatch.context() as m:
        if not block:
            m.setattr(layers, "_block_ok", lambda *a: False)
        y = layer.apply(p["x"], p["W1"], p["W2"], p["b1"], p["b2"], sparse_data=buf,
                        pack_sbit=store.endswith("packed"), **{kw: E4M3 if store.startswith("e4m3") else torch.bfloat16})
    if y.requires_grad:
        # (a block none of whose operands but b2 asks for a gradient leaves b2's node alone)
        taken = any(n.name() == "_FFNBlockBackward" or n.name().endswith("Biased>") for n in _graph_nodes(y))
        assert taken == block, "the node that was asked for"
    return y


def _params(p, need=NAMES):
    return {k: None if t is None else t.clone().requires_grad_(k in need) for k, t in p.items()}


def _compare(got, want, T):
    """y, dx, dW1, dW2 bit for bit; the bias gradients (fp32 sums of T values in
    another order, rounded once each) to their rounding."""
    assert got.keys() == want.keys()
    for name, a in got.items():
        b = want[name]
        if name in ("b1", "b2"):
            assert ((a - b).double().abs() <= 2.0 ** -7 * b.double().abs() + 1e-2).all(), name
        else:
            _same(a, b, name)


def _step(p, dY, store, square, block, need=NAMES, buf=None):
    q = _params(p, need)
    y = _block(q, store, square, block, buf)
    out = {"y": y.detach()}
    if need:
        y.backward(dY)
        out.update({k: t.grad for k, t in q.items() if t is not None and k in need})
    return out


# tokens, in, hidden, out: ordinary; one token; rows and columns that end inside a tile and a
# GEMM's tile, in != out; (fp8: multiples of 16)
@pytest.mark.parametrize("shape", [(208, 144, 528, 144), (1, 8, 8, 8), (67, 20, 136, 12), (300, 72, 1416, 40),
                                   (16, 48, 32, 80)])
@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("biases", [(), ("b1",), ("b2",), ("b1", "b2")])
def test_block_equals_the_separate_nodes(dev, shape, square, store, biases):
    if store.startswith("e4m3") and any(n % 16 for n in shape):
        shape = tuple(-(-n // 16) * 16 for n in shape)
    p, dY = _operands(dev, *shape, biases)
    _compare(_step(p, dY, store, square, True), _step(p, dY, store, square, False), shape[0])


@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", STORES)
def test_block_with_frozen_operands(dev, square, store):
    """Every subset of the operands that may ask for a gradient."""
    p, dY = _operands(dev, 80, 48, 144, 32)
    for n in range(len(NAMES) + 1):
        for need in itertools.combinations(NAMES, n):
            _compare(_step(p, dY, store, square, True, need), _step(p, dY, store, square, False, need), 80)


@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan"), 3.0e38, 1.0e-38])
def test_block_special_values(dev, square, store, value):
    p, dY = _operands(dev, 80, 48, 144, 32)
    p["x"][3, 5] = value
    got, want = (_step(p, dY, store, square, block) for block in (True, False))
    for name in ("y", "x", "W1", "W2"):
        a, b = got[name], want[name]
        assert torch.equal(a.isnan(), b.isnan()), name
        _same(a.nan_to_num(1.5), b.nan_to_num(1.5), name)
    for name in ("b1", "b2"):
        a, b = got[name], want[name]
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()), name
        ok = a.isfinite()
        assert ((a[ok] - b[ok]).double().abs() <= 2.0 ** -7 * b[ok].double().abs() + 1e-2).all(), name


@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("layout", ["3d", "transposed", "padded", "one_row"])
def test_block_input_layouts(dev, store, layout):
    p, dY = _operands(dev, 96, 48, 144, 48)
    base, view = {"3d": (p["x"].reshape(2, 48, 48), lambda t: t),
                  "transposed": (p["x"].t().contiguous(), lambda t: t.t()),
                  "padded": (torch.nn.functional.pad(p["x"], (0, 16)), lambda t: t[:, :48]),
                  "one_row": (p["x"][:1], lambda t: t.expand(96, 48))}[layout]
    outs = []
    for block in (True, False):
        q = _params(p)
        leaf = base.clone().requires_grad_()
        q["x"] = view(leaf)
        y = _block(q, store, True, block)
        y.backward(dY.reshape(y.shape))
        outs.append({"y": y.detach(), "x": leaf.grad, **{k: q[k].grad for k in NAMES[1:]}})
    _compare(*outs, 96)


@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("biases", [(), ("b1",), ("b2",), ("b1", "b2")])
@pytest.mark.parametrize("dims", [2, 3])
def test_block_result_changed_in_place(dev, store, biases, dims):
    """In-place calls on y: what the separate nodes' result allows, with their gradients."""
    p, dY = _operands(dev, 96, 48, 144, 48, biases)
    if dims == 3:
        p["x"], dY = p["x"].reshape(2, 48, 48), dY.reshape(2, 48, 48)
    outs, views = [], []
    for block in (True, False):
        q = _params(p)
        y = _block(q, store, False, block)
        views.append(y._is_view())
        if "b2" in biases:
            assert not _block(q, store, False, block).detach_().requires_grad
        y.mul_(2.0)
        y.backward(dY)
        outs.append({"y": y.detach(), **{k: t.grad for k, t in q.items() if t is not None}})
    assert views[0] == views[1]
    _compare(*outs, 96)


@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("dims", [2, 3])
def test_gradient_of_b2_alone(dev, store, dims):
    """A walk for b2 alone, for one gradient and for a batch of them, needs nothing of
    the block: the whole walk after it finds the compressed activation."""
    p, dY = _operands(dev, 96, 48, 144, 48)
    if dims == 3:
        p["x"], dY = p["x"].reshape(2, 48, 48), dY.reshape(2, 48, 48)
    outs = []
    for block in (True, False):
        q = _params(p)
        y = _block(q, store, True, block)
        one, = torch.autograd.grad(y, q["b2"], dY, retain_graph=True)
        batch, = torch.autograd.grad(y, q["b2"], torch.stack([dY, 2 * dY]), retain_graph=True, is_grads_batched=True)
        y.backward(dY)
        bound = 2.0 ** -8 * one.double().abs() + 1e-2          # sums in another order, rounded once
        assert ((q["b2"].grad - one).double().abs() <= bound).all()
        assert ((batch[0] - one).double().abs() <= bound).all()
        assert ((batch[1] - 2 * one).double().abs() <= 2 * bound).all()
        outs.append({"y": y.detach(), **{k: t.grad for k, t in q.items()}})
    _compare(*outs, 96)


@pytest.mark.parametrize("store", ["bf16", "e4m3"])
@pytest.mark.parametrize("biases", [("b2",), ("b1", "b2")])
@pytest.mark.parametrize("leaf", [True, False])
def test_walks_for_some_operands(dev, store, biases, leaf, monkeypatch):
    """Walks after some of the operands' gradients form those alone, with the values of
    a whole walk; all operands ask for gradients."""
    from bitsparse_amd._lib import native
    p, dY = _operands(dev, 96, 48, 144, 48, biases)
    names = [n for n in NAMES if p[n] is not None]
    whole = _step(p, dY, store, True, True)
    inner, formed = native().block_backward, []

    def spy(*args):
        out = inner(*args)
        formed.append({n for n, t in zip(("x", "W1", "b1", "W2"), out) if t is not None})
        return out
    monkeypatch.setattr(native(), "block_backward", spy)
    for n in range(1, len(names) + 1):
        for ask in itertools.combinations(names, n):
            for walk in ("grad", "backward") if leaf else ("grad",):     # (backward's inputs are leaves here)
                q = _params(p)
                if not leaf:
                    q["x"] = q["x"] * 1
                y = _block(q, store, True, True)
                formed.clear()
                if walk == "grad":
                    got = dict(zip(ask, torch.autograd.grad(y, [q[k] for k in ask], dY)))
                else:
                    torch.autograd.backward(y, dY, inputs=[q[k] for k in ask])
                    got = {k: q[k].grad for k in ask}
                _compare(got, {k: whole[k] for k in ask}, 96)
                assert formed == ([set(ask) - {"b2"}] if set(ask) != {"b2"} else []), ask


@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("in_place", [False, True])
def test_blocks_of_one_buffer(dev, store, in_place):
    """Blocks appended to one buffer, backwards in the reverse order; then
    over again after a reset."""
    ps = [_operands(dev, 80, 48, 144, 48, seed=s) for s in (1, 2, 3)]
    want = [_step(p, dY, store, True, False) for p, dY in ps]
    buf = _buffer(4 * 80 * 144, dev, store)
    buf.inplace_offset = in_place
    for _ in range(2):
        buf.reset_buffer()
        qs = [_params(p) for p, _ in ps]
        ys = [_block(q, store, True, True, buf) for q in qs]
        for y, (_, dY) in reversed(list(zip(ys, ps))):
            y.backward(dY)
        for q, y, w in zip(qs, ys, want):
            _compare({"y": y.detach(), **{k: t.grad for k, t in q.items()}}, w, 80)
    assert not buf.overflowed()


@pytest.mark.parametrize("block", [True, False])
@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", ["bf16", "e4m3"])
def test_backward_under_autocast(dev, block, square, store):
    """A backward that runs inside autocast: in bfloat16 nothing changes, in
    float16 the bf16 products would come in a type the activation's gradient
    does not take, and are refused (the fp8 ones are not autocast)."""
    p, dY = _operands(dev, 80, 48, 144, 32)
    want = _step(p, dY, store, square, block)
    for dtype in (torch.bfloat16, torch.float16):
        q = _params(p)
        y = _block(q, store, square, block)
        refused = dtype == torch.float16 and store == "bf16"
        with torch.autocast("cuda", dtype=dtype), pytest.raises(TypeError) if refused else contextlib.nullcontext():
            y.backward(dY)
        if not refused:
            _compare({"y": y.detach(), **{k: t.grad for k, t in q.items()}}, want, 80)


@pytest.mark.parametrize("block", [True, False])
@pytest.mark.parametrize("store", ["bf16", "e4m3"])
@pytest.mark.parametrize("name", ["x", "W1", "W2"])
@pytest.mark.parametrize("kind", ["float32", "float16", "cpu", "flat", "wider", "longer"])
def test_saved_tensors_of_another_kind(dev, block, store, name, kind):
    """A saved-tensor hook that hands the backward an operand in another type,
    on another device or of another shape: an error, and nothing read as what
    it is not."""
    p, dY = _operands(dev, 80, 48, 144, 32)
    q = _params(p)
    shape = tuple(q[name].shape)

    def unpack(t):
        # (x @ W1.T saves W1 as a transposed view)
        if tuple(t.shape) not in (shape, shape[::-1]):
            return t
        # (zeros around it: other shapes, all fp8 products of them possible by themselves)
        pad = torch.nn.functional.pad
        return {"float32": t.float, "float16": t.half, "cpu": t.cpu, "flat": t.flatten,
                "wider": lambda: pad(t, (0, 64)), "longer": lambda: pad(t, (0, 0, 0, 64))}[kind]()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        y = _block(q, store, False, block)
    with pytest.raises((RuntimeError, TypeError, ValueError, IndexError, AssertionError)):
        y.backward(dY)
    torch.cuda.synchronize(dev)


@pytest.mark.parametrize("store", STORES)
@pytest.mark.parametrize("layout", ["misaligned", "transposed", "padded"])
def test_saved_tensors_in_another_layout(dev, store, layout):
    """... and one that hands back the same values at another address (a view
    into a flat buffer) or with other strides changes nothing."""
    p, dY = _operands(dev, 80, 48, 144, 32)
    want = _step(p, dY, store, False, False)

    def unpack(t):
        t = t.contiguous()
        if layout == "misaligned":
            return torch.cat([t.flatten()[:1], t.flatten()])[1:].view(t.shape)
        return t.t().contiguous().t() if layout == "transposed" else torch.nn.functional.pad(t, (0, 8))[:, :t.shape[1]]
    q = _params(p)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        y = _block(q, store, False, True)
    y.backward(dY)
    _compare({"y": y.detach(), **{k: t.grad for k, t in q.items()}}, want, 80)


@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", STORES)
def test_block_in_a_buffer_too_small(dev, square, store):
    """Values that do not fit are dropped and flagged; y does not depend on them."""
    p, _ = _operands(dev, 208, 48, 528, 48)
    outs, bufs = [], []
    for block in (True, False):
        bufs.append(_buffer(208 * 528 // 5 // 32 * 32, dev, store))
        with torch.no_grad():
            outs.append(_block(p, store, square, block, bufs[-1]))
    _same(*outs, "y")
    _same(bufs[0].vals, bufs[1].vals, "values")
    _same(bufs[0].offset, bufs[1].offset, "cursor")
    assert bufs[0].overflowed() and bufs[1].overflowed()


@pytest.mark.parametrize("store", STORES)
def test_epoch_wrap_inside_a_block(dev, store):
    """The workspace's counter wraps (and clears the amax slot) at every place
    inside a forward and backward."""
    from bitsparse_amd import _lib
    p, dY = _operands(dev, 80, 48, 144, 32)
    want = _step(p, dY, store, True, False)
    ws = _lib.workspace_for(p["x"].device)
    _step(p, dY, store, True, True)
    before = ws.epoch
    _step(p, dY, store, True, True)
    took = ws.epoch - before
    for left in range(took + 2):
        ws.buf.zero_()                   # (the counter is set back: no word of a later epoch)
        ws.epoch = _lib._EPOCH_LIMIT - left
        _compare(_step(p, dY, store, True, True), want, 80)
        assert 0 < ws.epoch <= _lib._EPOCH_LIMIT


@pytest.mark.parametrize("store", STORES)
def test_block_on_another_stream(dev, store):
    p, dY = _operands(dev, 304, 64, 528, 64)
    want = _step(p, dY, store, True, False)
    s = torch.cuda.Stream(dev)
    for _ in range(3):
        s.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(s):
            got = _step(p, dY, store, True, True)
        torch.cuda.current_stream(dev).wait_stream(s)
        _compare(got, want, 304)


@pytest.mark.parametrize("own_streams", [False, True])
@pytest.mark.parametrize("store", ["bf16", "e4m3"])
def test_blocks_of_two_threads(dev, store, own_streams):
    """Two threads, on one stream (one workspace) or on a stream each."""
    jobs = [_operands(dev, 144, 64, 272, 64, seed=s) for s in (1, 2)]
    want = [_step(p, dY, store, True, True) for p, dY in jobs]
    torch.cuda.synchronize(dev)
    errors = []

    def work(i):
        try:
            stream = torch.cuda.Stream(dev) if own_streams else torch.cuda.current_stream(dev)
            with torch.cuda.device(dev), torch.cuda.stream(stream):
                got = [_step(*jobs[i], store, True, True) for _ in range(20)]
                stream.synchronize()
            for g in got:
                for k in g:
                    _same(g[k], want[i][k], k)
        except BaseException as e:      # noqa: B036 (handed to the test's thread)
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


def _graph_nodes(t):
    """Every autograd node behind t."""
    nodes, seen = [t.grad_fn], set()
    while nodes:
        n = nodes.pop()
        if n is None or n in seen:
            continue
        seen.add(n)
        yield n
        nodes += [m for m, _ in n.next_functions]


@pytest.mark.parametrize("how", ["default_hooks", "node_hooks", "data"])
@pytest.mark.parametrize("grow", [4.0, 0.25])
def test_backward_scales_the_values_it_reads(dev, how, grow, monkeypatch):
    """The backward's operands need not hold what the forward saw: saved-tensor
    hooks (the default ones, or set on the node afterwards) and writes through
    .data change them without autograd's notice.  They are quantized with
    their own scales: no code past the format, none lost below it."""
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd import config
    from bitsparse_amd.layers import FFNRelu2
    monkeypatch.setattr(config, "FP8_GRAD_DTYPE", torch.bfloat16)
    g = torch.Generator().manual_seed(21)
    x, W1, W2, dY = (torch.randn(s, generator=g).to(torch.bfloat16).to(dev) * 0.1
                     for s in ((64, 64), (128, 64), (64, 128), (64, 64)))
    grads = []
    for factor in (1.0, grow):
        p = [t.clone().requires_grad_() for t in (x, W1, W2)]
        buf = TensorBuffer(64 * 128, device=dev, dtype=E4M3)

        def unpack(t):
            return t * factor
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack) if how == "default_hooks" else \
                contextlib.nullcontext():
            y = FFNRelu2.apply(*p, sparse_data=buf, storage_dtype=E4M3)
        if how == "node_hooks":
            for saved in next(n for n in _graph_nodes(y) if n.name() == "_FFNBlockBackward")._raw_saved_tensors:
                saved.register_hooks(lambda t: t, unpack)
        elif how == "data":
            for t in p:
                t.data.mul_(factor)
        y.backward(dY)
        grads.append([t.grad for t in p])
    # dx = (dY W2 . 2 r) W1 and dW1 = (dY W2 . 2 r)^T x with all three scaled; r is the
    # forward's, and a power of two moves no code
    for i in (0, 1):
        assert torch.equal(grads[1][i].float(), grads[0][i].float() * grow * grow), i
    assert torch.equal(grads[1][2], grads[0][2])


@pytest.mark.parametrize("store", ["bf16", "e4m3", "bf16_packed"])
@pytest.mark.parametrize("block", [True, False])
@pytest.mark.parametrize("layout", ["one_row", "one_value", "column", "transposed", "padded", "misaligned", "overlapping"])
def test_gradient_layouts(dev, store, block, layout, monkeypatch):
    """The gradients that y.sum(0), y.mean() and slices of a wider output
    deliver: expanded, transposed, strided and misaligned ones give what their
    contiguous copy gives."""
    from bitsparse_amd import layers
    from bitsparse_amd.bitsparse import TensorBuffer
    if not block:
        monkeypatch.setattr(layers, "_block_ok", lambda *a: False)
    g = torch.Generator().manual_seed(31)
    T, D, Hn = 80, 48, 144
    x, W1, b1, W2, b2, base = (torch.randn(s, generator=g).to(torch.bfloat16).to(dev) * 0.1
                               for s in ((T, D), (Hn, D), (Hn,), (D, Hn), (D,), (T * (D + 8) + 8,)))
    strides = {"one_row": (0, 1), "one_value": (0, 0), "column": (1, 0), "transposed": (1, T), "padded": (D + 8, 1),
               "misaligned": (D, 1), "overlapping": (8, 1)}[layout]
    dY = base.as_strided((T, D), strides, 1 if layout == "misaligned" else 0)
    fp8, pack = store == "e4m3", store.endswith("packed")
    outs = []
    for grad in (dY, dY.contiguous()):
        p = [t.clone().requires_grad_() for t in (x, W1, W2, b1, b2)]
        buf = TensorBuffer(2 * T * Hn + 64, device=dev, dtype=E4M3 if fp8 else torch.bfloat16, pack_sbit=pack)
        y = layers.FFNRelu.apply(*p, sparse_data=buf, pack_sbit=pack, dtype=E4M3 if fp8 else torch.bfloat16)
        y.backward(grad)
        outs.append([t.grad for t in p])
    for a, b, name in zip(*outs, ("dx", "dW1", "dW2", "db1")):
        _same(a, b, name)
    # another summation order where torch sums a strided gradient: fp32 sums, one rounding each
    a, b = outs[0][4].double(), outs[1][4].double()
    assert ((a - b).abs() <= 2.0 ** -8 * (a.abs() + b.abs()) + T * 2.0 ** -23 * dY.double().abs().sum(0)).all()


@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", ["bf16", "e4m3", "bf16_packed"])
@pytest.mark.parametrize("bias", [False, True])
def test_peak_memory(dev, square, store, bias, monkeypatch):
    """The single node holds no more at its peak than the separate ones, whose
    square is in place and whose product goes at the bias add (the biased
    operand is a second [T, H] beside z like theirs, but with the bitmask
    there already)."""
    from bitsparse_amd import layers
    from bitsparse_amd.bitsparse import TensorBuffer
    g = torch.Generator().manual_seed(41)
    T, D, Hn = 2048, 128, 2048
    fp8, pack = store == "e4m3", store.endswith("packed")
    p = [(torch.randn(s, generator=g).to(torch.bfloat16).to(dev) * 0.1).requires_grad_()
         for s in ((T, D), (Hn, D), (D, Hn), (Hn,), (D,))]
    dY = torch.randn((T, D), generator=g).to(torch.bfloat16).to(dev)
    buf = TensorBuffer(2 * T * Hn + 64, device=dev, dtype=E4M3 if fp8 else torch.bfloat16, pack_sbit=pack)
    layer, kw = (layers.FFNRelu2, "storage_dtype") if square else (layers.FFNRelu, "dtype")
    peaks = []
    for block in (True, False):
        if not block:
            monkeypatch.setattr(layers, "_block_ok", lambda *a: False)
        for _ in range(2):                       # the second has its workspaces
            buf.reset_buffer()
            base = torch.cuda.memory_allocated(dev)
            torch.cuda.reset_peak_memory_stats(dev)
            y = layer.apply(*p[:3], *(p[3:] if bias else ()), sparse_data=buf, pack_sbit=pack,
                            **{kw: E4M3 if fp8 else torch.bfloat16})
            forward = torch.cuda.max_memory_allocated(dev) - base
            torch.cuda.reset_peak_memory_stats(dev)
            y.backward(dY)
            backward = torch.cuda.max_memory_allocated(dev) - base
            del y
            for t in p:
                t.grad = None
        peaks.append((forward, backward))
    slack = 64 * 1024                            # rows of N, cursors, scales: each its own 512-byte block
    assert peaks[0][0] <= peaks[1][0] + slack + (T * Hn // 8 + T * Hn // 1024 if bias else 0), peaks
    assert peaks[0][1] <= peaks[1][1] + slack, peaks


@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", STORES)
def test_gradients_with_a_graph(dev, square, store):
    """create_graph: the same gradients have a graph as those of the separate
    nodes, and it leads to the same second gradients."""
    p, dY = _operands(dev, 80, 48, 144, 32)
    outs = []
    for block in (True, False):
        q = _params(p)
        gy = dY.clone().requires_grad_()
        y = _block(q, store, square, block)
        leaves = [*q.values(), gy]
        first = torch.autograd.grad(y, list(q.values()), gy, create_graph=True)
        loss = sum((t.float() ** 2).sum() for t in first if t.requires_grad)
        second = torch.autograd.grad(loss, leaves, allow_unused=True)
        outs.append((first, second))
    (f1, s1), (f2, s2) = outs
    assert [t.requires_grad for t in f1] == [t.requires_grad for t in f2]
    assert [t is None for t in s1] == [t is None for t in s2]
    for name, a, b in zip(NAMES, f1, f2):
        err = (a.double() - b.double()).norm() / b.double().norm()
        assert float(err) <= (2.0 ** -7 if name in ("b1", "b2") else 0.0), name
    # bf16 sums of a few contributions each, in the order the engine comes by them: 2^-9 an addition
    for name, a, b in zip((*NAMES, "gy"), s1, s2):
        assert a is None or float((a.double() - b.double()).norm() / b.double().norm()) <= 2.0 ** -7, name
