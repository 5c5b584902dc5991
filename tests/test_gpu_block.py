"""The MLP block's single node and its activation / gradient kernels against
the separate steps they stand for, bit for bit (column sums: fp32 order)."""
import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn


def _z(shape, seed, special, dev):
    g = torch.Generator().manual_seed(seed)
    z = torch.randn(shape, generator=g).to(torch.bfloat16)
    b = (0.5 * torch.randn(shape[1], generator=g)).to(torch.bfloat16)
    if special:
        f = z.view(torch.int16).view(-1)
        n = f.numel()
        # -0, +Inf, -Inf, largest finite, a value whose square overflows, denormals
        for i, v in enumerate((-32768, 0x7f80, -128, 0x7f7f, 0x5f80, 1, 0x0080)):
            f[(i * 977 + 13) % n] = v
    return z.to(dev), b.to(dev)


def _same(a, b, what):
    assert a.shape == b.shape and torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what


# one tile, short last tile rows and columns, a row of several workgroups
@pytest.mark.parametrize("shape", [(1, 8), (64, 64), (65, 72), (80, 1416), (304, 528), (1000, 1024)])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", ["bf16", "e4m3", "bf16_packed", "e4m3_packed"])
@pytest.mark.parametrize("special", [False, True])
def test_activation_step(dev, shape, bias, square, store, special):
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd.fp8 import to_fp8
    from bitsparse_amd.src import functions as F
    fp8, pack = store.startswith("e4m3"), store.endswith("packed")
    z, b = _z(shape, 3, special, dev)
    n = z.numel()
    size = (n * (7 if fp8 else 15) + 7) // 8 + 16 if pack else n * (1 if fp8 else 2)
    bufs = [TensorBuffer(size, device=dev, dtype=E4M3 if fp8 else torch.bfloat16, pack_sbit=pack) for _ in range(2)]
    zz = z + b if bias else z.clone()
    if fp8:
        q, scale, want = F.relu_quantize_and_compress(zz, bufs[0], pack)
        operand, oscale = (q, scale) if not square else to_fp8(zz.square().mul_(1.0))
    else:
        operand, want = F.relu_and_compress(zz, bufs[0], pack)
        oscale = None
        if square:
            operand = operand.square().mul_(1.0)
    assert F.activate_ok(z, b if bias else None, bufs[1], 1.0)
    got_operand, got_scale, got = F.activate_and_compress(z, b if bias else None, bufs[1], pack, fp8, square)
    _same(want.bitmask, got.bitmask, "bitmask")
    _same(want.prefix, got.prefix, "prefix")
    _same(bufs[0].vals, bufs[1].vals, "values")
    _same(bufs[0].offset, bufs[1].offset, "cursor")
    _same(want.vals_offset.reshape(1), got.vals_offset.reshape(1), "start")
    _same(operand, got_operand, "operand")
    if fp8:
        _same(want.scale.reshape(1), got.scale.reshape(1), "stored scale")
        _same(oscale.reshape(1), got_scale.reshape(1), "operand scale")


@pytest.mark.parametrize("value", [2.0e25, 3.0e-25, float("inf"), float("nan"), -float("nan"), None])
@pytest.mark.parametrize("k", [1.0, 0.37, -2.0, 0.0])
def test_codes_of_the_square(dev, value, k, monkeypatch):
    """The codes of h = k r^2 over the whole range of scales: a square past
    bf16's range (an infinite scale), all squares underflowing, Inf, NaN of
    either sign, an all-negative pre-activation; k of either sign and 0."""
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd.fp8 import to_fp8
    from bitsparse_amd.src import functions as F
    from bitsparse_amd.src import hip_operators as H
    monkeypatch.setattr(H, "RELU2_SCALE", k)
    z, _ = _z((70, 136), 4, False, dev)
    if value is None:
        z = -z.abs()
    elif value == 3.0e-25:
        z = z * value
    else:
        z[3, 5] = value
    bufs = [TensorBuffer(z.numel(), device=dev, dtype=E4M3) for _ in range(2)]
    r = z.clone()
    want_sp = F.relu_quantize_and_compress(r, bufs[0], False)[2]
    want, wscale = to_fp8(r.square().mul_(k))
    got, gscale, sp = F.activate_and_compress(z, None, bufs[1], False, True, True)
    _same(wscale.reshape(1), gscale.reshape(1), "scale of h")
    _same(want, got, "codes of h")
    _same(want_sp.scale.reshape(1), sp.scale.reshape(1), "scale")
    _same(want_sp.bitmask, sp.bitmask, "bitmask")
    _same(bufs[0].vals, bufs[1].vals, "values")


@pytest.mark.parametrize("store", ["bf16", "e4m3"])
def test_activation_step_lookback_fallback(dev, store, monkeypatch):
    """With no patience every wait counts its predecessors from the dense
    input, where the bias has to be added too (and rows past the matrix, whose
    bias alone may be positive, count nothing)."""
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd.src import functions as F
    z, b = _z((72, 64 * 40), 12, False, dev)
    b = b.abs()
    dt = E4M3 if store == "e4m3" else torch.bfloat16
    outs = []
    for patience in (None, "0"):
        if patience is not None:
            monkeypatch.setenv("BITSPARSE_LOOKBACK_PATIENCE", patience)
        buf = TensorBuffer(2 * z.numel(), device=dev, dtype=dt)
        sp = F.activate_and_compress(z.clone(), b, buf, False, store == "e4m3", True)[2]
        outs.append((sp.prefix, buf.vals, buf.offset))
    for x, y, what in zip(*outs, ("prefix", "values", "cursor")):
        _same(x, y, what)


@pytest.mark.parametrize("shape", [(1, 8), (64, 64), (65, 72), (80, 1416), (1000, 1024), (4100, 192)])
@pytest.mark.parametrize("store", ["bf16", "e4m3", "bf16_packed", "e4m3_packed"])
@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("zeros", [0.0, 0.5, 1.0])
def test_gradient_sums(dev, shape, store, square, zeros):
    from bitsparse_amd.src import functions as F
    from bitsparse_amd.src import hip_operators as H
    z, _ = _z(shape, 6, False, dev)
    z = z.abs() + 1 if zeros == 0.0 else (-z.abs() if zeros == 1.0 else z)
    pack = store.endswith("packed")
    if store.startswith("e4m3"):
        sp = F.quantize_and_compress(z.relu(), None, pack)[2]
    else:
        sp = F.dense_to_tilesparse(z.relu(), None, None, pack)
    g = torch.randn(shape, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).to(dev)
    want = g.clone()
    (H.relu2_grad_sparse_ if square else H.mask_with_bitmask_)(want, sp)
    assert H.act_grad_sums_supported(g, sp, square)
    sums, epoch = H.act_grad_sums_(g, sp, square, True, True)
    q, scale = H.quantize_e4m3fn(g, epoch)
    _same(want, g, "gradient")
    wq, wscale = H.quantize_e4m3fn(want, H.amax_into_workspace(want))
    _same(wscale.reshape(1), scale.reshape(1), "scale")
    _same(wq, q, "codes")
    w64 = want.double().sum(0)
    bound = shape[0] * 2.0 ** -24 * want.double().abs().sum(0) + 2.0 ** -8 * w64.abs() + 1e-30
    assert ((sums.double() - w64).abs() <= bound).all()


@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("store", ["bf16", "e4m3", "bf16_packed"])
@pytest.mark.parametrize("use_buffer", [False, True])
def test_block_equals_the_separate_nodes(dev, square, store, use_buffer, monkeypatch):
    """y, dx, dW1, dW2 bit for bit; the bias gradients to their rounding."""
    from bitsparse_amd import layers
    from bitsparse_amd.bitsparse import TensorBuffer
    g = torch.Generator().manual_seed(11)
    T, D, Hn = 208, 144, 528
    fp8, pack = store == "e4m3", store.endswith("packed")
    x = torch.randn((2, T // 2, D), generator=g).to(torch.bfloat16).to(dev)
    W1 = (0.1 * torch.randn((Hn, D), generator=g)).to(torch.bfloat16).to(dev)
    W2 = (0.1 * torch.randn((D, Hn), generator=g)).to(torch.bfloat16).to(dev)
    b1 = (0.1 * torch.randn(Hn, generator=g)).to(torch.bfloat16).to(dev)
    b2 = (0.1 * torch.randn(D, generator=g)).to(torch.bfloat16).to(dev)
    dY = torch.randn((2, T // 2, D), generator=g).to(torch.bfloat16).to(dev)
    dt = E4M3 if fp8 else torch.bfloat16
    layer, kw = (layers.FFNRelu2, "storage_dtype") if square else (layers.FFNRelu, "dtype")
    outs = []
    for block in (True, False):
        if not block:
            monkeypatch.setattr(layers, "_block_ok", lambda *a: False)
        p = [t.clone().requires_grad_() for t in (x, W1, W2, b1, b2)]
        buf = TensorBuffer(2 * T * Hn + 64, device=dev, dtype=dt, pack_sbit=pack) if use_buffer else None
        y = layer.apply(p[0], p[1], p[2], p[3], p[4], sparse_data=buf, pack_sbit=pack, **{kw: dt})
        y.backward(dY)
        outs.append([y.detach()] + [t.grad for t in p])
    for a, b, name in zip(outs[0][:4], outs[1][:4], ("y", "dx", "dW1", "dW2")):
        _same(a, b, name)
    for a, b, name in zip(outs[0][4:], outs[1][4:], ("db1", "db2")):
        # two bf16 roundings of fp32 sums
        assert ((a - b).double().abs() <= 2.0 ** -7 * b.double().abs() + 1e-2).all(), name


def _graph_node(t, name):
    """The autograd node of that name behind t."""
    nodes = [t.grad_fn]
    while nodes:
        n = nodes.pop()
        if n is not None and n.name() == name:
            return n
        nodes += [m for m, _ in n.next_functions] if n is not None else []
    raise AssertionError(f"no {name}")


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
            for saved in _graph_node(y, "_FFNBlockBackward")._raw_saved_tensors:
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
