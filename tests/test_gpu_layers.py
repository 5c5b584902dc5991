"""Autograd layers with compressed activations against the dense-activation
comparators (experiments/experiment.py:242-384 semantics) on the same inputs.

Reference tolerance: experiment.py:24,160-164 compares loss and x.grad.std()
at 3e-6 for bf16.  Here every gradient tensor is compared: the forward output
and dx are bit-identical paths up to GEMM ordering, and dW2 comes from a
different GEMM (the reconstruct-into-LDS kernel vs hipBLASLt), so gradients
are compared to an fp32 CPU computation of the same math at bf16 tolerance
(2^-6 relative to the tensor's max)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _mlp_inputs(B, D, H, seed, shift=0.0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((B, D), generator=g).to(torch.bfloat16)
    W1 = (0.05 * torch.randn((H, D), generator=g) + shift).to(torch.bfloat16)
    W2 = (0.05 * torch.randn((D, H), generator=g)).to(torch.bfloat16)
    dY = torch.randn((B, D), generator=g).to(torch.bfloat16)
    return x, W1, W2, dY


def _close(a, b, name):
    scale = b.abs().max().item() + 1e-6
    err = (a.float().cpu() - b.float().cpu()).abs().max().item() / scale
    assert err < 2 ** -6, f"{name}: max error {err:.3e} of max |ref|"


@pytest.mark.parametrize("use_buffer", [False, True])
def test_ffn_relu_matches_dense(dev, use_buffer):
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd.dense import DenseFFNRelu
    from bitsparse_amd.layers import FFNRelu
    x, W1, W2, dY = _mlp_inputs(512, 256, 1024, seed=1)
    buf = TensorBuffer(2 * 512 * 1024, device=dev) if use_buffer else None
    xs, W1s, W2s = (t.to(dev).requires_grad_() for t in (x, W1, W2))
    y = FFNRelu.apply(xs, W1s, W2s, sparse_data=buf)
    y.backward(dY.to(dev))
    xd, W1d, W2d = (t.to(dev).requires_grad_() for t in (x, W1, W2))
    yd = DenseFFNRelu.apply(xd, W1d, W2d)
    yd.backward(dY.to(dev))
    assert torch.equal(y, yd)                         # same forward ops
    assert torch.equal(xs.grad, xd.grad)              # mask kernel == threshold_backward
    assert torch.equal(W1s.grad, W1d.grad)
    xf, W1f, W2f = (t.float().requires_grad_() for t in (x, W1, W2))
    (torch.relu(xf @ W1f.T) @ W2f.T).backward(dY.float())
    _close(W2s.grad, W2f.grad, "dW2")
    if buf is not None:
        assert not buf.overflowed()


def test_ffn_relu2_matches_dense(dev):
    from bitsparse_amd.dense import DenseFFNRelu2
    from bitsparse_amd.layers import FFNRelu2
    x, W1, W2, dY = _mlp_inputs(512, 256, 768, seed=2)
    xs, W1s, W2s = (t.to(dev).requires_grad_() for t in (x, W1, W2))
    ys = FFNRelu2.apply(xs, W1s, W2s)
    ys.backward(dY.to(dev))
    xd, W1d, W2d = (t.to(dev).requires_grad_() for t in (x, W1, W2))
    yd = DenseFFNRelu2.apply(xd, W1d, W2d)
    yd.backward(dY.to(dev))
    assert torch.equal(ys, yd)                        # the one-pass square and scale == square(); mul_(k)
    assert torch.equal(xs.grad, xd.grad)              # relu2 grad == grad_z * (2 k r)
    assert torch.equal(W1s.grad, W1d.grad)
    xf, W1f, W2f = (t.float().requires_grad_() for t in (x, W1, W2))
    (torch.relu(xf @ W1f.T).square() @ W2f.T).backward(dY.float())
    _close(W2s.grad, W2f.grad, "dW2")


def test_ffn_relu_leading_batch_dims_and_bias(dev):
    from bitsparse_amd.layers import FFNRelu
    g = torch.Generator().manual_seed(3)
    x = torch.randn((4, 64, 128), generator=g).to(torch.bfloat16).to(dev).requires_grad_()
    W1 = (0.05 * torch.randn((384, 128), generator=g)).to(torch.bfloat16).to(dev).requires_grad_()
    W2 = (0.05 * torch.randn((128, 384), generator=g)).to(torch.bfloat16).to(dev).requires_grad_()
    b1 = torch.zeros(384, dtype=torch.bfloat16, device=dev, requires_grad=True)
    b2 = torch.zeros(128, dtype=torch.bfloat16, device=dev, requires_grad=True)
    y = FFNRelu.apply(x, W1, W2, b1, b2)
    assert y.shape == (4, 64, 128)
    y.sum().backward()
    assert x.grad.shape == x.shape and b1.grad is not None and b2.grad is not None


def test_ffn_relu2_fp8_storage_matches_fp8_dense(dev):
    """fp8 (e4m3fn) activation storage against the reference's fp8 dense
    comparator (experiment.py:330-384 with an fp8 DTYPE).  Both run every GEMM
    in per-tensor fp8; they differ only in bf16 rounding order of the ReLU^2
    reconstruction, which can move an fp8 re-quantization by one step, so the
    bound is fp8-sized: 2^-3 of each tensor's max."""
    from bitsparse_amd.dense import DenseFFNRelu2Fp8
    from bitsparse_amd.layers import FFNRelu2
    x, W1, W2, dY = _mlp_inputs(256, 256, 512, seed=4)
    xs, W1s, W2s = (t.to(dev).requires_grad_() for t in (x, W1, W2))
    ys = FFNRelu2.apply(xs, W1s, W2s, storage_dtype=torch.float8_e4m3fn)
    ys.backward(dY.to(dev))
    xd, W1d, W2d = (t.to(dev).requires_grad_() for t in (x, W1, W2))
    yd = DenseFFNRelu2Fp8.apply(xd, W1d, W2d)
    yd.backward(dY.to(dev))
    for name, a, b in (("y", ys, yd), ("dx", xs.grad, xd.grad), ("dW1", W1s.grad, W1d.grad),
                       ("dW2", W2s.grad, W2d.grad)):
        scale = b.abs().max().item() + 1e-6
        err = (a.float() - b.float()).abs().max().item() / scale
        assert err < 2 ** -3, f"{name}: {err:.3e}"


@pytest.mark.parametrize("k", [1.0, 0.5, 3.0])
@pytest.mark.parametrize("case", ["finite", "inf", "nan"])
def test_relu2_square_amax_matches_torch_ops(dev, k, case):
    """The fused pass of the fp8 ReLU^2 forward (reference layers.py:103-120:
    h.square_(); h.mul_(k); to_fp8(h)) against torch's own ops on the same GPU:
    h bit for bit (-0, subnormals, negatives; with Inf, or NaN of both signs,
    or values whose square overflows), then the amax it leaves gives the same
    codes and the same scale bits as to_fp8(h)."""
    from bitsparse_amd.fp8 import to_fp8
    from bitsparse_amd.src import hip_operators as H
    from tests.helpers import special_bf16
    xb = special_bf16((257, 136), seed=31).view(torch.int16).clone()
    mag = xb.view(torch.int16).to(torch.int32) & 0x7fff
    xb[mag >= 0x7f80] = 0x3f80                           # no Inf / NaN unless asked for
    xb[mag == 0x7f7f] = 0x4100
    if case == "inf":
        xb.view(-1)[:3] = torch.tensor([0x7f80, -0x80, 0x5f80], dtype=torch.int16)   # +-Inf, 2^64 (square -> Inf)
    if case == "nan":
        xb.view(-1)[:2] = torch.tensor([0x7fc0, -0x40], dtype=torch.int16)           # +-NaN
    x = xb.to(dev).view(torch.bfloat16)
    want = x.clone()
    want.square_()
    want.mul_(k)
    h = x.clone()
    epoch = H.relu2_square_amax_(h, k)
    assert torch.equal(h.view(torch.int16), want.view(torch.int16))
    q, s = H.quantize_e4m3fn(h, epoch)
    qt, st = to_fp8(want)
    assert torch.equal(q.view(torch.uint8), qt.view(torch.uint8))
    assert torch.equal(s.view(torch.int32), st.view(torch.int32))
    if case == "finite":
        assert 0 < int((q.view(torch.uint8) & 0x7f).max().item()) < 0x7f   # real codes, not NaN


def test_ffn_relu2_fp8_forward_bit_identical_to_dense(dev):
    """With the fused square / scale / amax pass the compressed fp8 layer's y
    is bit-identical to the fp8 dense comparator's (the same h8, scale and
    GEMM), and z ends up holding k * relu(z)^2 as the in-place ops leave it."""
    from bitsparse_amd.dense import DenseFFNRelu2Fp8
    from bitsparse_amd.fp8 import matmul
    from bitsparse_amd.layers import FFNRelu2, Relu2Linear
    from bitsparse_amd.config import RELU2_SCALE
    x, W1, W2, _ = _mlp_inputs(256, 256, 512, seed=9)
    xs, W1s, W2s = (t.to(dev) for t in (x, W1, W2))
    ys = FFNRelu2.apply(xs, W1s, W2s, storage_dtype=torch.float8_e4m3fn)
    yd = DenseFFNRelu2Fp8.apply(xs, W1s, W2s)
    assert torch.equal(ys.view(torch.int16), yd.view(torch.int16))
    z = matmul(xs, W1s.T, True)
    want = z.clone().relu_()
    want.square_()
    want.mul_(RELU2_SCALE)
    Relu2Linear.apply(z, W2s, None, False, torch.float8_e4m3fn)
    assert torch.equal(z.view(torch.int16), want.view(torch.int16))


def _relu2_special_inputs(dev, B=304, D=192, H=528, seed=9):
    """MLP operands for the ReLU^2 layer (B and H not multiples of 64, but
    multiples of 16 as the fp8 library GEMMs need); the test writes -0,
    +-Inf, +-NaN and values whose square overflows bf16 into z."""
    x, W1, W2, dY = _mlp_inputs(B, D, H, seed=seed, shift=0.01)
    return [t.to(dev) for t in (x, W1, W2, dY)]


@pytest.mark.parametrize("storage", ["bf16", "e4m3fn"])
def test_relu2_square_fused_into_compress(dev, monkeypatch, storage):
    """Relu2Linear with the square written back by the compress pass (and,
    for fp8 storage, amax|k r^2| derived from amax|r|) against the same layer
    with the separate in-place square / square-and-amax pass: the output, z
    after the forward (k r^2, as the reference's in-place ops leave it), the
    compressed r and every gradient are bit-identical, on ordinary and on
    special pre-activations (-0, +-Inf, +-NaN, squares past bf16's range)."""
    from bitsparse_amd import layers
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd.src import functions as F
    dt = torch.bfloat16 if storage == "bf16" else torch.float8_e4m3fn
    x, W1, W2, dY = _relu2_special_inputs(dev)
    z0 = (x @ W1.T).contiguous()
    zb = z0.view(torch.int16).view(-1)
    zb[[0, 7, 64, 200, 333, 4099, 7000, 9001]] = torch.tensor(
        [-32768, 0x7f80, -128, 0x7fc0, -64, 0x7f7f, 0x5f00, -0x1f00], dtype=torch.int16, device=dev)
    for special in (False, True):
        z_in = z0 if special else (x @ W1.T).contiguous()
        if special and storage == "e4m3fn":
            z_in = z_in.clone()
            z_in.view(-1)[[200, 4099]] = 1.0        # no NaN / Inf: a finite scale for the codes
        outs = []
        for fused in (True, False):
            if not fused:
                monkeypatch.setattr(F, "relu2_fused_ok", lambda *a: False)
                monkeypatch.setattr(layers, "relu2_fused_ok", lambda *a: False)
            buf = TensorBuffer(z_in.numel() * (2 if storage == "bf16" else 1), device=dev, dtype=dt)
            z = z_in.clone().requires_grad_()
            Wq = W2.clone().requires_grad_()
            y = layers.Relu2Linear.apply(z, Wq, buf, False, dt)
            zf = z.detach().clone()
            y.backward(dY)
            nbytes = int(buf.offset.item()) * buf.vals.element_size()
            outs.append((y.detach(), zf, z.grad, Wq.grad, buf.vals.view(torch.uint8)[:nbytes].clone()))
            monkeypatch.undo()
        for a, b, name in zip(outs[0], outs[1], ("y", "z after forward", "dz", "dW2", "stored values")):
            assert a.shape == b.shape, name
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), (name, special)


@pytest.mark.parametrize("k", [1.0, 0.5, 3.0, -2.0, 0.0])
def test_relu2_amax_derived_from_relu_amax(dev, k):
    """amax|bf16(bf16(r*r) * k)| from amax|relu(z)| (bs_amax_relu2_from)
    equals the amax the square-and-amax pass takes of the squared tensor,
    through the quantizer's output, for ordinary, huge and NaN inputs."""
    from bitsparse_amd.src import hip_operators as H
    g = torch.Generator().manual_seed(int(abs(k) * 10) + 3)
    for kind in ("normal", "huge", "nan", "all_negative"):
        z = torch.randn((257, 333), generator=g).to(torch.bfloat16)
        if kind == "huge":
            z[5, 7] = 3.0e19
        elif kind == "nan":
            z[100, 3] = float("nan")
        elif kind == "all_negative":
            z = -z.abs() - 1
        z = z.to(dev)
        r = z.relu()
        e1 = H.amax_into_workspace(z, relu=True, reserve=2)
        e2 = H.amax_relu2_from(z.device, e1, k)
        q_derived, s_derived = H.quantize_e4m3fn(r.clone(), e2)    # a quantizer over any tensor with that amax
        h = r.clone()
        e3 = H.relu2_square_amax_(h, k)
        q_pass, s_pass = H.quantize_e4m3fn(r.clone(), e3)
        sd, sp = float(s_derived.item()), float(s_pass.item())
        assert (sd == sp) or (sd != sd and sp != sp), (kind, sd, sp)
        if sd == sd:
            assert torch.equal(q_derived.view(torch.uint8), q_pass.view(torch.uint8)), kind
