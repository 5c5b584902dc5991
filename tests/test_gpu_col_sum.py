"""bs_col_sum (the bias gradients) against torch's sum in 64 bits."""
import pytest
import torch

from bitsparse_amd import _lib

pytestmark = pytest.mark.gpu


# one row, fewer rows than a row lane pass, remainders of the unrolled loop,
# columns ending inside a workgroup (256) and inside the second pass's 64
@pytest.mark.parametrize("shape", [(1, 8), (7, 264), (63, 256), (65, 1000), (129, 776), (1000, 3072), (4096, 72),
                                   (2055, 4096)])
def test_col_sum(dev, shape):
    g = torch.Generator().manual_seed(shape[0])
    x = torch.randn(shape, generator=g).to(torch.bfloat16)
    xd = x.to(dev)
    L, need = _lib.load(), _lib.load().bs_col_sum_workspace_bytes(*shape)
    out = torch.full((shape[1] + 8,), 7.0, device=dev, dtype=torch.bfloat16)
    part = torch.empty(need, device=dev, dtype=torch.uint8)
    _lib.check(L.bs_col_sum(xd.data_ptr(), *shape, out.data_ptr(), part.data_ptr(), need, _lib.stream_handle(xd.device)),
               "bs_col_sum")
    assert bool((out[shape[1]:] == 7).all())
    got, want = out[:shape[1]].cpu().double(), x.double().sum(0)
    # fp32 sums of R values: R * 2^-24 of the sum of magnitudes; then one bf16 rounding
    bound = shape[0] * 2.0 ** -24 * x.double().abs().sum(0) + 2.0 ** -8 * want.abs() + 1e-30
    assert ((got - want).abs() <= bound).all()
    assert torch.equal(_lib.native().col_sum(xd.requires_grad_()).cpu(),      # (its own sum: gradients on)
                       xd.sum(0).cpu())
    with torch.no_grad():
        assert torch.equal(_lib.native().col_sum(xd).cpu().view(torch.int16), out[:shape[1]].cpu().view(torch.int16))


@pytest.mark.parametrize("shape", [(5, 12), (0, 16), (40, 64)])
def test_col_sum_of_other_forms(dev, shape):
    """What the kernel does not take -- columns not in chunks of 8, no rows, a
    strided or misaligned matrix -- is summed all the same."""
    x = torch.randn(shape, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(dev)
    forms = [x, x.t().contiguous().t(), torch.nn.functional.pad(x, (0, 4))[:, :shape[1]]]
    if x.numel():
        forms.append(torch.cat([x.flatten()[:1], x.flatten()])[1:].view(shape))
    with torch.no_grad():
        for v in forms:
            got, want = _lib.native().col_sum(v).double(), x.double().sum(0)
            assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + shape[0] * 2.0 ** -23 * x.double().abs().sum(0)).all()


@pytest.mark.parametrize("buffer", [False, True], ids=["separate", "block"])
def test_ffn_bias_gradients(dev, buffer):
    """b1 and b2 of the layers, by the single node (a buffer to compress into)
    and the separate ones: column sums of the gradients they receive, for a
    3-D input and a gradient that is an expanded view."""
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd.layers import FFNRelu, FFNRelu2
    g = torch.Generator().manual_seed(5)
    x = torch.randn((3, 50, 64), generator=g).to(torch.bfloat16).to(dev)
    W1 = (0.1 * torch.randn((256, 64), generator=g)).to(torch.bfloat16).to(dev)
    W2 = (0.1 * torch.randn((72, 256), generator=g)).to(torch.bfloat16).to(dev)
    b1 = (0.1 * torch.randn(256, generator=g)).to(torch.bfloat16).to(dev)
    b2 = (0.1 * torch.randn(72, generator=g)).to(torch.bfloat16).to(dev)
    dY = torch.randn((3, 50, 72), generator=g).to(torch.bfloat16).to(dev)
    for layer, sq in ((FFNRelu, False), (FFNRelu2, True)):
        for grad in (dY, dY[:, :1].expand(3, 50, 72)):
            p = [t.clone().requires_grad_() for t in (x, W1, W2, b1, b2)]
            buf = TensorBuffer(2 * 150 * 256, device=dev) if buffer else None
            y = layer.apply(p[0], p[1], p[2], p[3], p[4], sparse_data=buf)
            assert (y.grad_fn.next_functions[0][0].name() == "_FFNBlockBackward") == buffer
            y.backward(grad)
            # the same bf16 GEMMs in plain autograd: dz differs at most by its rounding
            f = [t.clone().requires_grad_() for t in (x, W1, W2, b1, b2)]
            h = torch.relu(f[0] @ f[1].T + f[3])
            z_grad = []
            h.register_hook(lambda t: z_grad.append(t))
            ((h * h if sq else h) @ f[2].T + f[4]).backward(grad)
            dz = (z_grad[0] * (h > 0)).double().reshape(-1, 256)
            db1, db2 = dz.sum(0), grad.double().reshape(-1, 72).sum(0)
            # b2: one bf16 rounding of an fp32 sum; b1: 2^-7 per rounded term more
            assert ((p[4].grad.double() - db2).abs() <= 2.0 ** -8 * db2.abs() + 1e-4).all()
            assert ((p[3].grad.double() - db1).abs() <= 2.0 ** -8 * db1.abs() + 2.0 ** -7 * dz.abs().sum(0)).all()
