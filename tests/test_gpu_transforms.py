"""The layers under torch's function transforms and tracers."""
import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn
T, D, H = 128, 64, 256


def _operands(dev):
    g = torch.Generator().manual_seed(3)
    p = [(m * torch.randn(s, generator=g)).to(torch.bfloat16).to(dev).requires_grad_()
         for s, m in (((T, D), 1.0), ((H, D), 0.1), ((D, H), 0.1), ((H,), 0.1), ((D,), 0.1))]
    return p, torch.randn((T, D), generator=g).to(torch.bfloat16).to(dev)


def _layer(square, dtype, buf):
    from bitsparse_amd.layers import FFNRelu, FFNRelu2
    layer, kw = (FFNRelu2, "storage_dtype") if square else (FFNRelu, "dtype")
    return lambda *p: layer.apply(*p, sparse_data=buf, **{kw: dtype})


def _buf(dev, dtype, buffer):
    from bitsparse_amd.bitsparse import TensorBuffer
    return TensorBuffer(2 * T * H, device=dev, dtype=dtype) if buffer else None


@pytest.mark.parametrize("buffer", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, E4M3])
def test_function_transforms_are_refused_alike(dev, dtype, buffer):
    """torch.func transforms do not take autograd functions of this kind: one
    error, whichever path the layer would go."""
    p, _ = _operands(dev)
    rest = [t.detach() for t in p[1:]]
    fn = _layer(True, dtype, _buf(dev, dtype, buffer))
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.func.grad(lambda x: fn(x, *rest).float().sum())(p[0].detach())
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.vmap(lambda x: fn(x, *rest))(p[0].detach().reshape(2, T // 2, D))


