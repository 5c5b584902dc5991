"""Rows whose length is no multiple of 8 elements (chunks at any alignment, a
partial chunk at each row's end) against the oracle, bit for bit."""
import pytest
import torch

from oracle import oracle as O
from tests.helpers import bits, relu_input

pytestmark = pytest.mark.gpu

KIND = {torch.bfloat16: O.BF16, torch.float8_e4m3fn: O.E4M3FN, torch.float8_e5m2: O.E5M2}


# every remainder of 8, below and above one chunk, one tile and one unit of 8
# tiles; last tile rows of 1, 57 and 64 rows
@pytest.mark.parametrize("N", [1, 7, 8, 9, 10, 13, 63, 65, 71, 127, 515, 2049])
@pytest.mark.parametrize("M", [1, 64, 121])
@pytest.mark.parametrize("dtype", list(KIND))
def test_compress_and_decompress(dev, M, N, dtype):
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd.src.functions import dense_to_tilesparse
    from bitsparse_amd.src.hip_operators import unpack_batch_
    x = relu_input((M, N), 0.5, seed=N, dtype=dtype)
    bm, pf, v = O.compress(bits(x), KIND[dtype])
    buf = TensorBuffer(x.numel() * x.element_size(), device=dev, dtype=dtype)
    for sp in (dense_to_tilesparse(x.to(dev), None, buf), dense_to_tilesparse(x.to(dev), None)):
        assert (bits(sp.bitmask) == bm).all() and (bits(sp.prefix) == pf).all()
        assert (bits(sp.vals)[:v.size] == v).all()
        out = torch.full((M * N + 16,), 7, device=dev, dtype=torch.uint8 if x.element_size() == 1 else torch.int16)
        got = out[:M * N].view(dtype).view(M, N)
        unpack_batch_(sp, got, 0, sp.grid_n, N, M, sp.num_tiles)
        assert (bits(got) == bits(x)).all() and bool((out[M * N:] == 7).all())


@pytest.mark.parametrize("N", [9, 71, 515])
@pytest.mark.parametrize("M", [1, 121])
def test_quantizing_and_gradients(dev, M, N):
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd.src import functions as F
    from bitsparse_amd.src import hip_operators as H
    x = relu_input((M, N), 0.5, seed=N + 1) * 3
    qo, so = O.to_fp8(bits(x))
    bm, pf, v = O.compress(qo, O.E4M3FN)
    buf = TensorBuffer(x.numel(), device=dev, dtype=torch.float8_e4m3fn)
    q, s, sp = F.quantize_and_compress(x.to(dev), buf)
    assert float(s.item()) == so and (bits(q) == qo).all()
    assert (bits(sp.bitmask) == bm).all() and (bits(sp.prefix) == pf).all()
    assert (bits(sp.vals)[:v.size] == v).all()
    g = torch.randn((M, N), generator=torch.Generator().manual_seed(2)).to(torch.bfloat16)
    spb = F.dense_to_tilesparse(x.to(dev), None)
    masked = H.mask_with_bitmask_(g.to(dev), spb).cpu()
    assert torch.equal(masked.view(torch.int16), torch.where(x > 0, g, torch.zeros_like(g)).view(torch.int16))
    r2 = H.relu2_grad_sparse_(g.to(dev), spb).cpu()
    want = torch.where(x > 0, (g.float() * (2.0 * x.float())).to(torch.bfloat16), torch.zeros_like(g))
    assert torch.equal(r2.view(torch.int16), want.view(torch.int16))
