"""The streaming compress at the extremes of a round (64 chunks, 8 tile rows):
empty and full rounds side by side in every order inside a tile, and the fused
ReLU over every bf16 bit pattern.  Bit for bit, for raw and streamed
(nontemporal) values."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import bits, from_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[False, True], ids=["cached", "streamed"])
def streamed(request, dev):
    from bitsparse_amd import _lib
    L = _lib.load()
    prev = L.bs_nontemporal_min_bytes(0) if request.param else None
    yield request.param
    if prev is not None:
        L.bs_nontemporal_min_bytes(prev)


# a tile's rounds are 8 rows each: round k of tile t is full iff bit k of t,
# so a 16 x 16 grid of tiles has every combination of empty and full rounds
# (totals 0, 512 and runs of 0 .. 4096 values)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("N", [1024, 1021])
def test_empty_and_full_rounds(dev, streamed, dtype, N):
    from bitsparse_amd.bitsparse import TensorBuffer
    from bitsparse_amd.src.functions import dense_to_tilesparse
    M = 1024
    r, c = np.arange(M)[:, None], np.arange(N)[None, :]
    full = ((r // 64 * 16 + c // 64) >> (r % 64 // 8)) & 1
    v = (1 + (r * 31 + c * 7) % 64) * full                   # small integers are exact in both types
    x = torch.from_numpy(v.astype(np.float32)).to(dtype)
    kind = O.BF16 if dtype == torch.bfloat16 else O.E4M3FN
    bm, pf, vals = O.compress(bits(x), kind)
    buf = TensorBuffer(x.numel() * x.element_size(), device=dev, dtype=dtype)
    for sp in (dense_to_tilesparse(x.to(dev), None, buf), dense_to_tilesparse(x.to(dev), None)):
        assert (bits(sp.bitmask) == bm).all() and (bits(sp.prefix) == pf).all()
        assert (bits(sp.vals)[:vals.size] == vals).all()


@pytest.mark.parametrize("N", [256, 255])
def test_relu_every_bit_pattern(dev, streamed, N):
    """x <= 0 becomes +0; NaN of either sign and positives keep their bits."""
    from bitsparse_amd.src import hip_operators as H
    M = 65536 // N + 1
    zb = np.resize(np.random.default_rng(5).permutation(np.arange(65536, dtype=np.uint32)), (M, N)).astype(np.uint16)
    rb = np.where((zb >= 0x8000) & (zb <= 0xff80), 0, zb).astype(np.uint16)
    bm, pf, vals = O.compress(rb, O.BF16)
    z = from_bits(zb, torch.bfloat16).to(dev)
    out, got_v = torch.empty_like(z), torch.empty(M * N, dtype=torch.bfloat16, device=dev)
    got_bm = torch.empty(bm.size, dtype=torch.uint8, device=dev)
    got_pf = torch.empty(pf.size, dtype=torch.uint32, device=dev)
    H.compress_into(z, got_bm, got_pf, got_v, None, None, None, relu=True, relu_out=out)
    assert (bits(out) == rb).all()
    assert (bits(got_bm) == bm.reshape(-1)).all() and (bits(got_pf) == pf).all()
    assert (bits(got_v)[:vals.size] == vals).all()
