"""GPU parity of the HIP codec kernels against the CPU oracle.

Bar: bit-exact for bitmask, prefix, values, decompressed tiles and the
gradient kernels; at the 16384x16384 size (beyond the oracle's budget)
size-independent properties are checked with torch ops on the GPU.
Everything goes through bitsparse_amd's ctypes binding of the C ABI.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import all_fp8_patterns, bits, from_bits, preact_input, relu_input, special_bf16

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (64, 64), (128, 128), (129, 131), (200, 70), (5, 300), (256, 8), (320, 1024)]
SPARSITIES = [0.0, 0.5, 0.9, 1.0]


def _bs():
    import bitsparse_amd.src.functions as F
    import bitsparse_amd.src.hip_operators as H
    from bitsparse_amd.bitsparse import TensorBuffer
    return F, H, TensorBuffer


def decompress(sparse):
    _, H, _ = _bs()
    M, N = sparse.shape
    out = torch.empty((M, N), device=sparse.vals.device, dtype=sparse.vals.dtype)
    return H.unpack_batch_(sparse, out, 0, sparse.grid_n, N, M, sparse.grid_m * sparse.grid_n)


def check_sparse(sp, x_cpu, code):
    bm, pf, v = O.compress(bits(x_cpu), code)
    assert (bits(sp.bitmask) == bm).all(), "bitmask"
    assert (bits(sp.prefix) == pf).all(), "prefix"
    off = int(sp.vals_offset.reshape(-1)[0].item())
    got = bits(sp.vals)[off:off + v.size]
    assert (got == v).all(), "vals"
    return bm, pf, v


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("sparsity", SPARSITIES)
def test_compress_standalone_bf16(dev, shape, sparsity):
    F, _, _ = _bs()
    x = relu_input(shape, sparsity, seed=1)
    sp = F.dense_to_tilesparse(x.to(dev), None)
    bm, pf, v = check_sparse(sp, x, O.BF16)
    assert sp.vals.numel() == v.size
    d = decompress(sp)
    assert torch.equal(d.cpu(), x)


@pytest.mark.parametrize("shape", SHAPES)
def test_compress_special_values(dev, shape):
    F, _, TB = _bs()
    x = special_bf16(shape, seed=2)
    sp = F.dense_to_tilesparse(x.to(dev), None)
    bm, pf, v = check_sparse(sp, x, O.BF16)
    buf = TB(2 * max(1, x.numel()), device=dev)
    sp2 = F.dense_to_tilesparse(x.to(dev), None, buf)
    check_sparse(sp2, x, O.BF16)
    ref = O.decompress(v, O.BF16, bm, pf, *shape)
    assert (bits(decompress(sp)) == ref).all()
    assert (bits(decompress(sp2)) == ref).all()


@pytest.mark.parametrize("dt,code", [(torch.float8_e4m3fn, O.E4M3FN), (torch.float8_e5m2, O.E5M2)])
@pytest.mark.parametrize("shape", [(64, 64), (129, 131), (70, 200), (512, 384)])
def test_compress_fp8_inputs(dev, dt, code, shape):
    F, _, TB = _bs()
    xb = all_fp8_patterns(shape, seed=3)
    x = from_bits(xb, dt)
    sp = F.dense_to_tilesparse(x.to(dev), torch.ones((), device=dev))
    bm, pf, v = check_sparse(sp, x, code)
    assert (bits(decompress(sp)) == O.decompress(v, code, bm, pf, *shape)).all()
    buf = TB(x.numel() + 64, device=dev, dtype=dt)
    sp2 = F.dense_to_tilesparse(x.to(dev), None, buf)
    check_sparse(sp2, x, code)


def test_shared_buffer_decompress_after_all_writes(dev):
    """validate.py:128-139: several tensors share one TensorBuffer; every
    tensor is decompressed only after all were written."""
    F, _, TB = _bs()
    xs = [relu_input(s, sp, seed=10 + i) for i, (s, sp) in
          enumerate([(s, sp) for s in [(128, 128), (129, 131)] for sp in SPARSITIES])]
    cap = sum(x.numel() for x in xs)
    buf = TB(2 * cap, device=dev)
    sps = [F.dense_to_tilesparse(x.to(dev), None, buf) for x in xs]
    total = 0
    for x, sp in zip(xs, sps):
        assert sp.vals is buf.vals
        assert int(sp.vals_offset.item()) == total
        check_sparse(sp, x, O.BF16)
        assert torch.equal(decompress(sp).cpu(), x)
        total += int((x.float() > 0).sum())
    assert int(buf.offset.item()) == total
    assert not buf.overflowed()
    buf.reset_buffer()
    assert int(buf.offset.item()) == 0


def test_buffer_overflow_is_flagged_and_contained(dev):
    F, _, TB = _bs()
    x = relu_input((256, 256), 0.0, seed=20)          # 65536 positives
    buf = TB(2 * 1000, device=dev)
    guard = torch.full((1000 + 4096,), 0x1234, dtype=torch.int16, device=dev).view(torch.bfloat16)
    buf.vals = guard[:1000]                           # capacity 1000, guard region behind it
    sp = F.dense_to_tilesparse(x.to(dev), None, buf)
    torch.cuda.synchronize()
    assert buf.overflowed()
    assert (guard[1000:].view(torch.int16) == 0x1234).all()
    v = O.compress(bits(x), O.BF16)[2]
    assert (bits(guard[:1000]) == v[:1000]).all()


def test_empty_inputs(dev):
    F, _, TB = _bs()
    for shape in [(0, 5), (5, 0), (0, 0)]:
        x = torch.zeros(shape, dtype=torch.bfloat16, device=dev)
        sp = F.dense_to_tilesparse(x, None)
        assert sp.prefix.numel() == 1 and int(sp.prefix[0].item()) == 0
        assert sp.vals.numel() == 0
        buf = TB(64, device=dev)
        sp = F.dense_to_tilesparse(x, None, buf)
        assert int(buf.offset.item()) == 0


def test_c1_round_trip_bit_exact(dev):
    """4096x4096 bf16, pre-activation N(0,1) seed 0, ReLU, compress,
    decompress; bit-exact against the oracle."""
    F, _, TB = _bs()
    x = torch.randn((4096, 4096), generator=torch.Generator().manual_seed(0)).to(torch.bfloat16).relu()
    bm, pf, v = O.compress(bits(x), O.BF16)
    buf = TB(2 * x.numel(), device=dev)
    sp = F.dense_to_tilesparse(x.to(dev), None, buf)
    assert (bits(sp.bitmask) == bm).all() and (bits(sp.prefix) == pf).all()
    assert (bits(sp.vals)[:v.size] == v).all()
    assert torch.equal(decompress(sp).cpu(), x)
    sp2 = F.dense_to_tilesparse(x.to(dev), None)
    assert (bits(sp2.vals) == v).all()


def _torch_tile_bitmask(x: torch.Tensor) -> torch.Tensor:
    """Bitmask of a [M, N] GPU tensor (M, N multiples of 64) with torch ops."""
    M, N = x.shape
    pos = (x.float() > 0).to(torch.uint8)
    t = pos.reshape(M // 64, 64, N // 64, 64).permute(0, 2, 1, 3).reshape(-1, 512, 8)
    w = (2 ** torch.arange(8, device=x.device, dtype=torch.int32)).to(torch.uint8)
    return (t * w).sum(-1, dtype=torch.int32).to(torch.uint8).reshape(-1)


@pytest.mark.parametrize("quant", [False, True])
def test_lookback_fallback_path(dev, monkeypatch, quant):
    """The compress look-back's safety net: with BITSPARSE_LOOKBACK_PATIENCE=0 a
    unit that finds a predecessor unpublished counts that predecessor's tiles
    from the dense input at once.  Every wave still finishes (each wait ends
    after one poll); the output must be bit-identical to the normal path and
    the fallback counter must show the path ran."""
    from bitsparse_amd import _lib
    from bitsparse_amd.src.functions import dense_to_tilesparse, quantize_and_compress
    M, N = 8192, 8192
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn((M, N), device=dev, generator=g).to(torch.bfloat16).relu_()

    def run():
        if quant:
            _, _, sp = quantize_and_compress(x, None)
        else:
            sp = dense_to_tilesparse(x, None)
        torch.cuda.synchronize()
        return sp

    ref = run()
    ws = _lib.workspace_for(x.device)
    before = ws.fallback_count()
    monkeypatch.setenv("BITSPARSE_LOOKBACK_PATIENCE", "0")
    got = run()
    after = ws.fallback_count()
    monkeypatch.delenv("BITSPARSE_LOOKBACK_PATIENCE")
    assert after > before
    assert torch.equal(got.bitmask, ref.bitmask)
    assert torch.equal(got.prefix, ref.prefix)
    n = int(ref.prefix[-1].item())
    assert torch.equal(got.vals[:n].view(torch.uint8), ref.vals[:n].view(torch.uint8))


@pytest.mark.parametrize("shape", [(129, 131), (300, 200), (448, 512)])
def test_unpack_row_batches(dev, shape):
    F, H, _ = _bs()
    x = relu_input(shape, 0.5, seed=30)
    sp = F.dense_to_tilesparse(x.to(dev), None)
    M, N = shape
    gn = sp.grid_n
    bm, pf, v = O.compress(bits(x), O.BF16)
    for first in range(sp.grid_m):
        for nrows in (1, 2):
            if first + nrows > sp.grid_m:
                continue
            rows = min(nrows * 64, M - first * 64)
            out = torch.empty((rows, N), dtype=torch.bfloat16, device=dev)
            H.unpack_batch_(sp, out, first, gn, N, rows, nrows * gn)
            ref = O.unpack(v, O.BF16, bm, pf, 0, first, gn, N, rows, nrows * gn)
            assert (bits(out) == ref).all()


@pytest.mark.parametrize("code", [O.E4M3FN, O.E5M2])
@pytest.mark.parametrize("shape", [(129, 144), (448, 512), (300, 200), (70, 24)])
@pytest.mark.parametrize("packed", [False, True])
def test_unpack_row_batches_fp8(dev, code, shape, packed):
    """fp8 storage decompressed in row batches, bit-exact against the oracle.
    Rows of whole 16-byte pieces (K % 16 == 0) take the 16-byte-store kernel,
    other widths and an output that is not 16-byte aligned the chunk kernel."""
    F, H, _ = _bs()
    dt = torch.float8_e4m3fn if code == O.E4M3FN else torch.float8_e5m2
    x = from_bits(all_fp8_patterns(shape, seed=31), dt)
    xr = torch.where(x.float() > 0, x.float(), torch.zeros(())).to(dt)     # stored values are positive
    sp = F.dense_to_tilesparse(xr.to(dev), None, pack_sbit=packed)
    M, N = shape
    gn = sp.grid_n
    bm, pf, v = O.compress(bits(xr), code)
    for first in range(sp.grid_m):
        for nrows in (1, 2):
            if first + nrows > sp.grid_m:
                continue
            rows = min(nrows * 64, M - first * 64)
            ref = O.unpack(v, code, bm, pf, 0, first, gn, N, rows, nrows * gn)
            out = torch.empty((rows, N), dtype=dt, device=dev)
            H.unpack_batch_(sp, out, first, gn, N, rows, nrows * gn)
            assert (bits(out) == ref).all()
            # the same batch into an output 8 bytes past a 16-byte boundary
            raw = torch.empty(rows * N + 16, dtype=torch.uint8, device=dev)
            out8 = raw[8:8 + rows * N].view(dt).view(rows, N)
            H.unpack_batch_(sp, out8, first, gn, N, rows, nrows * gn)
            assert (bits(out8) == ref).all()


def test_relu_grad(dev):
    F, H, _ = _bs()
    for shape in [(129, 131), (512, 768), (64, 8)]:
        x = special_bf16(shape, seed=40)
        g = preact_input(shape, seed=41)
        sp = F.dense_to_tilesparse(x.to(dev), None)
        gd = g.to(dev)
        out = H.mask_with_bitmask_(gd, sp)
        assert out is gd
        bm = O.compress(bits(x), O.BF16)[0]
        assert (bits(out) == O.relu_grad(bits(g), bm)).all()


@pytest.mark.parametrize("shape", [(129, 131), (256, 512), (64, 24)])
def test_relu2_grad_bf16(dev, shape):
    F, H, _ = _bs()
    r = preact_input(shape, seed=50).relu()
    g = preact_input(shape, seed=51)
    sp = F.dense_to_tilesparse(r.to(dev), None)
    out = H.relu2_grad_sparse_(g.to(dev), sp)
    bm, pf, v = O.compress(bits(r), O.BF16)
    assert (bits(out) == O.relu2_grad(bits(g), v, O.BF16, bm, pf)).all()


@pytest.mark.parametrize("shape", [(129, 131), (256, 512)])
def test_relu2_grad_and_square_fp8_scaled(dev, shape):
    F, H, TB = _bs()
    xb = all_fp8_patterns(shape, seed=52)
    xb[(xb & 0x7F) == 0x7F] = 0x10            # NaN-free payloads
    x = from_bits(xb, torch.float8_e4m3fn)
    g = preact_input(shape, seed=53)
    s = torch.tensor(0.0123, device=dev)
    buf = TB(x.numel() + 100, device=dev, dtype=torch.float8_e4m3fn)
    buf.offset.fill_(37)
    sp = F.dense_to_tilesparse(x.to(dev), s, buf)
    bm, pf, v = O.compress(xb, O.E4M3FN)
    out = H.relu2_grad_sparse_(g.to(dev), sp)
    assert (bits(out) == O.relu2_grad(bits(g), v, O.E4M3FN, bm, pf, scale=0.0123)).all()
    sq = torch.empty(shape, dtype=torch.bfloat16, device=dev)
    H.unpack_relu2_batch_(sp, sq, 0, sp.grid_n, shape[1], shape[0], sp.grid_m * sp.grid_n)
    ref = O.decompress(v, O.E4M3FN, bm, pf, *shape, square=True)
    ref = O.bf16_mul_scalar_tensor(ref, float(np.float32(0.0123) * np.float32(0.0123)))
    assert (bits(sq) == ref).all()


def test_relu2_paths_every_bit_pattern(dev):
    """relu2_grad and the ReLU^2 unpack over every stored value and every
    gradient bit pattern: bf16 r and g each a permutation of all 65536
    patterns (r's positives, +Inf included, are the stored values; g's NaN
    payloads, denormals, infinities and zeros all meet every kind of r), and
    e4m3fn storage with every fp8 pattern and a scale.  Bit-exact against the
    oracle, so every rounding inside the kernels (products to bf16 with RNE,
    NaN kept quiet) is pinned on all the inputs they can receive."""
    F, H, TB = _bs()
    rng = np.random.default_rng(70)
    shape = (256, 256)
    rb = rng.permutation(np.arange(65536, dtype=np.uint32)).astype(np.uint16).reshape(shape)
    gb = rng.permutation(np.arange(65536, dtype=np.uint32)).astype(np.uint16).reshape(shape)
    r, g = from_bits(rb, torch.bfloat16), from_bits(gb, torch.bfloat16)
    sp = F.dense_to_tilesparse(r.to(dev), None)
    bm, pf, v = O.compress(rb, O.BF16)
    out = H.relu2_grad_sparse_(g.to(dev), sp)
    assert (bits(out) == O.relu2_grad(gb, v, O.BF16, bm, pf)).all(), "relu2_grad bf16"
    sq = torch.empty(shape, dtype=torch.bfloat16, device=dev)
    H.unpack_relu2_batch_(sp, sq, 0, sp.grid_n, shape[1], shape[0], sp.grid_m * sp.grid_n)
    assert (bits(sq) == O.decompress(v, O.BF16, bm, pf, *shape, square=True)).all(), "unpack_relu2 bf16"

    xb = all_fp8_patterns(shape, seed=71)
    x = from_bits(xb, torch.float8_e4m3fn)
    for s in (0.0123, 3.0e4):
        st = torch.tensor(s, device=dev)
        spq = F.dense_to_tilesparse(x.to(dev), st)
        bmq, pfq, vq = O.compress(xb, O.E4M3FN)
        outq = H.relu2_grad_sparse_(g.to(dev), spq)
        assert (bits(outq) == O.relu2_grad(gb, vq, O.E4M3FN, bmq, pfq, scale=s)).all(), f"relu2_grad e4m3fn s={s}"
        H.unpack_relu2_batch_(spq, sq, 0, spq.grid_n, shape[1], shape[0], spq.grid_m * spq.grid_n)
        ref = O.decompress(vq, O.E4M3FN, bmq, pfq, *shape, square=True)
        ref = O.bf16_mul_scalar_tensor(ref, float(np.float32(s) * np.float32(s)))
        assert (bits(sq) == ref).all(), f"unpack_relu2 e4m3fn s={s}"


def test_unpack_relu2_bf16(dev):
    F, H, _ = _bs()
    r = relu_input((129, 131), 0.5, seed=54)
    sp = F.dense_to_tilesparse(r.to(dev), None)
    sq = torch.empty((129, 131), dtype=torch.bfloat16, device=dev)
    H.unpack_relu2_batch_(sp, sq, 0, sp.grid_n, 131, 129, sp.grid_m * sp.grid_n)
    assert torch.equal(sq.cpu(), r.square())


def test_torch_scalar_tensor_multiply_semantics(dev):
    """Pins the oracle's rule for bf16_tensor.mul_(fp32 0-d device tensor)
    (triton_operators.py:160-161, :200-201) against torch on the GPU."""
    x = preact_input((257, 129), seed=60)
    for s in [0.0123, 1.0 / 3.0, 7.77e-5, 3.14159]:
        st = torch.tensor(s, dtype=torch.float32, device=dev)
        got = x.to(dev).mul_(st)
        assert (bits(got) == O.bf16_mul_scalar_tensor(bits(x), s)).all()
        sq = x.to(dev).mul_(st.square())
        assert (bits(sq) == O.bf16_mul_scalar_tensor(bits(x), float(np.float32(s) * np.float32(s)))).all()


@pytest.mark.parametrize("shape", [(1, 1), (129, 131), (1000, 4096)])
def test_to_fp8(dev, shape):
    from bitsparse_amd.fp8 import to_fp8
    x = preact_input(shape, seed=70) * 5
    q, s = to_fp8(x.to(dev))
    qo, so = O.to_fp8(bits(x))
    assert s.dtype == torch.float32 and float(s.item()) == so
    assert (bits(q) == qo).all()
    qt, st = to_fp8(x.to(dev).T)
    assert qt.shape == x.T.shape and (bits(qt.contiguous()) == qo.T).all()


def test_to_fp8_misaligned_input(dev):
    """A contiguous view starting 2 bytes into its storage, of odd length: the
    amax and the quantizer take their per-element paths (no 16-byte vectors),
    the quantizer reading each code from its LDS table."""
    from bitsparse_amd.fp8 import to_fp8
    x = preact_input((1000, 4097), seed=75) * 5
    flat = x.to(dev).reshape(-1)[1:]
    assert flat.data_ptr() % 16 != 0 and flat.numel() % 8 != 0
    q, s = to_fp8(flat)
    qo, so = O.to_fp8(bits(x).reshape(-1)[1:])
    assert float(s.item()) == so
    assert (bits(q) == qo).all()


@pytest.mark.parametrize("shape", [(129, 131), (512, 1024)])
def test_quantize_and_compress(dev, shape):
    F, _, TB = _bs()
    x = preact_input(shape, seed=71).relu() * 3
    qo, so = O.to_fp8(bits(x))
    bm, pf, v = O.compress(qo, O.E4M3FN)
    for buf in (None, TB(x.numel(), device=dev, dtype=torch.float8_e4m3fn)):
        q, s, sp = F.quantize_and_compress(x.to(dev), buf)
        assert float(s.item()) == so
        assert (bits(q) == qo).all()
        assert (bits(sp.bitmask) == bm).all() and (bits(sp.prefix) == pf).all()
        assert (bits(sp.vals)[:v.size] == v).all()


def test_tile_pack_and_compact_vals_api(dev):
    """The reference's lower-level names keep their signatures."""
    from bitsparse_amd.src.triton_operators import compact_vals, tile_pack
    x = relu_input((129, 131), 0.5, seed=80)
    xd = x.to(dev)
    T = 3 * 3
    counts = torch.empty(T, dtype=torch.int32, device=dev)
    bmask = torch.empty(T * 512, dtype=torch.uint8, device=dev)
    tile_pack(xd, counts, bmask, 129, 131, 3, 3, 64, 64, 4096, 512)
    bm, cnt = O.tile_pack(bits(x), O.BF16)
    assert (bits(bmask) == bm).all() and (counts.cpu().numpy() == cnt).all()
    pf = torch.zeros(T + 1, dtype=torch.uint32, device=dev)
    torch.cumsum(counts, 0, out=pf.view(torch.int32)[1:])
    vals, off = compact_vals(xd, bmask, pf, None, None, 129, 131, 3, T, 64, 64, 4096, False)
    assert (bits(vals) == O.compress(bits(x), O.BF16)[2]).all() and int(off.item()) == 0


def _all_finite_bf16_upto(amax_bits):
    """Every finite bf16 pattern with magnitude <= the given one, both signs."""
    mags = np.arange(0, amax_bits + 1, dtype=np.uint16)
    return np.concatenate([mags, mags | np.uint16(0x8000)])


_AMAXES = [448.0, 1.0, 3.0e38, 1e-30, 6.5, 0.0173, 1234.5, 2.0 ** -20] + \
    [float(v) for v in np.random.default_rng(5).lognormal(0.0, 6.0, 16)]


@pytest.mark.parametrize("amax", _AMAXES)
def test_to_fp8_all_bf16_patterns(dev, amax):
    """Every finite bf16 input at a given amax (scale = amax / 448) against the
    oracle's division and RNE rounding: pins the reciprocal/FMA quotient and the
    hardware e4m3 conversion of the quantizer."""
    from bitsparse_amd.fp8 import to_fp8
    a_bits = int(np.array([amax], dtype=np.float32).view(np.uint32)[0] >> 16)
    a_bits = min(a_bits, 0x7f7f)
    x_bits = _all_finite_bf16_upto(a_bits)
    x = torch.from_numpy(x_bits.view(np.int16).copy()).view(torch.bfloat16).reshape(-1, 2)
    q, s = to_fp8(x.to(dev))
    qo, so = O.to_fp8(bits(x))
    assert float(s.item()) == so
    assert (bits(q) == qo).all()


@pytest.mark.parametrize("amax", _AMAXES)
def test_quantizing_compress_all_bf16_patterns(dev, amax):
    """quantize_and_compress over every finite bf16 input at a given amax
    (zero padding to whole rows leaves the amax alone): the compress kernel's
    code table, which holds the exponents around the scale's and one code for
    every magnitude below or above them, against the oracle's division and RNE
    rounding, through the dense codes, the bitmask, the prefix and the values."""
    F, _, _ = _bs()
    a_bits = int(np.array([amax], dtype=np.float32).view(np.uint32)[0] >> 16)
    a_bits = min(a_bits, 0x7f7f)
    x_bits = _all_finite_bf16_upto(a_bits)
    cols = 256
    xb = np.zeros(-(-x_bits.size // cols) * cols, np.uint16)
    xb[:x_bits.size] = x_bits
    xb = xb.reshape(-1, cols)
    qo, so = O.to_fp8(xb)
    bm, pf, v = O.compress(qo, O.E4M3FN)
    q, s, sp = F.quantize_and_compress(from_bits(xb, torch.bfloat16).to(dev), None)
    assert float(s.item()) == so
    assert (bits(q) == qo).all()
    assert (bits(sp.bitmask) == bm).all() and (bits(sp.prefix) == pf).all()
    assert (bits(sp.vals)[:v.size] == v).all()


def test_quantizing_compress_nan_input(dev):
    """A NaN input makes the scale NaN and every code NaN: the scale's
    (positive) NaN for a non-NaN x whatever its sign, x's own for a NaN x (a
    quotient with one NaN operand is that NaN), as in the oracle's division."""
    F, _, _ = _bs()
    x = preact_input((129, 131), seed=74)
    xb = bits(x).copy()
    xb[7, 9], xb[30, 40], xb[100, 3] = 0x7fc0, 0xffc0, 0xff80      # +NaN, -NaN, -Inf
    x = from_bits(xb, torch.bfloat16)
    qo, so = O.to_fp8(bits(x))
    bm, pf, v = O.compress(qo, O.E4M3FN)
    q, s, sp = F.quantize_and_compress(x.to(dev), None)
    assert np.isnan(float(s.item())) and np.isnan(so)
    assert (bits(q) == qo).all()
    assert (bits(sp.bitmask) == bm).all() and (bits(sp.prefix) == pf).all()
    assert (bits(sp.vals)[:v.size] == v).all()


def test_to_fp8_and_quantizing_compress_inf_input(dev):
    """An infinite input makes amax and the scale infinite (1/s = 0): finite
    values, +-0 included, quantize to zeros of their sign and the infinities
    to NaN, in to_fp8 and in the fused quantizing compress alike."""
    from bitsparse_amd.fp8 import to_fp8
    from bitsparse_amd.src.functions import quantize_and_compress
    x = special_bf16((129, 131), seed=73)
    xb = bits(x).copy()
    xb[(xb & 0x7fff) > 0x7f80] = 0x3f80          # no NaN: the scale must be +Inf
    xb.reshape(-1)[[5, 77, 900]] = [0x7f80, 0xff80, 0x8000]
    x = from_bits(xb, torch.bfloat16)
    q, s = to_fp8(x.to(dev))
    qo, so = O.to_fp8(xb)
    assert float(s.item()) == float("inf") and so == float("inf")
    assert (bits(q) == qo).all()
    q2, s2, sp = quantize_and_compress(x.to(dev), None)
    assert (bits(q2) == qo).all() and float(s2.item()) == float("inf")
    bm, pf, v = O.compress(qo, O.E4M3FN)
    assert (bits(sp.bitmask) == bm).all() and (bits(sp.prefix) == pf).all()


def test_to_fp8_nan_input(dev):
    from bitsparse_amd.fp8 import to_fp8
    x = preact_input((64, 64), seed=72)
    x[3, 5] = float("nan")
    q, s = to_fp8(x.to(dev))
    qo, so = O.to_fp8(bits(x))
    assert np.isnan(float(s.item())) and np.isnan(so)
    assert (bits(q) == qo).all()
