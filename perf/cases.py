"""The work a user of this framework has it do, as cases whose speed is measured.

Three kinds of case, each through the public entry points that a training
program calls:

* ``codec``: compress one activation (into a preallocated ``TensorBuffer``, or
  standalone into storage of its exact size) and decompress all of it;
* ``dw``: the weight gradient dW = dY^T act(r) of a down-projection with the
  activation r held compressed (``AspB`` / ``AspRelu2B``);
* ``ffn``: forward and backward of a whole MLP block (``FFNRelu`` /
  ``FFNRelu2``) whose activation is saved compressed.

Sizes are those of the repository's benchmark, tests and configurations (the
16384 x 16384 activation, the 8192-token 768 -> 3072 block, the 4096-token
4096 -> 16384 ReLU^2 block with 90% zeros) and generic ones around them.
"""
import math

import torch

from bitsparse_amd.bitsparse import TensorBuffer
from bitsparse_amd.fp8 import to_fp8
from bitsparse_amd.layers import FFNRelu, FFNRelu2
from bitsparse_amd.src.functions import dense_to_tilesparse, quantize_and_compress
from bitsparse_amd.src.hip_operators import unpack_batch_
from bitsparse_amd.src.sparse_matmul import AspB, AspRelu2B

E4M3 = torch.float8_e4m3fn

# pre-activation mean (in standard deviations) for a share of zeros
MU = {0.5: 0.0, 0.75: -0.6745, 0.9: -1.2816, 0.95: -1.6449}


def _codec(name, M, N, zeros, store="bf16", pack=False, buffer=True):
    return {"name": name, "kind": "codec", "M": M, "N": N, "zeros": zeros, "store": store, "pack": pack,
            "buffer": buffer}


def _ffn(name, T, D, H, act, zeros, store="bf16", pack=False, bias=False):
    return {"name": name, "kind": "ffn", "T": T, "D": D, "H": H, "act": act, "zeros": zeros, "store": store,
            "pack": pack, "bias": bias}


def _dw(name, T, D, H, act, zeros, store="bf16", pack=False):
    return {"name": name, "kind": "dw", "T": T, "D": D, "H": H, "act": act, "zeros": zeros, "store": store,
            "pack": pack}


def listed():
    return [
        # a unit test's or a toy model's activation: launches and host latency only
        _codec("codec_tiny_bf16", 256, 512, 0.5),
        # one layer's activation of an 8192-token batch of a 768 -> 3072 block
        _codec("codec_block_bf16", 8192, 3072, 0.5),
        # the benchmark's headline activation: the largest, streamed from memory
        _codec("codec_large_bf16", 16384, 16384, 0.5),
        # the activation of a sparse 4096 -> 16384 ReLU^2 block in fp8 storage, with the
        # dense codes the next GEMM takes
        _codec("codec_sparse_e4m3", 4096, 16384, 0.9, store="e4m3"),
        # the 15-bit stream, a shape that ends inside a tile in both directions
        _codec("codec_packed_bf16", 5053, 6152, 0.75, pack=True),
        # no buffer (exact-size storage), odd sizes: rows that no vector load is aligned to
        _codec("codec_alone_odd_bf16", 1999, 3001, 0.5, buffer=False),
        # a small model's training step: many small launches
        _ffn("ffn_relu_tiny_bf16", 128, 256, 1024, "relu", 0.5),
        # the 768 -> 3072 -> 768 block on 8192 tokens, the benchmark's bf16 training step
        _ffn("ffn_relu_block_bf16", 8192, 768, 3072, "relu", 0.5),
        # biases, packed storage and a ragged number of tokens
        _ffn("ffn_relu2_packed_bf16", 3005, 1024, 4096, "relu2", 0.75, pack=True, bias=True),
        # the large sparse ReLU^2 block, fp8 storage and fp8 GEMMs: the benchmark's fp8 training step
        _ffn("ffn_relu2_large_e4m3", 4096, 4096, 16384, "relu2", 0.9, store="e4m3", bias=True),
        # the weight gradient alone, bf16 storage, the large block's size
        _dw("dw_relu_large_bf16", 4096, 4096, 16384, "relu", 0.5),
        # the weight gradient alone, fp8 storage, ReLU^2
        _dw("dw_relu2_large_e4m3", 4096, 4096, 16384, "relu2", 0.9, store="e4m3"),
    ]


MAX_GEMM = 4096 * 4096 * 16384          # T * D * H of a drawn dw or ffn case


def _log(rng, lo, hi, step=1):
    """An integer of [lo, hi], its logarithm spread evenly, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, int(round(v / step)) * step)


def _rows(rng, lo, hi, whole):
    """A number of rows of whole tiles of 64, or (not `whole`) up to 7 short of
    it.  A last tile row with fewer rows is left out where the columns are a
    multiple of 8: the compress kernel that these cases were first measured
    on reads past the end of such an input, so the two could not be compared."""
    full = -(-_log(rng, lo, hi) // 64) * 64
    return full if whole or rng.random() < 0.4 else full - rng.randint(1, 7)


def draw(rng):
    kind = rng.choice(["codec", "codec", "ffn", "ffn", "dw"])
    store = rng.choice(["bf16", "bf16", "e4m3"])
    pack = rng.random() < 0.25
    zeros = rng.choice(sorted(MU))
    if kind == "codec":
        N = _log(rng, 64, 16384, rng.choice([1, 8, 64]))
        M = _log(rng, 64, 16384) if N % 8 else _rows(rng, 64, 16384, False)
        c = _codec("", M, N, zeros, store, pack, rng.random() < 0.8)
    else:
        while True:
            # hipBLASLt's fp8 products take multiples of 16 in every dimension
            T = _rows(rng, 64, 16384, store == "e4m3")
            D, H = _log(rng, 128, 4096, 16), _log(rng, 512, 16384, 16)
            if T * D * H <= MAX_GEMM:
                break
        act = rng.choice(["relu", "relu2"])
        if kind == "ffn":
            c = _ffn("", T, D, H, act, zeros, store, pack, rng.random() < 0.5)
        else:
            c = _dw("", T, D, H, act, zeros, store, pack)
    del c["name"]
    return c


def _randn(g, *shape, mul=1.0, add=0.0):
    return (torch.randn(shape, generator=g, device="cuda") * mul + add).to(torch.bfloat16)


def _activation(g, M, N, zeros):
    """relu of a bf16 N(mu, 1) pre-activation"""
    return _randn(g, M, N, add=MU[zeros]).relu_()


def _buffer(M, N, store, pack, count=None):
    """The TensorBuffer of one activation: `count` values, or room for a dense one."""
    count = M * N if count is None else count
    dtype = E4M3 if store == "e4m3" else torch.bfloat16
    size = (count * (7 if store == "e4m3" else 15) + 7) // 8 if pack else count * (1 if store == "e4m3" else 2)
    return TensorBuffer(size, device="cuda", dtype=dtype, pack_sbit=pack)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    st = {"case": case}
    if case["kind"] == "codec":
        M, N = case["M"], case["N"]
        st["x"] = _activation(g, M, N, case["zeros"])
        if case["buffer"]:
            # a program sizes its buffer for the values it expects, with some slack
            count = min(M * N, int(M * N * (1 - case["zeros"]) * 1.1) + 1024)
            st["buf"] = _buffer(M, N, case["store"], case["pack"], count)
        else:
            st["buf"] = None
        return st
    st["buf"] = _buffer(case["T"], case["H"], case["store"], case["pack"])
    if case["kind"] == "dw":
        dY, r = _dw_inputs(case, g)
        if case["store"] == "e4m3":
            st["dY"], st["scale"] = to_fp8(dY)
            st["sp"] = quantize_and_compress(r, st["buf"], case["pack"], dense_out=False)[2]
        else:
            st["dY"], st["scale"] = dY, None
            st["sp"] = dense_to_tilesparse(r, None, st["buf"], case["pack"])
        return st
    st.update(_ffn_inputs(case, g))
    return st


def _dw_inputs(case, g):
    return _randn(g, case["T"], case["D"]), _activation(g, case["T"], case["H"], case["zeros"])


def _ffn_inputs(case, g):
    T, D, H = case["T"], case["D"], case["H"]
    std, st = 0.02, {}
    st["x"] = _randn(g, T, D).requires_grad_()
    st["W1"] = _randn(g, H, D, mul=std).requires_grad_()
    st["W2"] = _randn(g, D, H, mul=std).requires_grad_()
    st["dY"] = _randn(g, T, D)
    st["b1"] = st["b2"] = None
    if case["bias"] or case["zeros"] != 0.5:
        # the first bias shifts the pre-activation to the case's share of zeros
        shift = MU[case["zeros"]] * std * math.sqrt(D)
        st["b1"] = _randn(g, H, mul=0.02, add=shift).requires_grad_()
    if case["bias"]:
        st["b2"] = _randn(g, D, mul=0.02).requires_grad_()
    return st


def _bits(t):
    """Stored values as whole numbers (they are moved, not computed)."""
    return t.view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[t.element_size()])


def _run_codec(st):
    c, x, buf = st["case"], st["x"], st["buf"]
    M, N = x.shape
    if buf is not None:
        buf.reset_buffer()
    out = {}
    if c["store"] == "e4m3":
        q, scale, sp = quantize_and_compress(x, buf, c["pack"])
        out["codes"], out["scale"] = _bits(q), scale
    else:
        sp = dense_to_tilesparse(x, None, buf, c["pack"])
    dense = torch.empty((M, N), device=x.device, dtype=sp.dtype)
    unpack_batch_(sp, dense, 0, sp.grid_n, N, M, sp.num_tiles)
    out.update(bitmask=sp.bitmask, prefix=_bits(sp.prefix), dense=dense)
    if buf is not None:      # standalone storage has as many values as the input: dense holds them
        out["vals"] = _bits(sp.vals)
    return out


def _run_ffn(st):
    c = st["case"]
    params = {k: st[k] for k in ("x", "W1", "W2", "b1", "b2") if st[k] is not None}
    for p in params.values():
        p.grad = None
    st["buf"].reset_buffer()
    dtype = E4M3 if c["store"] == "e4m3" else torch.bfloat16
    if c["act"] == "relu":
        y = FFNRelu.apply(st["x"], st["W1"], st["W2"], st["b1"], st["b2"], sparse_data=st["buf"],
                          pack_sbit=c["pack"], dtype=dtype)
    else:
        y = FFNRelu2.apply(st["x"], st["W1"], st["W2"], st["b1"], st["b2"], sparse_data=st["buf"],
                           pack_sbit=c["pack"], storage_dtype=dtype)
    y.backward(st["dY"])
    return {"y": y.detach(), **{"d" + k: p.grad for k, p in params.items()}}


def run(state):
    kind = state["case"]["kind"]
    if kind == "codec":
        return _run_codec(state)
    if kind == "ffn":
        return _run_ffn(state)
    product = AspB if state["case"]["act"] == "relu" else AspRelu2B
    return {"dW2": product(state["dY"].T, state["sp"], A_scale=state["scale"])}


def work(case):
    z = case["zeros"]
    vb = 1 if case["store"] == "e4m3" else 2
    bits = (7 if vb == 1 else 15) if case["pack"] else 8 * vb
    if case["kind"] == "codec":
        n = case["M"] * case["N"]
        stored = n * (1 - z) * bits / 8 + n / 8       # values and bitmask
        # compress: read dense, write the compressed form (fp8: the dense codes
        # too); decompress: read it, write dense
        return {"bytes": 2 * n + (n if vb == 1 else 0) + 2 * stored + vb * n, "flops": 0}
    T, D, H = case["T"], case["D"], case["H"]
    stored = T * H * (1 - z) * bits / 8 + T * H / 8
    if case["kind"] == "dw":
        return {"bytes": vb * T * D + stored + 2 * D * H, "flops": 2 * T * D * H}
    # x, dY, W1, W2 read; y, dx, dW1, dW2 written; the activation stored and read back
    return {"bytes": 2 * (4 * T * D + 4 * D * H) + 2 * stored, "flops": 12 * T * D * H}


def tolerance(case):
    if case["kind"] == "codec":
        return "exact"
    # Sums in fp32, results rounded to bf16: 0.0017 from `exact` at every size.
    # The fp8 block's gradients come back in e4m3fn and a step of z's rounding
    # may move a code: 0.005-0.007 from `exact`.  About four times either.
    return {"rel": 0.02 if case["store"] == "e4m3" and case["kind"] == "ffn" else 0.007}


# ---------------------------------------------------------------------------
# the same results in plain torch, sums in 64 bits, rounded to the formats
# that the path itself stores its intermediates in
# ---------------------------------------------------------------------------
def _bf(x):
    return x.to(torch.bfloat16).double()


def _q8(x):
    """(x as its nearest e4m3fn multiples of max|x| / 448, that scale)"""
    s = (x.abs().amax() / 448.0).clamp(min=1e-9).float()
    return (x.float() / s).to(E4M3).double() * s.double(), s


def _e4m3_grad(x):
    """bf16 gradient that went through e4m3fn, saturating"""
    return x.clamp(-448.0, 448.0).float().to(E4M3).double()


def _square8(r8, s):
    """the ReLU^2 operand rebuilt from fp8 storage, re-quantized"""
    v = (r8 / s.double())
    return _q8(_bf(_bf(v * v) * _bf(s.double() * s.double())))[0]


def _exact_ffn(case, st):
    e4m3, sq = case["store"] == "e4m3", case["act"] == "relu2"
    x, W1, W2, dY = (st[k].detach().double() for k in ("x", "W1", "W2", "dY"))
    out = {}
    q = (lambda t: _q8(t)[0]) if e4m3 else (lambda t: t)
    xq, W1q, W2q, gq = q(x), q(W1), q(W2), q(dY)
    z = _bf(xq @ W1q.T)
    if st["b1"] is not None:
        z = _bf(z + st["b1"].detach().double())
    r = z.clamp(min=0)
    h = _bf(r * r) if sq else r
    y = _bf(q(h) @ W2q.T)
    if st["b2"] is not None:
        y = _bf(y + st["b2"].detach().double())
        out["db2"] = dY.sum(0)
    dh = _bf(gq @ W2q)
    if e4m3:
        r8, s = _q8(r)
        kept = r8 > 0
        out["dW2"] = gq.T @ (_square8(r8, s) if sq else r8)
        dz = _bf(_bf(dh * 2 * (r8 / s.double())) * _bf(s.double())) * kept if sq else dh * kept
        dzq = _q8(dz)[0]
        out["dx"], out["dW1"] = _e4m3_grad(dzq @ W1q), _e4m3_grad(dzq.T @ xq)
    else:
        out["dW2"] = dY.T @ h
        dz = _bf(dh * 2 * r) if sq else dh * (r > 0)
        out["dx"], out["dW1"] = dz @ W1, dz.T @ x
    out["y"] = y
    if st["b1"] is not None:
        out["db1"] = dz.sum(0)
    return out


def exact(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "codec":
        x = _activation(g, case["M"], case["N"], case["zeros"])
        if case["store"] == "e4m3":
            # the decompressed codes are the quantized values over their scale
            v, s = _q8(x.double())
            return {"scale": s.double(), "dense": v / s.double()}
        return {"dense": x.double()}
    if case["kind"] == "dw":
        dY, r = (t.double() for t in _dw_inputs(case, g))
        sq = case["act"] == "relu2"
        if case["store"] == "e4m3":
            r8, s = _q8(r)
            return {"dW2": _q8(dY)[0].T @ (_square8(r8, s) if sq else r8)}
        return {"dW2": dY.T @ (_bf(r * r) if sq else r)}
    return _exact_ffn(case, _ffn_inputs(case, g))
