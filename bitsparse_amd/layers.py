"""Autograd MLP layers whose ReLU / ReLU^2 activation is saved compressed.

Mirrors reference lib_sparse/layers.py: ``ReluLinear`` (:20-66), ``FFNRelu``
(:69-94), ``Relu2Linear`` (:100-151), ``FFNRelu2`` (:154-177) — same
signatures, including the reference's ``dtype`` (FFNRelu) vs
``storage_dtype`` (FFNRelu2) keyword names.  Forward: GEMM -> ReLU (in
place) -> [fp8 quantize] -> compress (HIP) -> GEMM.  Backward: dW from the
compressed activation (reconstruct-into-LDS GEMM for bf16), dZ from the
bitmask (HIP mask / ReLU^2-gradient kernels).
"""
from __future__ import annotations

import math

import torch
from torch import Tensor
from torch.autograd import Function, forward_ad

from . import config
from .bitsparse import BitsparseTensor, TensorBuffer, plain_cursor
from .config import BLOCK_M, BLOCK_N, RELU2_SCALE
from .fp8 import is_fp8, matmul, to_fp8
from ._lib import native
from .src import sparse_matmul
from .src.functions import (fused_linear_relu_ok, linear_relu_and_compress, relu2_and_compress,
                            relu2_fused_ok, relu2_quantize_and_compress, relu_and_compress,
                            relu_quantize_and_compress)
from .src.hip_operators import mask_with_bitmask_, quantize_e4m3fn, relu2_grad_sparse_, relu2_square_amax_
from .src.sparse_matmul import AspB, AspRelu2B

# FFNRelu / FFNRelu2 with bf16 storage into a TensorBuffer run the up-projection
# GEMM, ReLU and compress as one kernel (bs_linear_relu_compress) when the
# operands qualify; False keeps the library GEMM + bias add + compress path.
USE_FUSED_UP = False


# ------------------------------------------------------------
# ReLU layers
# ------------------------------------------------------------
class ReluLinear(Function):
    """y = relu(z) @ W.T with relu(z) saved compressed."""

    @staticmethod
    def forward(ctx, z, W, sparse_data: TensorBuffer | None = None, pack_sbit: bool = False,
                dtype: torch.dtype = torch.bfloat16):
        ctx.dtype = dtype
        ctx.save_for_backward(W)
        y, ctx.h_sparse = ReluLinear.activate_and_project(z, W, sparse_data, pack_sbit, dtype)
        return y

    @staticmethod
    def activate_and_project(z, W, sparse_data, pack_sbit, dtype) -> tuple[Tensor, BitsparseTensor]:
        # h = z.relu_() fused into the compress pass (z is still updated in place)
        if is_fp8(dtype):
            # any fp8 dtype stores e4m3fn codes + scale: the reference quantizes
            # with to_fp8, whose output is e4m3fn for e5m2 too (fp8.py:123-129)
            h, scale, h_sparse = relu_quantize_and_compress(z, sparse_data, pack_sbit)
        else:
            scale = None
            h, h_sparse = relu_and_compress(z, sparse_data, pack_sbit)
        return matmul(h, W.T, is_fp8(dtype), a_scale=scale), h_sparse

    @staticmethod
    @torch.compiler.disable
    def backward(ctx, grad_output: Tensor):
        W = ctx.saved_tensors[0]
        needs_z = ctx.needs_input_grad[0]
        h: BitsparseTensor = ctx.h_sparse
        ctx.h_sparse = None

        fp8 = is_fp8(ctx.dtype)
        if fp8:
            grad_output, scale = to_fp8(grad_output)
        else:
            grad_output, scale = grad_output, None

        grad_W2 = AspB(grad_output.T, h, A_scale=scale)

        if needs_z:
            grad_h = matmul(grad_output, W, fp8=fp8, a_scale=scale)
            grad_z = mask_with_bitmask_(grad_h, h)
        else:
            grad_z = None
        return grad_z, grad_W2, None, None, None


class FFNRelu:
    """FFN block with ReLU activation: y = relu(x @ W1.T + b1) @ W2.T + b2."""

    @staticmethod
    def apply(x, W1, W2, b1=None, b2=None, *,
              sparse_data: TensorBuffer | None = None, pack_sbit: bool = False,
              dtype: torch.dtype = torch.bfloat16):
        """x [*bs, d_in], W1 [d_ff, d_in], W2 [d_out, d_ff], b1 [d_ff], b2 [d_out]
        -> [*bs, d_out]."""
        bs_dims = x.shape[:-1]
        x = x.reshape(-1, x.shape[-1])

        if _block_ok(x, W1, W2, b1, b2, sparse_data, pack_sbit, dtype):
            return _block(x, W1, b1, W2, b2, bs_dims, sparse_data, is_fp8(dtype), False)
        if not is_fp8(dtype) and not pack_sbit and USE_FUSED_UP and fused_linear_relu_ok(x, W1, b1, sparse_data):
            y = _UpReluLinear.apply(x, W1, b1, W2, sparse_data, False)
        else:
            z = matmul(x, W1.T, is_fp8(dtype))
            if b1 is not None:
                z = z + b1
            y = ReluLinear.apply(z, W2, sparse_data, pack_sbit, dtype)

        y = y.reshape(*bs_dims, y.shape[-1])
        if b2 is not None:
            y = y + b2
        return y


# ------------------------------------------------------------
# ReLU^2 layers
# ------------------------------------------------------------
class Relu2Linear(Function):
    """y = (k * relu(z)^2) @ W.T with r = relu(z) saved compressed."""

    @staticmethod
    def forward(ctx, z, W, sparse_data: TensorBuffer | None, pack_sbit: bool = False,
                storage_dtype: torch.dtype = torch.bfloat16):
        ctx.dtype = storage_dtype
        ctx.save_for_backward(W)
        y, ctx.h_sparse = Relu2Linear.activate_and_project(z, W, sparse_data, pack_sbit, storage_dtype)
        return y

    @staticmethod
    def activate_and_project(z, W, sparse_data, pack_sbit, storage_dtype) -> tuple[Tensor, BitsparseTensor]:
        # h = z.relu_() fused into the compress pass (z is still updated in place)
        fused_sq = relu2_fused_ok(z, sparse_data, pack_sbit, RELU2_SCALE)
        if is_fp8(storage_dtype):
            # e4m3fn codes for every fp8 storage dtype, as to_fp8 makes them;
            # the forward multiplies the bf16 square, so no dense e4m3fn copy
            if fused_sq:
                # the compress also writes h = k r^2 into z; amax|h| follows
                # from the amax of r
                _, h_sparse, epoch = relu2_quantize_and_compress(z, sparse_data, RELU2_SCALE)
            else:
                _, _, h_sparse = relu_quantize_and_compress(z, sparse_data, pack_sbit, dense_out=False)
                # h.square_(); h.mul_(k) and the amax of to_fp8(h) in one pass
                epoch = relu2_square_amax_(z, RELU2_SCALE)
            # h ends up in z, as the reference's in-place ops leave it
            h8, h_scale = quantize_e4m3fn(z, epoch)
            return matmul(h8, W.T, True, a_scale=h_scale), h_sparse
        if fused_sq:
            h_sparse = relu2_and_compress(z, sparse_data, RELU2_SCALE)
            h = z
        else:
            h, h_sparse = relu_and_compress(z, sparse_data, pack_sbit)
            if h.is_contiguous():
                # h.square_(); h.mul_(k) in one pass, bit for bit (its amax goes unused)
                relu2_square_amax_(h, RELU2_SCALE)
            else:
                h.square_()
                h.mul_(RELU2_SCALE)
        return matmul(h, W.T, False), h_sparse

    @staticmethod
    @torch.compiler.disable
    def backward(ctx, grad_output: Tensor):
        W = ctx.saved_tensors[0]
        needs_z = ctx.needs_input_grad[0]
        h: BitsparseTensor = ctx.h_sparse
        ctx.h_sparse = None

        fp8 = is_fp8(ctx.dtype)
        if fp8:
            grad_output, scale = to_fp8(grad_output)
        else:
            grad_output, scale = grad_output, None

        grad_W2 = AspRelu2B(grad_output.T, h, A_scale=scale)

        if needs_z:
            grad_h = matmul(grad_output, W, fp8=fp8, a_scale=scale)
            grad_z = relu2_grad_sparse_(grad_h, h)
        else:
            grad_z = None
        return grad_z, grad_W2, None, None, None


class FFNRelu2:
    """FFN block with ReLU^2 activation: y = k*relu(x @ W1.T + b1)^2 @ W2.T + b2."""

    @staticmethod
    def apply(x, W1, W2, b1=None, b2=None, *,
              sparse_data: TensorBuffer | None = None, pack_sbit: bool = False,
              storage_dtype: torch.dtype = torch.bfloat16):
        bs_dims = x.shape[:-1]
        x = x.reshape(-1, x.shape[-1])
        if _block_ok(x, W1, W2, b1, b2, sparse_data, pack_sbit, storage_dtype):
            return _block(x, W1, b1, W2, b2, bs_dims, sparse_data, is_fp8(storage_dtype), True)
        if (not is_fp8(storage_dtype) and not pack_sbit and USE_FUSED_UP
                and fused_linear_relu_ok(x, W1, b1, sparse_data)):
            y = _UpReluLinear.apply(x, W1, b1, W2, sparse_data, True)
        else:
            z = matmul(x, W1.T, is_fp8(storage_dtype))
            if b1 is not None:
                z = z + b1
            y = Relu2Linear.apply(z, W2, sparse_data, pack_sbit, storage_dtype)
        y = y.reshape(*bs_dims, y.shape[-1])
        if b2 is not None:
            y = y + b2
        return y


# ------------------------------------------------------------
# the whole block as one autograd node (its body: csrc/native.cpp)
# ------------------------------------------------------------
def _plain(t: Tensor) -> bool:
    return type(t) in (Tensor, torch.nn.Parameter) and t.is_cuda and t.dtype == torch.bfloat16


def _block_ok(x: Tensor, W1: Tensor, W2: Tensor, b1: Tensor | None, b2: Tensor | None,
              sparse_data: TensorBuffer | None, pack_sbit: bool, dtype: torch.dtype) -> bool:
    """The MLP block runs as one node (``_FFNBlock``): plain bf16 matrices and bias
    rows on one GPU in the shapes and alignments its kernels take, a
    TensorBuffer of the stored type, outside autocast, tracing, forward-mode
    AD and the options that choose another path.  Everything else takes the
    layers' separate nodes, with their errors."""
    # first: neither tracers nor function transforms follow the addresses below
    if torch.compiler.is_compiling() or torch._C._are_functorch_transforms_active():
        return False
    if sparse_data is None or not (_plain(x) and _plain(W1) and _plain(W2) and plain_cursor(sparse_data)):
        return False
    if USE_FUSED_UP or config.CACHE_FP8_MATMUl or not sparse_matmul.USE_LDS_GEMM or not math.isfinite(RELU2_SCALE):
        return False
    if x.dim() != 2 or W1.dim() != 2 or W2.dim() != 2 or not (W1.is_contiguous() and W2.is_contiguous()):
        return False
    T, D = x.shape
    H, O = W1.shape[0], W2.shape[0]
    if W1.shape[1] != D or W2.shape[1] != H or 0 in (T, D, H, O) or H % 8 or T * H >= 2 ** 31:
        return False
    fp8 = is_fp8(dtype)
    if fp8 and (T % 16 or D % 16 or H % 16 or O % 16 or T * D >= 2 ** 31 or D * H >= 2 ** 31 or H * O >= 2 ** 31
                or any(t.data_ptr() % 16 for t in (x, W1, W2))):
        return False
    for b, n in ((b1, H), (b2, O)):
        if b is not None and not (_plain(b) and b.shape == (n,) and b.is_contiguous() and b.data_ptr() % 16 == 0):
            return False
    buf = sparse_data.vals
    stored = torch.float8_e4m3fn if fp8 else torch.bfloat16
    if (bool(sparse_data.pack_sbit) != bool(pack_sbit) or sparse_data.dtype != stored
            or (not pack_sbit and buf.dtype != stored) or buf.data_ptr() % (4 if pack_sbit else 16)):
        return False
    if not (x.device == W1.device == W2.device == buf.device) or any(
            b is not None and b.device != x.device for b in (b1, b2)):
        return False
    return not torch.is_autocast_enabled("cuda") and forward_ad._current_level < 0


def _block(x, W1, b1, W2, b2, bs_dims, sparse_data: TensorBuffer, fp8: bool, square: bool) -> Tensor:
    """The block's y in the shape of its input.  The node adds b2; b2's
    gradient, which needs nothing of the node, has one of its own."""
    y = _FFNBlock.apply(x, W1, b1, W2, (b2,), sparse_data, fp8, square)     # (in a tuple: no edge to b2)
    if b2 is None:
        return y.reshape(*bs_dims, y.shape[-1])
    return native().biased(y, b2, (*bs_dims, y.shape[-1]))


class _FFNBlock(Function):
    """y = act(x @ W1.T + b1) @ W2.T + b2 with act(z) = relu(z) or
    k * relu(z)^2 saved compressed, for operands ``_block_ok`` accepts."""

    @staticmethod
    def forward(ctx, x, W1, b1, W2, b2, buf, fp8, square):
        offset, in_place = buf.native_cursor()
        y, bitmask, prefix, start, buf._offset, scale = native().block_forward(
            x, W1, b1, W2, b2[0], buf.vals, offset, buf.err_flags, in_place, buf.pack_sbit, fp8, square,
            float(RELU2_SCALE))
        M, N = x.shape[0], W1.shape[0]
        ctx.h_sparse = BitsparseTensor(buf.vals, bitmask, prefix, (M, N), torch.float8_e4m3fn if fp8 else torch.bfloat16,
                                       (M + BLOCK_M - 1) // BLOCK_M, (N + BLOCK_N - 1) // BLOCK_N, BLOCK_M, BLOCK_N,
                                       scale=scale, vals_offset=start, pack_sbit=buf.pack_sbit)
        ctx.fp8, ctx.square = fp8, square
        ctx.save_for_backward(x, W1, W2)
        return y

    @staticmethod
    @torch.compiler.disable
    def backward(ctx, grad_output: Tensor):
        x, W1, W2 = ctx.saved_tensors
        h: BitsparseTensor = ctx.h_sparse
        ctx.h_sparse = None
        held, shape, packed = [h.vals, h.bitmask, h.prefix, h.vals_offset, h.scale], h.shape, h.pack_sbit
        del h
        dh = None
        # create_graph: the fp8 product has its graph from MatmulFp8
        if ctx.fp8 and torch.is_grad_enabled() and any(ctx.needs_input_grad[:3]):
            g8, scale = to_fp8(grad_output)
            dh = matmul(g8, W2, True, a_scale=scale)
        grads = native().block_backward(
            grad_output, x, W1, W2, held, *shape, packed, ctx.fp8, ctx.square, float(RELU2_SCALE), config.FP8_GRAD_DTYPE,
            ctx.needs_input_grad[:4], dh)
        return *grads, None, None, None, None


# ------------------------------------------------------------
# fused up-projection (bf16 storage into a TensorBuffer)
# ------------------------------------------------------------
class _UpReluLinear(Function):
    """The autograd node of ``z = x @ W1.T + b1`` followed by ReluLinear
    (square=False) or Relu2Linear (square=True), with z, relu(z) and its
    compressed form produced by one kernel.  Backward repeats the calls of the
    two-node graph: the same dz from the bitmask (or the ReLU^2 gradient), then
    autograd's own products for x, W1 and b1."""

    @staticmethod
    def forward(ctx, x, W1, b1, W2, sparse_data: TensorBuffer, square: bool):
        h, h_sparse = linear_relu_and_compress(x, W1, b1, sparse_data)
        ctx.h_sparse = h_sparse
        ctx.square = square
        ctx.has_b1 = b1 is not None
        ctx.save_for_backward(x, W1, W2)
        if square:
            h.square_()
            h.mul_(RELU2_SCALE)
        return matmul(h, W2.T, False)

    @staticmethod
    @torch.compiler.disable
    def backward(ctx, grad_output: Tensor):
        x, W1, W2 = ctx.saved_tensors
        h: BitsparseTensor = ctx.h_sparse
        ctx.h_sparse = None
        if ctx.square:
            grad_W2 = AspRelu2B(grad_output.T, h)
        else:
            grad_W2 = AspB(grad_output.T, h)
        grad_x = grad_W1 = grad_b1 = None
        if any(ctx.needs_input_grad[:3]):
            grad_h = matmul(grad_output, W2, fp8=False)
            grad_z = relu2_grad_sparse_(grad_h, h) if ctx.square else mask_with_bitmask_(grad_h, h)
            # the products autograd forms for z = x @ W1.T + b1
            if ctx.needs_input_grad[0]:
                grad_x = grad_z.mm(W1)
            if ctx.needs_input_grad[1]:
                grad_W1 = grad_z.t().mm(x)          # W1's own layout, as autograd forms it for x @ W1.T
            if ctx.has_b1 and ctx.needs_input_grad[2]:
                grad_b1 = grad_z.sum(0)
        # the forward kernel's look-back must not have given up: checked once
        # this node's kernels are queued (the check waits for that forward
        # kernel, so checking first would leave the GPU idle while the host
        # queues them); gradients from a misplaced value run are never returned
        h.lookback_check.raise_if_timed_out()
        return grad_x, grad_W1, grad_b1, grad_W2, None, None
