"""ctypes binding of libbitsparse_hip.so (the C ABI in include/bitsparse_hip.h).

The shared library is built in-tree next to this file by
``bitsparse_amd.build.build_library()`` (or ``__graft_entry__.build()``).
There is no fallback: if the library is missing or a call fails, an
exception is raised.
"""
from __future__ import annotations

import ctypes
import os
import threading

import torch

LIB_NAME = "libbitsparse_hip.so"
# BITSPARSE_HIP_LIB points at another build of the same sources (tuning sweeps)
LIB_PATH = os.environ.get("BITSPARSE_HIP_LIB") or os.path.join(
    os.path.dirname(os.path.abspath(__file__)), LIB_NAME)
ABI_VERSION = 17

BS_OK = 0
BS_ERR_INVALID = 1
BS_ERR_HIP = 2

# dtype codes == reference codec ids (lib_sparse/bitsparse.py:8-18)
DT_BF16, DT_E4M3FN, DT_E5M2 = 0, 1, 2

_i64 = ctypes.c_int64
_u32 = ctypes.c_uint32
_int = ctypes.c_int
_vp = ctypes.c_void_p
_f32 = ctypes.c_float

# name -> argtypes (restype int unless listed in _RESTYPES)
_SIGNATURES = {
    "bs_last_error": [],
    "bs_abi_version": [],
    "bs_compress_workspace_bytes": [_i64, _i64],
    "bs_compress": [_vp, _int, _i64, _i64, _int, _vp, _u32, _vp, _vp, _vp, _vp, _vp, _i64, _vp,
                    _int, _vp, _vp, _int, _vp, _vp, _i64, _u32, _vp],
    "bs_compress_relu": [_vp, _int, _i64, _i64, _int, _vp, _u32, _vp, _vp, _vp, _vp, _vp, _i64, _vp,
                         _int, _vp, _vp, _int, _vp, _vp, _i64, _u32, _vp, _vp],
    "bs_linear_relu_compress": [_vp, _i64, _i64, _i64, _vp, _i64, _i64, _vp, _vp, _i64, _vp, _vp, _vp, _i64,
                                _vp, _int, _vp, _vp, _vp, _vp, _i64, _vp, _i64, _u32, _vp],
    "bs_linear_relu_compress_max_n": [_int],
    "bs_host_device_pointer": [_vp, _vp],
    "bs_compress_packed": [_vp, _int, _i64, _i64, _int, _vp, _u32, _vp, _vp, _vp, _vp, _vp, _i64, _vp,
                           _vp, _vp, _vp, _vp, _i64, _u32, _int, _vp, _vp],
    "bs_amax_relu": [_vp, _i64, _vp, _i64, _u32, _vp],
    "bs_tile_pack": [_vp, _int, _i64, _i64, _vp, _vp, _vp],
    "bs_prefix_from_counts": [_vp, _i64, _vp, _vp],
    "bs_compact_vals": [_vp, _int, _i64, _i64, _vp, _vp, _vp, _i64, _vp, _i64, _i64, _vp, _vp],
    "bs_decompress": [_vp, _int, _i64, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _int, _f32,
                      _vp, _vp],
    "bs_relu_grad": [_vp, _i64, _i64, _vp, _vp],
    "bs_relu2_grad": [_vp, _i64, _i64, _vp, _int, _i64, _vp, _vp, _vp, _f32, _vp, _vp],
    "bs_amax": [_vp, _i64, _vp, _i64, _u32, _vp],
    "bs_quantize_e4m3fn": [_vp, _i64, _vp, _vp, _vp, _i64, _u32, _vp],
    "bs_quantize_e4m3fn_t": [_vp, _i64, _i64, _vp, _vp, _vp, _vp, _i64, _u32, _vp],
    "bs_transpose_u8": [_vp, _i64, _i64, _i64, _vp, _i64, _vp],
    "bs_widen_e4m3fn": [_vp, _i64, _vp, _vp],
    "bs_relu2_square_amax": [_vp, _i64, ctypes.c_float, _vp, _i64, _u32, _vp],
    "bs_compress_relu2": [_vp, _int, _i64, _i64, _vp, _u32, _vp, _vp, _vp, _vp, _vp, _i64, _vp, _vp, _vp,
                          _vp, _i64, _u32, _vp, ctypes.c_float, _vp],
    "bs_amax_relu2_from": [_vp, _i64, _u32, _u32, ctypes.c_float, _vp],
    "bs_gemm_compressed_b_workspace_bytes": [_i64, _i64, _i64, _int],
    "bs_gemm_compressed_b": [_vp, _i64, _i64, _i64, _int, _vp, _int, _i64, _vp, _vp, _vp, _i64, _int, _f32,
                             _vp, _vp, _vp, _i64, _vp],
    "bs_gemm_compressed_b_fp8_workspace_bytes": [_i64, _i64, _i64, _int, _int],
    "bs_gemm_compressed_b_fp8": [_vp, _vp, _i64, _i64, _i64, _int, _vp, _int, _i64, _vp, _vp, _vp, _i64, _int,
                                 _f32, _vp, _vp, _vp, _vp, _i64, _vp],
    "bs_gemm_compressed_b_packed_workspace_bytes": [_i64, _i64, _i64, _int],
    "bs_gemm_compressed_b_packed": [_vp, _i64, _i64, _i64, _int, _vp, _int, _i64, _vp, _vp, _vp, _i64, _int,
                                    _f32, _vp, _vp, _vp, _i64, _vp],
    "bs_gemm_compressed_b_fp8_packed": [_vp, _vp, _i64, _i64, _i64, _int, _vp, _int, _i64, _vp, _vp, _vp, _i64,
                                        _int, _f32, _vp, _vp, _vp, _vp, _i64, _vp],
    "bs_pack_bits": [_vp, _int, _vp, _i64, _vp, _i64, _vp, _vp, _vp],
    "bs_decompress_packed": [_vp, _int, _i64, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _int,
                             _f32, _vp, _vp],
    "bs_relu2_grad_packed": [_vp, _i64, _i64, _vp, _int, _i64, _vp, _vp, _vp, _f32, _vp, _vp],
    "bs_workspace_amax_slot": [_vp, _i64],
    "bs_workspace_fallback_counter": [_vp, _i64],
    "bs_compress_noalloc": [_vp, _int, _i64, _i64, _int, _int, _vp, _vp, _vp, _vp, _vp, _i64, _vp, _int,
                            _vp, _vp, _int, _vp, _vp, _vp],
    "bs_compress_noalloc_max_tiles": [],
    "bs_compress_act": [_vp, _vp, _i64, _i64, _int, _f32, _int, _vp, _u32, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64,
                        _int, _vp, _vp, _vp, _vp, _vp, _i64, _u32, _vp],
    "bs_amax_bias_relu": [_vp, _i64, _i64, _vp, _vp, _i64, _u32, _vp],
    "bs_grad_sums_workspace_bytes": [_i64, _i64],
    "bs_act_grad_sums": [_vp, _i64, _i64, _int, _vp, _int, _i64, _int, _vp, _vp, _vp, _f32, _vp, _vp, _vp, _u32, _vp,
                         _i64, _vp],
    "bs_col_sum_workspace_bytes": [_i64, _i64],
    "bs_col_sum": [_vp, _i64, _i64, _vp, _vp, _i64, _vp],
    "bs_launch_timing": [_int],
    "bs_nontemporal_min_bytes": [_i64],
    "bs_launch_timing_read": [_vp, _vp, _int, _vp],
    "bs_stream_probe": [_int, _vp, _i64, _i64, _vp, _i64, _i64, _vp, _i64, _int, _vp],
}
_RESTYPES = {
    "bs_last_error": ctypes.c_char_p,
    "bs_compress_workspace_bytes": _i64,
    "bs_gemm_compressed_b_workspace_bytes": _i64,
    "bs_gemm_compressed_b_fp8_workspace_bytes": _i64,
    "bs_gemm_compressed_b_packed_workspace_bytes": _i64,
    "bs_compress_noalloc_max_tiles": _i64,
    "bs_linear_relu_compress_max_n": _i64,
    "bs_grad_sums_workspace_bytes": _i64,
    "bs_col_sum_workspace_bytes": _i64,
    "bs_nontemporal_min_bytes": _i64,
    "bs_workspace_amax_slot": _vp,
    "bs_workspace_fallback_counter": _vp,
}

_lib = None
_lock = threading.Lock()


_native_module = None


def native():
    """The native host path (csrc/native.cpp, built as ``_native``), bound to
    the library this module loaded."""
    global _native_module
    if _native_module is None:
        load()
        try:
            from . import _native
        except ImportError as e:
            raise ImportError(f"bitsparse_amd/_native is missing or does not load ({e}): build it with "
                              f"`python -c 'import __graft_entry__ as g; g.build()'`") from e
        _native.init(LIB_PATH)
        _native_module = _native
    return _native_module


class LaunchTimer:
    """Kernel durations of this thread's compress / decompress launches,
    recorded by the library at each kernel's own start and end
    (``bs_launch_timing``), so launch gaps between kernels are not counted.

        with LaunchTimer() as t:
            ... compress / decompress calls ...
        t.times("compress")   # ms per launch, in launch order

    Leaving the block waits for the recorded kernels."""
    KINDS = {0: "compress", 1: "decompress"}
    MAX_LAUNCHES = 1 << 16

    def __enter__(self):
        check(load().bs_launch_timing(1), "bs_launch_timing")
        self.records = []
        return self

    def __exit__(self, *exc):
        L = load()
        ms = (ctypes.c_float * self.MAX_LAUNCHES)()
        kinds = (ctypes.c_int * self.MAX_LAUNCHES)()
        n = ctypes.c_int(0)
        rc = L.bs_launch_timing_read(ms, kinds, self.MAX_LAUNCHES, ctypes.byref(n))
        check(L.bs_launch_timing(0), "bs_launch_timing")
        check(rc, "bs_launch_timing_read")
        self.records = [(self.KINDS.get(kinds[i], str(kinds[i])), ms[i])
                        for i in range(min(n.value, self.MAX_LAUNCHES))]
        return False

    def times(self, kind: str) -> list:
        return [t for k, t in self.records if k == kind]


class BitsparseHipError(RuntimeError):
    """A libbitsparse_hip.so call returned an error status."""


def exported_symbols() -> list[str]:
    return list(_SIGNATURES)


def load() -> ctypes.CDLL:
    """Load the in-tree library (raises if it was not built)."""
    global _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(LIB_PATH):
            raise ImportError(
                f"{LIB_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; "
                f"g.build()'` (hipcc --offload-arch=gfx950)")
        L = ctypes.CDLL(LIB_PATH)
        for name, args in _SIGNATURES.items():
            fn = getattr(L, name)
            fn.argtypes = args
            fn.restype = _RESTYPES.get(name, ctypes.c_int)
        v = L.bs_abi_version()
        if v != ABI_VERSION:
            raise ImportError(f"{LIB_PATH} has ABI {v}, expected {ABI_VERSION}; rebuild it")
        _lib = L
        return L


def check(rc: int, what: str) -> None:
    if rc != BS_OK:
        msg = load().bs_last_error().decode(errors="replace")
        if rc == BS_ERR_INVALID:
            raise ValueError(f"{what}: {msg}")
        raise BitsparseHipError(f"{what} failed ({rc}): {msg}")


def ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def stream_handle(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def require_device(t: torch.Tensor, what: str) -> None:
    """The HIP kernels run on ROCm device tensors only; there is no CPU path."""
    if not t.is_cuda:
        raise RuntimeError(
            f"{what}: bitsparse_amd runs on a ROCm GPU; got a tensor on {t.device}")


# ---------------------------------------------------------------------------
# per-(device, stream) workspace for the single-pass compress and the amax
# (the native module's Workspace: an epoch counter over zero-initialised
# device scratch)
# ---------------------------------------------------------------------------
_EPOCH_LIMIT = (1 << 30) - 1


def workspace_for(device: torch.device):
    return native().workspace(-1 if device.index is None else device.index)
