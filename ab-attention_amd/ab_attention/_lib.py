"""ctypes binding of the gfx950 libraries.

``libab_attention_hip.so`` carries every entry point of
``include/ab_attention.h``. ``libab_attention_static.so`` carries only
``ab_ibcs_sip_static`` (``include/ab_attention_static.h``) and its static
512 MiB device scratch; it is loaded by ``load_static()`` on first use, so a
process that never asks for it holds no such array. torch is imported first
so that the library binds to the HIP runtime torch already loaded (both carry
the soname ``libamdhip64.so.7``), which makes torch's streams valid handles
for the library. There is no fallback: if the library is missing or fails to
load, every entry point raises.
"""
from __future__ import annotations

import contextlib
import ctypes
import os

import torch

LIB_NAME = "libab_attention_hip.so"
LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), LIB_NAME)
STATIC_LIB_NAME = "libab_attention_static.so"
STATIC_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), STATIC_LIB_NAME)

_P = ctypes.c_void_p
_I64 = ctypes.c_int64
_SZ = ctypes.c_size_t



PREFILL_DENSE = -1  # AB_PREFILL_DENSE


class PrefillArgs(ctypes.Structure):
    """ab_prefill_args of include/ab_attention.h."""

    _fields_ = [("q", _P), ("k", _P), ("v", _P), ("order", _P), ("ids", _P), ("log_weights", _P), ("out", _P),
                ("lse", _P), ("batch", _I64), ("heads", _I64), ("q_tokens", _I64), ("kv_tokens", _I64),
                ("samples", _I64), ("q_stride", _I64 * 3), ("k_stride", _I64 * 3), ("v_stride", _I64 * 3),
                ("out_stride", _I64 * 3), ("tail_ids", _P), ("tail_log_weights", _P), ("tail_samples", _I64),
                ("workspace", _P), ("workspace_bytes", _SZ)]


class PlanArgs(ctypes.Structure):
    """ab_plan_args of include/ab_attention.h."""

    _fields_ = [("q", _P), ("k", _P), ("order", _P), ("offsets", _P), ("ids", _P), ("log_weights", _P),
                ("batch", _I64), ("heads", _I64), ("first_head", _I64), ("head_count", _I64), ("tokens", _I64),
                ("samples", _I64), ("q_stride", _I64 * 3), ("k_stride", _I64 * 3), ("workspace", _P),
                ("workspace_bytes", _SZ)]


# name -> (restype, argtypes); mirrors include/ab_attention.h
SIGNATURES = {
    "ab_last_error": (ctypes.c_char_p, []),
    "ab_abi_version": (ctypes.c_int, []),
    "ab_ibcs_workspace_bytes": (_SZ, [_I64, _I64]),
    "ab_ibcs": (ctypes.c_int, [_P, _P, _I64, _I64, _P, _SZ, _P, _P]),
    "ab_ibcs_lse_stride": (_I64, [_I64]),
    "ab_ibcs_cluster_pool": (ctypes.c_int, [_P, _P, _I64, _I64, _P, _P, _P, _P]),
    "ab_ibcs_lse": (ctypes.c_int, [_P, _P, _I64, _I64, _P, _P, _P, _P]),
    "ab_ibcs_masses": (ctypes.c_int, [_P, _P, _P, _P, _I64, _I64, _P, _P]),
    "ab_sip": (ctypes.c_int, [_P, _P, _I64, _I64, _I64, _P, _P, _P]),
    "ab_paged_prefill": (ctypes.c_int, [_P, _P, _P, _I64, _I64, _P, _P, _I64, _P, _P, _P]),
    "ab_paged_prefill_kv": (ctypes.c_int, [_P, _P, _P, _I64, _I64, _I64, _P, _P, _I64, _P, _P, _P]),
    "ab_merge_states": (ctypes.c_int, [_P, _P, _P, _P, _I64, _P, _P, _P]),
    "ab_ibcs_ordered": (ctypes.c_int, [_P, _P, _P, _I64, _I64, _P, _SZ, _P, _P]),
    "ab_remap_ids": (ctypes.c_int, [_P, _I64, _P, _I64, _P, _P]),
    "ab_paged_prefill_ordered": (ctypes.c_int, [_P, _P, _P, _P, _I64, _I64, _P, _P, _I64, _P, _P, _P]),
    "ab_ibcs_sip_workspace_bytes": (_SZ, [_I64, _I64]),
    "ab_ibcs_sip": (ctypes.c_int, [_P, _P, _P, _I64, _I64, _P, _I64, _P, _SZ, _P, _P, _P]),
    "ab_ibcs_sip_exact_draws": (ctypes.c_int, [_P, _P, _P, _I64, _I64, _P, _I64, _P, _SZ, _P, _P, _P]),
    "ab_plan": (ctypes.c_int, [ctypes.POINTER(PlanArgs), _P]),
    "ab_dense_prefill": (ctypes.c_int, [_P, _P, _P, _I64, _I64, _I64, _P, _P, _P]),
    "ab_prefill_launch_slots": (_I64, [_I64, _I64]),
    "ab_prefill_workspace_bytes": (_SZ, [_I64, _I64, _I64, _I64]),
    "ab_prefill": (ctypes.c_int, [ctypes.POINTER(PrefillArgs), _P]),
}

# name -> (restype, argtypes); mirrors include/ab_attention_static.h
STATIC_SIGNATURES = {
    "ab_ibcs_sip_static": (ctypes.c_int, [_P, _P, _P, _I64, _I64, _P, _I64, _P, _P, _P]),
}

ABI_VERSION = 7
_lib = None
_static = None


class NativeLibraryError(RuntimeError):
    """The HIP library is missing, stale or failed to load."""


def load():
    """Load (once) and return the ctypes handle with typed entry points."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise NativeLibraryError(
            f"{LIB_NAME} is not built (expected at {LIB_PATH}); run __graft_entry__.build() "
            "or `make -C ab-attention_amd/csrc`")
    try:
        handle = ctypes.CDLL(LIB_PATH)
    except OSError as exc:  # pragma: no cover - depends on the runtime
        raise NativeLibraryError(f"failed to load {LIB_PATH}: {exc}") from exc
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(handle, name)
        fn.restype = restype
        fn.argtypes = argtypes
    if handle.ab_abi_version() != ABI_VERSION:
        raise NativeLibraryError(f"{LIB_NAME} ABI {handle.ab_abi_version()} != expected {ABI_VERSION}")
    _lib = handle
    return _lib


def load_static():
    """Load (once) ``libab_attention_static.so`` after the main library and
    return its handle; its failures are reported by the main library's
    ``ab_last_error``."""
    global _static
    if _static is not None:
        return _static
    load()
    if not os.path.exists(STATIC_LIB_PATH):
        raise NativeLibraryError(
            f"{STATIC_LIB_NAME} is not built (expected at {STATIC_LIB_PATH}); run __graft_entry__.build() "
            "or `make -C ab-attention_amd/csrc`")
    try:
        handle = ctypes.CDLL(STATIC_LIB_PATH)
    except OSError as exc:  # pragma: no cover - depends on the runtime
        raise NativeLibraryError(f"failed to load {STATIC_LIB_PATH}: {exc}") from exc
    for name, (restype, argtypes) in STATIC_SIGNATURES.items():
        fn = getattr(handle, name)
        fn.restype = restype
        fn.argtypes = argtypes
    _static = handle
    return _static


def check(rc: int) -> None:
    """Raise RuntimeError (as the reference's TORCH_CHECK does) on a nonzero status."""
    if rc != 0:
        raise RuntimeError(load().ab_last_error().decode(errors="replace"))


def ptr(t: torch.Tensor | None) -> ctypes.c_void_p:
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def stream(device: torch.device) -> ctypes.c_void_p:
    """The current torch stream of ``device`` as a hipStream_t (the raw handle;
    ``torch.cuda.current_stream`` makes a Stream object for it, 1.8 us)."""
    return ctypes.c_void_p(torch._C._cuda_getCurrentRawStream(device.index))


_HERE = contextlib.nullcontext()


def on(device: torch.device):
    """``torch.cuda.device(device)``, free where it is the current device."""
    return _HERE if torch.cuda.current_device() == device.index else torch.cuda.device(device)


def address(t: torch.Tensor | None) -> int:
    """``ptr`` for a field of PrefillArgs or PlanArgs."""
    return 0 if t is None else t.data_ptr()


def in_place(t: torch.Tensor):
    """(tensor, its (batch, head, token) strides in elements) for t [B, H, N,
    128]: t itself where the library can read its rows in place (contiguous
    rows of 128 that start on 16 bytes, at any batch, head and token strides
    with at most 24-bit page sizes and 4 GiB per head), else a contiguous copy."""
    if not t.is_contiguous():
        batch, head, token, dim = t.stride()
        if (dim == 1 and not (batch | head | token) & 7 and max(batch, head) < (1 << 34) and 0 < token < (1 << 21)
                and t.shape[2] * token < (1 << 31) and t.data_ptr() % 16 == 0):
            return t, (batch, head, token)
        t = t.contiguous()
    _, heads, tokens, dim = t.shape  # not t.stride(): it may be anything where a size is 1
    return t, (heads * tokens * dim, tokens * dim, dim)


MAX_STRIDE = 1 << 34


def in_one_batch(*tensors):
    """``in_place`` of tensors of which some (contiguous) one has a batch stride
    of MAX_STRIDE elements or more: the library takes that only where every
    tensor's batch items follow its heads at the head stride, so the others are
    copied if need be."""
    return tuple((t, stride) if stride[0] == t.shape[1] * stride[1] else in_place(t.contiguous())
                 for t, stride in map(in_place, tensors))
