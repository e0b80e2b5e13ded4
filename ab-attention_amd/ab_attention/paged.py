"""Weighted paged sparse prefill on gfx950.

``paged_attention`` keeps the reference's signature, validation (ValueError)
and output/LSE layout (ab_attention/flashinfer_backend.py:164-242). The
arithmetic is ``ab_prefill`` in libab_attention_hip.so: a bf16 MFMA
flash-attention kernel that reads each row's KV4 blocks straight from K and
V by their per-head ids and adds the SIP weight of each block to its logits
(the reference's ABSipAttention variant, flashinfer_backend.py:30-59).
``_prefill_dense`` runs the library's dense attention kernel, which walks
every KV4 block of K/V at weight 0 with no page list in memory
(the same rings and pipeline on 16x16x32 MFMA tiles).

The reference translates per-head ids into a global page table and caches it
per descriptor (flashinfer_backend.py:62-74, :202-217); the kernel here
indexes K/V by (head, id) directly, so there is no table and no cache to keep
coherent. Queries are not padded either: the tail of the last query block is
simply not stored (the reference computes it on zero-padded queries and drops
it, flashinfer_backend.py:77-91, :236-242).
"""
from __future__ import annotations

import math

import torch

from . import _lib

_HEAD_DIM = 128
_QUERY_BLOCK = 128
_PAGE_SIZE = 4


def _run(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, ids, weights, samples: int, order, return_lse: bool,
         tail=(None, None, 0), out=None):
    """ab_prefill of q, k, v, read where they lie (samples: _lib.PREFILL_DENSE for
    dense; tail: ids, weights and count of the blocks every row attends to as
    well; out: a view with rows of 128 to write to). The workspace of a call
    that splits its rows over more workgroups lives for the call only (the
    caching allocator keeps it on this stream)."""
    batch, heads, tokens, dim = q.shape
    kv_tokens, device = k.shape[2], q.device
    (q, q_stride), (k, k_stride), (v, v_stride) = _lib.in_place(q), _lib.in_place(k), _lib.in_place(v)
    out_stride = (heads * tokens * dim, tokens * dim, dim) if out is None else out.stride()[:3]
    if batch > 1 and max(q_stride[0], k_stride[0], v_stride[0], out_stride[0]) >= _lib.MAX_STRIDE:
        (q, q_stride), (k, k_stride), (v, v_stride) = _lib.in_one_batch(q, k, v)
    output = torch.empty_like(q, memory_format=torch.contiguous_format) if out is None else out
    lse = torch.empty((batch, heads, tokens), dtype=torch.float32, device=device) if return_lse else None
    lib, address = _lib.load(), _lib.address
    tail_ids, tail_weights, tail_samples = tail
    with _lib.on(device):
        ws_bytes = lib.ab_prefill_workspace_bytes(batch * heads, tokens, kv_tokens, samples + tail_samples)
        workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=device) if ws_bytes else None
        args = _lib.PrefillArgs(address(q), address(k), address(v), address(order), address(ids), address(weights),
                                address(output), address(lse), batch, heads, tokens, kv_tokens, samples, q_stride,
                                k_stride, v_stride, out_stride, address(tail_ids), address(tail_weights),
                                tail_samples, address(workspace), ws_bytes)
        _lib.check(lib.ab_prefill(args, _lib.stream(device)))
    return (output, lse) if return_lse else output


def _prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, ids: torch.Tensor, weights: torch.Tensor,
             order: torch.Tensor | None, return_lse: bool, *, samples: int | None = None, tail=(None, None, 0), out=None):
    """The weighted prefill, with a query token order when one is given;
    ids/weights [rows, S], or any shape of ``samples`` entries per row. Shapes
    are checked by the callers."""
    if ids.dtype != torch.int32 or not ids.is_contiguous():
        ids = ids.to(torch.int32).contiguous()
    if weights.dtype != torch.float32 or not weights.is_contiguous():
        weights = weights.to(torch.float32).contiguous()
    return _run(q, k, v, ids, weights, ids.shape[-1] if samples is None else samples, order, return_lse, tail, out)


def check_prefill_inputs(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> None:
    """paged_attention's Q/K/V checks (reference: flashinfer_backend.py:176-186)."""
    if q.ndim != 4 or q.shape != k.shape or q.shape != v.shape:
        raise ValueError("Q/K/V must have the same [B,H,N,D] shape")
    if q.device != k.device or q.device != v.device:
        raise ValueError("Q/K/V must be on the same CUDA device")
    if q.device.type != "cuda":
        raise ValueError("paged attention requires GPU tensors")
    if q.dtype != torch.bfloat16 or k.dtype != q.dtype or v.dtype != q.dtype:
        raise ValueError("paged attention requires BF16 Q/K/V")
    if q.shape[-1] != _HEAD_DIM or q.shape[2] % _PAGE_SIZE:
        raise ValueError("paged attention requires head_dim=128 and N divisible by 4")


@torch.no_grad()
def paged_attention(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    descriptor: torch.Tensor,
    log_weights: torch.Tensor,
    *,
    return_lse: bool = False,
):
    """Weighted sparse attention over the plan's KV4 blocks; returns o (and base-2 lse)."""
    return _paged_attention(q, k, v, descriptor, log_weights, return_lse)


def _paged_attention(q, k, v, descriptor, log_weights, return_lse):
    """paged_attention for callers that have turned gradients off (each nested
    torch.no_grad costs a small call a microsecond)."""
    check_prefill_inputs(q, k, v)
    batch, heads, tokens, _ = q.shape
    rows = batch * heads * math.ceil(tokens / _QUERY_BLOCK)
    if (descriptor.ndim != 3 or descriptor.shape != log_weights.shape
            or descriptor.shape[0] != rows or descriptor.shape[-1] != 32):
        raise ValueError(f"descriptor and log_weights must share [{rows}, pages, 32] shape")
    if descriptor.device != q.device or log_weights.device != q.device:
        raise ValueError("descriptor and log_weights must be on the Q device")
    return _prefill(q, k, v, descriptor, log_weights, None, return_lse, samples=descriptor.shape[1] * 32)


def _prefill_kv(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, ids: torch.Tensor, weights: torch.Tensor,
                *, return_lse: bool = False, tail=(None, None, 0), out=None):
    """The weighted prefill with K/V of their own length (tail, out: see _run).

    q bf16 [B,H,Nq,128], k/v bf16 [B,H,Nk,128] with Nk % 4 == 0, ids int32 /
    weights f32 [B*H*ceil(Nq/128), S] with S % 8 == 0 (per-head KV4 ids; a -inf
    weight removes its block). Shapes are checked by the callers.
    """
    return _prefill(q, k, v, ids, weights, None, return_lse, tail=tail, out=out)


def _prefill_dense(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, *, return_lse: bool = False, out=None):
    """Dense attention of q bf16 [B,H,Nq,128] over every key of k/v bf16
    [B,H,Nk,128] (Nk % 4 == 0) on the dense kernel (ab_prefill); the
    page list is implicit, so nothing of size rows x blocks is built. Shapes
    are checked by the callers."""
    return _run(q, k, v, None, None, _lib.PREFILL_DENSE, None, return_lse, out=out)


def _remap_ids(ids: torch.Tensor, page_map: torch.Tensor) -> torch.Tensor:
    """int32 ids -> page_map[ids] (ab_remap_ids; ids clamped into the map)."""
    ids = ids.to(torch.int32).contiguous()
    out = torch.empty_like(ids)
    lib = _lib.load()
    with _lib.on(ids.device):
        _lib.check(lib.ab_remap_ids(_lib.ptr(ids), ids.numel(), _lib.ptr(page_map), page_map.numel(),
                                    _lib.ptr(out), _lib.stream(ids.device)))
    return out


def _prefill_ordered(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, order: torch.Tensor, ids: torch.Tensor,
                     weights: torch.Tensor, *, return_lse: bool = False):
    """The weighted prefill of the token-permuted q (query t is stored row
    order[t]) over stored-order k/v pages; output and lse in stored order.
    Shapes are checked by the callers."""
    return _prefill(q, k, v, ids, weights, order.to(torch.int32).contiguous(), return_lse)
