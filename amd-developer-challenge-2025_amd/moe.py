"""MoE routing on the GPU: top-k selection, row_offsets and the expert-contiguous row order.

Wraps ``fp8bs_moe_topk`` / ``fp8bs_moe_route`` of libfp8bs.so.  Roles in the reference
(2-amd-moe/amd-moe-submission.py): ``top4_nre32`` / ``topk`` (:32-105), ``calculate_index`` (:107-156)
and the host read of the counts (:230-234); here nothing synchronises with the host and the row order is
deterministic (by expert, then token id).  The outputs plug into ``quant.quantize_a(x, row_map)`` and
``grouped_kernel``.  No fallback: without the library the import of ``_lib`` raises.
"""
from typing import Optional, Tuple

import torch

from . import _lib
from .submission import _PLANS_MAX, _call, _check_operands, _experts_kmajor, _experts_native, _grouped_workspace, _is_kmajor, _plan_cache, _remember, _stream_ptr, _workspace


_route_ws = {}     # (device index, stream) -> uint8 tensor: the routing kernels' scratch, grown on demand, reused across
                   # calls on that stream (calls that overlap on two streams of one GPU must not share the count tables)


def topk(scores: torch.Tensor, k: int, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """scores fp32 [T, E] row-major on the GPU -> int32 [T, k], best first, lowest index first among equals.
    ``out`` (contiguous int32 [T, k] on the same GPU) is filled and returned if given: no allocation."""
    native = _lib.native() if out is None else None
    if native is not None:
        got = native.topk(scores, k)
        if type(got) is int:
            _lib.check(got)
        if got is not None:
            return got
    if scores.dtype != torch.float32 or scores.dim() != 2 or not scores.is_cuda or not scores.is_contiguous():
        raise ValueError("scores must be a contiguous float32 [tokens, experts] tensor on the GPU")
    t, e = scores.shape
    if out is None:
        out = torch.empty(t, k, dtype=torch.int32, device=scores.device)
    elif out.dtype != torch.int32 or tuple(out.shape) != (t, k) or out.device != scores.device or not out.is_contiguous():
        raise ValueError("out must be a contiguous int32 [tokens, k] tensor on the scores' device")
    _call(_lib.calls().moe_topk, scores.device, scores.data_ptr(), t, e, k, out.data_ptr())
    return out


def route(top_idx: torch.Tensor, experts: int, out: Optional[Tuple[torch.Tensor, torch.Tensor, torch.Tensor]] = None
          ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """top_idx int32 [T, k] -> (row_offsets int32 [E+1], row_map int32 [T*k], slot_of int32 [T, k]).

    Expert e owns rows [row_offsets[e], row_offsets[e+1]); ``row_map[row]`` is the token of that row
    (rows of an expert ordered by token id); ``slot_of[t, j]`` is the row of token t's j-th choice.
    Rows beyond ``row_offsets[E]`` (only if some entries of ``top_idx`` are outside [0, E)) are -1.
    ``out`` = the three tensors of a previous call (or any of those shapes, contiguous int32 on the same GPU)
    are filled and returned: a layer that routes every step then allocates nothing per call.
    """
    if top_idx.dtype != torch.int32 or top_idx.dim() != 2 or not top_idx.is_cuda or not top_idx.is_contiguous():
        raise ValueError("top_idx must be a contiguous int32 [tokens, topk] tensor on the GPU")
    t, k = top_idx.shape
    dev = top_idx.device
    need = _plan_cache.get(("route", t, experts))
    if need is None:
        if len(_plan_cache) >= _PLANS_MAX:
            _plan_cache.clear()
        need = _plan_cache[("route", t, experts)] = _lib.load().fp8bs_moe_route_workspace_bytes(t, experts)
    ws = _workspace(dev, need, _stream_ptr(dev), _route_ws, 4096)
    native = _lib.native() if out is None else None
    if native is not None:
        got = native.route(top_idx, experts, ws.data_ptr(), ws.numel())
        if type(got) is int:
            _lib.check(got)
        if got is not None:
            return got
    if out is None:
        row_offsets = torch.empty(experts + 1, dtype=torch.int32, device=dev)
        row_map = torch.empty(t * k, dtype=torch.int32, device=dev)
        slot_of = torch.empty(t, k, dtype=torch.int32, device=dev)
    else:
        row_offsets, row_map, slot_of = out
        for name, x, shape in (("row_offsets", row_offsets, (experts + 1,)), ("row_map", row_map, (t * k,)), ("slot_of", slot_of, (t, k))):
            if x.dtype != torch.int32 or tuple(x.shape) != shape or x.device != dev or not x.is_contiguous():
                raise ValueError("out: %s must be a contiguous int32 tensor of shape %s on top_idx's device" % (name, shape))
    _call(_lib.calls().moe_route, dev, top_idx.data_ptr(), t, experts, k, row_offsets.data_ptr(), row_map.data_ptr(),
          slot_of.data_ptr(), ws.data_ptr(), ws.numel())
    return row_offsets, row_map, slot_of


def gate_up_silu(data):
    """Gate/up projection with silu(gate) * up fused into the GEMM: ``data = (a, b, a_scale, b_scale, row_offsets, h)``.

    ``b`` holds gate and up weights interleaved by row (row 2i = gate_i, row 2i+1 = up_i), [E, n, k] with
    every expert K-major (or [n, k] K-major with ``row_offsets=None`` for one dense weight); ``h`` is
    bf16 [rows, n/2].  Role of re_silu_mul_kernel (2-amd-moe/amd-moe-submission.py:366-407) fused as in
    2-amd-moe/5-amd-fp8-moe-hip-fuse.py:366-408.  Fills and returns ``h``.
    A call that splits K keeps its workspace (grouped: up to 64 MiB) for this device and stream, the one `custom_kernel` uses.
    """
    if _experts_native(data, True):
        return data[5]
    a, b, a_scale, b_scale, row_offsets, h = data
    if a.dim() != 2:
        raise ValueError("a must be a [rows, k] tensor")
    rows, k = a.shape
    grouped = row_offsets is not None
    if b.dim() != (3 if grouped else 2):
        raise ValueError("b must be [E, n, k] with row_offsets and [n, k] without")
    num_experts = b.shape[0] if grouped else 0
    n = b.shape[1] if grouped else b.shape[0]
    if n % 2:
        raise ValueError("n must be even: gate and up rows come in pairs")
    nb, kb = (n + 127) // 128, k // 128
    if grouped:
        if b.shape != (num_experts, n, k) or b_scale.shape != (num_experts, nb, kb):
            raise ValueError("b / b_scale shapes do not match [E, n, k] / [E, ceil(n/128), k/128]")
        if not _experts_kmajor(b) or not _experts_kmajor(b_scale):
            raise ValueError("every expert of b and b_scale must be K-major")
        if row_offsets.dtype != torch.int32 or row_offsets.shape != (num_experts + 1,) or row_offsets.device != a.device \
                or not row_offsets.is_contiguous():
            raise ValueError("row_offsets must be a contiguous int32 tensor with num_experts+1 entries on the operands' GPU")
    else:
        if b.shape != (n, k) or b_scale.shape != (nb, kb):
            raise ValueError("b / b_scale shapes do not match [n, k] / [ceil(n/128), k/128]")
        if not _is_kmajor(b) or not _is_kmajor(b_scale):
            raise ValueError("b and b_scale must be K-major")
    # dtypes, devices, shapes and K-major strides of a, a_scale and h ([rows, n/2]) as for the plain GEMM's c
    _check_operands(a, b, a_scale, b_scale, h, rows, n // 2, k)
    dev = a.device
    if grouped:
        ws_ptr, ws_len = _grouped_workspace(dev, _stream_ptr(dev), num_experts, rows, n, k)
        _remember(True, num_experts, rows, n, k, _plan_cache.get(("grouped", num_experts, rows, n, k)))
    else:
        need = _plan_cache.get(("silu", rows, n, k))
        if need is None:
            if len(_plan_cache) >= _PLANS_MAX:
                _plan_cache.clear()
            with torch.cuda.device(dev):             # planned for the CU count of the device it runs on
                need = _plan_cache[("silu", rows, n, k)] = int(_lib.load().fp8bs_silu_mul_workspace_bytes(rows, n, k))
        ws = _workspace(dev, need, _stream_ptr(dev)) if need else None
        ws_ptr, ws_len = (ws.data_ptr(), ws.numel()) if need else (None, 0)
        _remember(True, 0, rows, n, k, need)
    _call(_lib.calls().gemm_silu_mul_ws, dev, a.data_ptr(), b.data_ptr(), a_scale.data_ptr(), b_scale.data_ptr(), h.data_ptr(),
          row_offsets.data_ptr() if grouped else None, num_experts, rows, n, k, 0, 0, ws_ptr, ws_len)
    return h


def combine(y: torch.Tensor, slot_of: torch.Tensor, weights: torch.Tensor) -> torch.Tensor:
    """out[t] = sum_j weights[t, j] * y[slot_of[t, j]]  (y bf16 [rows, d], weights fp32 [T, k]) -> bf16 [T, d].

    Role of pack_output (2-amd-moe/amd-moe-submission.py:239-301); fp32 accumulation in the order of j.
    """
    native = _lib.native()
    if native is not None:
        got = native.combine(y, slot_of, weights)
        if type(got) is int:
            _lib.check(got)
        if got is not None:
            return got
    if y.dtype != torch.bfloat16 or y.dim() != 2 or not y.is_contiguous() or not y.is_cuda:
        raise ValueError("y must be a contiguous bfloat16 [rows, d] tensor on the GPU")
    if slot_of.dtype != torch.int32 or not slot_of.is_contiguous() or weights.dtype != torch.float32 \
            or not weights.is_contiguous() or slot_of.shape != weights.shape or slot_of.dim() != 2:
        raise ValueError("slot_of (int32) and weights (float32) must be contiguous [tokens, topk] tensors")
    t, k = slot_of.shape
    d = y.shape[1]
    for name, x in (("slot_of", slot_of), ("weights", weights)):
        if t and d and not x.is_cuda and not x.is_pinned():       # (the kernel would fault on pageable host memory; without outputs there is no launch)
            raise ValueError("%s must be on the GPU" % name)
    out = torch.empty(t, d, dtype=torch.bfloat16, device=y.device)
    _call(_lib.calls().moe_combine, y.device, y.data_ptr(), y.shape[0], slot_of.data_ptr(), weights.data_ptr(), out.data_ptr(), t, k, d)
    return out
