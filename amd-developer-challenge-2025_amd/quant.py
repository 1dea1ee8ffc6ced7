"""GPU block quantisers: row-major fp32/bf16 matrices -> the operands ``custom_kernel`` takes.

The reference has no quantiser (its operands arrive quantised, 1-amd-fp8-mm/0-amd-fp8-mm-new-begins.py:66-77);
these wrap ``fp8bs_quantize_a`` / ``fp8bs_quantize_b`` / ``fp8bs_gather_a`` of libfp8bs.so and return tensors with exactly
the shapes, dtypes and K-major strides of that contract.  The rule is the one of ``inputs.quantize_a`` /
``inputs.quantize_b`` (the host-side quantisers), bit for bit.  No fallback: without the library the
import of ``_lib`` raises.
"""
from typing import Optional, Tuple

import torch

from . import _lib
from .submission import _call

_DTYPES = {torch.float32: 0, torch.bfloat16: 1}


def _check_input(x: torch.Tensor, name: str) -> None:
    if x.dtype not in _DTYPES:
        raise TypeError("%s must be float32 or bfloat16, got %s" % (name, x.dtype))
    if x.dim() != 2 or not x.is_cuda:
        raise ValueError("%s must be a 2-D tensor on the GPU" % name)
    k = x.shape[1]
    if k % 128 != 0:
        raise ValueError("%s: K = %d is not a multiple of 128" % (name, k))
    if k > 0 and x.stride(1) != 1:
        raise ValueError("%s must be row-major (stride 1 along K), got strides %s" % (name, tuple(x.stride())))


def _k_major(rows: int, k: int, dtype: torch.dtype, device: torch.device) -> torch.Tensor:
    """An uninitialised [rows, k] tensor whose storage is [k][rows]."""
    return torch.empty_strided((rows, k), (1, rows or 1), dtype=dtype, device=device)


def _native_quantize(x, row_map, of_b: bool):
    """The native call's result, or None where it does not take this one."""
    native = _lib.native()
    out = native.quantize(x, row_map, of_b) if native is not None else None
    if type(out) is int:
        _lib.check(out)
    return out


def _quantise_then_gather(dtype: torch.dtype, t: int, m: int, k: int, row_map: torch.Tensor) -> bool:
    """Whether two kernels are faster than one for m gathered rows of t tokens, by measurement (us, one / two): where rows repeat
    often, the output is large and ``gather_a`` has a fast path that keeps 8 or 16 k rows of the source in LDS (T and M multiples
    of 4, T <= 8192; up to 6826 tokens three of its workgroups fit a CU, beyond that two).  Reading the tokens again costs fp32
    twice what it costs bf16, so its lines lie lower.

    bf16, 4096 tokens: to 8 of 7168 values 103 / 85, of 4096 47.4 / 47.7, of 2048 24.4 / 27.5; to 5 of 7168 65.9 / 61.7, of 4096
    30.5 / 38.7; to 4 of 7168 51.6 / 53.8.  6016 tokens to 8 of 7168 158 / 135, to 6 of 4096 59.3 / 61.8; 6976 to 8 of 7168 184 /
    189; 8192 to 8 of 7168 224 / 233, of 1024 24.4 / 32.5; 16384 to 8 of 7168 447 / 831.
    fp32, 4096 tokens: to 8 of 2048 31.5 / 28.9, of 1024 16.5 / 20.3; to 4 of 7168 83 / 68, of 4096 40.8 / 33.7, of 2048 17.6 /
    25.4; to 3 of 7168 63.5 / 63.0.  6016 tokens to 4 of 2048 28.9 / 28.5; 8192 to 8 of 2048 80.7 / 67.9, of 1024 30.7 / 32.8; to 5
    of 2048 51.4 / 54.5; to 4 of 7168 167 / 166; 16384 to 8 of 7168 712 / 900.
    """
    if t % 4 or m % 4 or not 0 < t <= 8192 or row_map.data_ptr() % 16:
        return False
    three_a_cu = t <= 6826
    if dtype == torch.bfloat16:
        return three_a_cu and m > 4 * t and m * k >= (100 if t <= 4096 else 144) << 20
    return m >= 4 * t and m * k >= (48 if three_a_cu else 84) << 20


def quantize_a(x: torch.Tensor, row_map: Optional[torch.Tensor] = None, fused: Optional[bool] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """x [T, K] -> (a e4m3fn [M, K] stride (1, M), a_scale fp32 [M, K/128] stride (1, M)).

    Without ``row_map`` M = T.  With ``row_map`` (int32 [M] on the GPU) output row i is input row
    ``row_map[i]``: the expert-contiguous gather of routed tokens.  Two routes, the same bytes: the gather fused into the
    quantiser (one kernel), or every token quantised once and the bytes gathered by ``gather_a`` (two kernels), see
    ``_quantise_then_gather``.  ``fused`` = True / False forces the one-kernel / two-kernel route.
    """
    if row_map is None and fused is None:
        out = _native_quantize(x, None, False)
        if out is not None:
            return out
    _check_input(x, "x")
    t, k = x.shape
    if row_map is not None:
        if row_map.dtype != torch.int32 or row_map.dim() != 1 or row_map.device != x.device or not row_map.is_contiguous():
            raise ValueError("row_map must be a contiguous int32 vector on x's device")
        m = row_map.numel()
        if fused is None:
            fused = not _quantise_then_gather(x.dtype, t, m, k, row_map)
        if not fused:
            return gather_a(*quantize_a(x), row_map)
        out = _native_quantize(x, row_map, False)
        if out is not None:
            return out
    else:
        m = t
    dev = x.device
    a, a_scale = _k_major(m, k, torch.float8_e4m3fn, dev), _k_major(m, k // 128, torch.float32, dev)
    _call(_lib.calls().quantize_a, dev, x.data_ptr(), _DTYPES[x.dtype], x.stride(0) if t > 1 else max(k, 1),
          row_map.data_ptr() if row_map is not None else None, t, a.data_ptr(), a_scale.data_ptr(), m, k)
    return a, a_scale


def quantize_b(w: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """w [N, K] -> (b e4m3fn [N, K] stride (1, N), b_scale fp32 [ceil(N/128), K/128] stride (1, NB))."""
    out = _native_quantize(w, None, True)
    if out is not None:
        return out
    _check_input(w, "w")
    n, k = w.shape
    dev = w.device
    b, b_scale = _k_major(n, k, torch.float8_e4m3fn, dev), _k_major((n + 127) // 128, k // 128, torch.float32, dev)
    _call(_lib.calls().quantize_b, dev, w.data_ptr(), _DTYPES[w.dtype], w.stride(0) if n > 1 else max(k, 1),
          b.data_ptr(), b_scale.data_ptr(), n, k)
    return b, b_scale


def gather_a(a: torch.Tensor, a_scale: torch.Tensor, row_map: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Rows ``row_map`` of quantised activations: (a [T, K], a_scale [T, K/128]) K-major -> the same for M rows.

    ``gather_a(*quantize_a(x), row_map)`` returns exactly what ``quantize_a(x, row_map)`` returns, but
    quantises every token once instead of once per routed copy (the reference copies rows into expert
    order, 2-amd-moe/3-amd-fp8-moe-hip-myhgemm.py:174-191).  Entries of ``row_map`` outside [0, T) give
    zero rows with scale 1e-12.
    """
    if a.dtype != torch.float8_e4m3fn or a_scale.dtype != torch.float32 or a.dim() != 2 or a_scale.dim() != 2 or not a.is_cuda:
        raise TypeError("a must be a float8_e4m3fn and a_scale a float32 2-D tensor on the GPU")
    t, k = a.shape
    if k % 128 != 0 or tuple(a_scale.shape) != (t, k // 128):
        raise ValueError("a [T, K] needs K %% 128 == 0 and a_scale [T, K/128]; got %s and %s" % (tuple(a.shape), tuple(a_scale.shape)))
    if not a.t().is_contiguous() or not a_scale.t().is_contiguous():
        raise ValueError("a and a_scale must be K-major (stride 1 along rows)")
    if row_map.dtype != torch.int32 or row_map.dim() != 1 or row_map.device != a.device or not row_map.is_contiguous():
        raise ValueError("row_map must be a contiguous int32 vector on a's device")
    m = row_map.numel()
    dev = a.device
    out, out_scale = _k_major(m, k, torch.float8_e4m3fn, dev), _k_major(m, k // 128, torch.float32, dev)
    _call(_lib.calls().gather_a, dev, a.data_ptr(), a_scale.data_ptr(), t, row_map.data_ptr(), out.data_ptr(), out_scale.data_ptr(), m, k)
    return out, out_scale
