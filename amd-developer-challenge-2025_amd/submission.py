"""``custom_kernel(data)``: the reference's Python entry point, backed by libfp8bs.so.

Mirrors 1-amd-fp8-mm/amd-fp8-mm-submission.py:594-604 (contract docstring:
1-amd-fp8-mm/0-amd-fp8-mm-new-begins.py:66-77): ``data = (a, b, a_scale, b_scale, c)``, ``c`` is
filled in place and the same tensor object is returned.  Tensors arrive in the reference's layouts:

    a        [m, k]          float8_e4m3fn   stride (1, m)      (K-major: storage is [k][m])
    b        [n, k]          float8_e4m3fn   stride (1, n)
    a_scale  [m, k/128]      float32         stride (1, m)
    b_scale  [ceil(n/128), k/128] float32    stride (1, ceil(n/128))
    c        [m, n]          bfloat16        contiguous

Differences from the reference, by design: OCP e4m3fn instead of e4m3fnuz (gfx950's FP8), the launch
goes to torch's current stream instead of the null stream, errors raise instead of being dropped,
the split-K workspace is cached per device instead of allocated per call
(amd-fp8-mm-submission.py:600), and ``a``/``b`` are never written (the reference's pre-transpose
branch overwrites them, :570-571).
"""
import ctypes

import torch

from . import _lib

_workspaces = {}   # (device index, stream) -> uint8 tensor, grown on demand, reused across calls on that stream
_held = {}         # (device index, stream) -> the tables' buffers whose address a graph holds that is not torch's


def _workspace(device: torch.device, nbytes: int, stream: int = 0, table=None, least: int = 1 << 20) -> torch.Tensor:
    """The K split's partial planes: one buffer per device and stream, so that calls that overlap on two
    streams do not write each other's planes (`table`, `least`: another table of such buffers, its smallest size).

    A call that is captured into a torch.cuda.CUDAGraph takes a buffer of its own from the graph's memory pool, which lives as
    long as the graph: one of the table could be outgrown, and freed, before a replay.  A capture that was begun with HIP
    itself has no such pool.  It is given the table's buffer, which from then on is kept until the process ends, also when a
    larger call outgrows it or the table drops its entry: nothing says how long the graph lives.  Replays of such graphs that
    were captured on one stream share it, as two calls on that stream do, and must not overlap."""
    table = _workspaces if table is None else table
    key = (device.index, stream)
    held = None
    if _capturing(device):
        if _allocates_for_the_graph(device):
            return torch.empty(nbytes, dtype=torch.uint8, device=device)
        held = _held.setdefault(key, [])
    ws = table.get(key)
    if ws is None or ws.numel() < nbytes:
        # A buffer that is outgrown stays alive until this stream's earlier kernels are done with it: the caching
        # allocator hands a freed block only to later work of the stream it was allocated on.
        if ws is None and len(table) >= 16:           # streams come and go: keep the table bounded (oldest entry out)
            table.pop(next(iter(table)))
        ws = None
        if held:                                      # what is kept is used again, and doubles: twice the largest in all
            ws = next((t for t in held if t.numel() >= nbytes), None)
            nbytes = max(nbytes, 2 * held[-1].numel())
        if ws is None:
            ws = torch.empty(max(nbytes, least), dtype=torch.uint8, device=device)
        table[key] = ws
    if held is not None and all(t is not ws for t in held):
        held.append(ws)
        held.sort(key=torch.Tensor.numel)
    return ws


def _capturing(device: torch.device) -> bool:
    """Whether torch's current stream of `device`, which the call goes to, is being captured."""
    if torch.cuda.current_device() == device.index:
        return torch.cuda.is_current_stream_capturing()
    with torch.cuda.device(device):
        return torch.cuda.is_current_stream_capturing()


def _allocates_for_the_graph(device: torch.device) -> bool:
    """Under capture: whether what is allocated now belongs to the graph, so that it may be dropped at once.  Torch's own
    captures allocate from a private pool.  (0.1 to 5 ms with 100 to 20000 live blocks, in captured calls only.)  Other
    allocators than torch's caching one are left to their own rules."""
    if torch.cuda.get_allocator_backend() != "native":
        return True
    probe = torch.empty(1, dtype=torch.uint8, device=device)
    at = probe.data_ptr()
    return any(tuple(s["segment_pool_id"]) != (0, 0) and s["address"] <= at < s["address"] + s["total_size"] for s in torch.cuda.memory_snapshot())


def _is_kmajor(t: torch.Tensor) -> bool:
    """True if the 2-D tensor's storage is its transpose laid out contiguously (stride (1, rows));
    the stride of a dimension of size 1 is immaterial."""
    if t.dim() != 2:
        return False
    r, c = t.shape
    s0, s1 = t.stride()
    return r == 0 or c == 0 or ((r == 1 or s0 == 1) and (c == 1 or s1 == r))


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_plan_cache = {}   # (m, n, k) and ("grouped" | "silu" | "route", sizes ...) -> workspace bytes the call asks for
_PLANS_MAX = 4096

# Dense sizes that the native call of custom_kernel may take, with the workspace bytes that each asks for.  It checks the tensors
# themselves at every call; what it is told here is a fact about the sizes alone.  As many as plans are kept: a server whose batches
# vary has two or three sizes of them for each, and a size that is not here pays for the native attempt and the Python path.
_CHECKED_MAX = _PLANS_MAX
_checked = {}      # (m, n, k) -> bytes
_checked_experts = {}      # the same for grouped_kernel and gate_up_silu: (silu, experts or 0, rows, n, k) -> bytes


def _remember(silu: bool, experts: int, rows: int, n: int, k: int, need) -> None:
    """Sizes that the native call may take from now on; called where the Python path has checked a call of them."""
    key = (int(silu), experts, rows, n, k)
    if need is not None and key not in _checked_experts:
        if len(_checked_experts) >= _CHECKED_MAX:
            _checked_experts.clear()
        _checked_experts[key] = need


def _experts_native(data, silu: bool) -> bool:
    """grouped_kernel's and gate_up_silu's checks and call in native code: whether it took the call."""
    native = _lib.native()
    if native is None:
        return False
    st = native.experts(data, _checked_experts, 0, 0, silu)
    if st < -1:                                   # all is well, and it wants a workspace
        dev = data[0].device
        ws = _workspace(dev, -st, _stream_ptr(dev))
        st = native.experts(data, _checked_experts, ws.data_ptr(), ws.numel(), silu)
    if st > 0:
        _lib.check(st)
    return st == 0


def _grouped_workspace(device, stream, num_experts, rows, n, k):
    """(address, bytes) of the workspace a grouped call can use, (None, 0) if it would not use any."""
    key = ("grouped", num_experts, rows, n, k)
    need = _plan_cache.get(key)
    if need is None:
        if len(_plan_cache) >= _PLANS_MAX:
            _plan_cache.clear()
        with torch.cuda.device(device):              # planned for the CU count of the device it runs on
            need = _plan_cache[key] = int(_lib.load().fp8bs_grouped_workspace_bytes(num_experts, rows, n, k))
    if not need:
        return None, 0
    ws = _workspace(device, need, stream)
    return ws.data_ptr(), ws.numel()


def _stream_ptr(device: torch.device) -> int:
    """Raw hipStream_t of torch's current stream on `device` (the stream the library launches on)."""
    if _raw_stream is not None:
        return _raw_stream(device.index)
    return torch.cuda.current_stream(device).cuda_stream


def _call(fn, device: torch.device, *args) -> None:
    """fn(*args, stream) on torch's current stream of `device`; the library launches on the current device.
    Entering torch.cuda.device costs 1.2 us, asking for the stream through torch.cuda 2.6: with ctypes' marshalling they
    were half of a quantiser call's 12.9 us of host time (now 7.4, of which 3 are the launch and 2 the two allocations)."""
    if torch.cuda.current_device() == device.index:
        st = fn(*args, _stream_ptr(device))
    else:
        with torch.cuda.device(device):
            st = fn(*args, _stream_ptr(device))
    if st:
        _lib.check(st)


_F8, _F32, _BF16 = torch.float8_e4m3fn, torch.float32, torch.bfloat16


def _experts_kmajor(t: torch.Tensor) -> bool:
    """True if every expert of the 3-D tensor is K-major and they lie one behind the other."""
    e, r, c = t.shape
    return t.stride() == (r * c, 1, r) or t.transpose(1, 2).is_contiguous()


def _check_operands(a, b, a_scale, b_scale, c, rows, n, k):
    dev = a.get_device()
    if a.dtype is _F8 and b.dtype is _F8 and a_scale.dtype is _F32 and b_scale.dtype is _F32 and c.dtype is _BF16 \
            and k % 128 == 0 and a.shape == (rows, k) and a_scale.shape == (rows, k // 128) and c.shape == (rows, n) \
            and a.stride() == (1, rows) and a_scale.stride() == (1, rows) and c.is_contiguous() and dev >= 0 \
            and b.get_device() == dev and a_scale.get_device() == dev and b_scale.get_device() == dev and c.get_device() == dev:
        return
    # not the usual layout: a dimension of size 1 or 0, or something to refuse
    if a.dtype != torch.float8_e4m3fn or b.dtype != torch.float8_e4m3fn:
        raise TypeError("a and b must be torch.float8_e4m3fn")
    if a_scale.dtype != torch.float32 or b_scale.dtype != torch.float32:
        raise TypeError("a_scale and b_scale must be torch.float32")
    if c.dtype != torch.bfloat16:
        raise TypeError("c must be torch.bfloat16")
    if k % 128 != 0:
        raise ValueError("k must be a multiple of 128 (got %d)" % k)
    if a.dim() != 2 or a.shape[1] != k or tuple(a_scale.shape) != (rows, k // 128):
        raise ValueError("a / a_scale shapes do not match [rows, k] / [rows, k/128]")
    if not _is_kmajor(a) or not _is_kmajor(a_scale):
        raise ValueError("a and a_scale must be K-major (stride (1, rows)), as the reference lays them out")
    if not c.is_contiguous() or tuple(c.shape) != (rows, n):
        raise ValueError("c must be a contiguous [rows, n] tensor")
    for name, t in (("a", a), ("b", b), ("a_scale", a_scale), ("b_scale", b_scale), ("c", c)):
        if not t.is_cuda:
            raise ValueError("%s must be a GPU tensor: this path has no CPU implementation" % name)
        if t.device != a.device:
            raise ValueError("all tensors must be on the same device")


def plan(m: int, n: int, k: int) -> _lib.Plan:
    """The kernel variant, split-K and grid the library would choose for a dense shape (host only).
    num_cus = 0: the library asks the current device for its CU count, as fp8bs_gemm does (256 without a GPU)."""
    p = _lib.Plan()
    _lib.check(_lib.load().fp8bs_plan(m, n, k, 0, ctypes.byref(p)))
    return p


def workspace_bytes(m: int, n: int, k: int) -> int:
    """Bytes of workspace that a dense call of a shape can make use of (no GPU needed)."""
    return int(_lib.load().fp8bs_workspace_bytes(m, n, k))


def custom_kernel(data, variant: int = 0, split_k: int = 0):
    """Block-scale fp8 gemm: fills and returns ``c`` (see module docstring for the layouts).

    ``variant``/``split_k`` force a kernel variant (FP8BS_VARIANT_*) and a K split for testing
    (``split_k | SPLIT_SUM_IN_KERNEL``: the partitions summed in the one kernel; ``split_k < 0``: K blocks
    dealt to the workgroups); the defaults let the library's planner decide.
    """
    if variant == 0 and split_k == 0:
        dense = _lib.dense()
        if dense is not None:
            st = dense(data, _checked, 0, 0)
            if st < -1:                               # all is well, and it wants a workspace
                dev = data[0].device
                ws = _workspace(dev, -st, _stream_ptr(dev))
                st = dense(data, _checked, ws.data_ptr(), ws.numel())
            if st == 0:
                return data[4]
            if st > 0:
                _lib.check(st)
    a, b, a_scale, b_scale, c = data
    gemm_ex = _lib.calls().gemm_ex
    m, k = a.shape
    n = b.shape[0]
    _check_operands(a, b, a_scale, b_scale, c, m, n, k)
    nb = (n + 127) // 128
    if b.shape != (n, k) or b_scale.shape != (nb, k // 128):
        raise ValueError("b / b_scale shapes do not match [n, k] / [ceil(n/128), k/128]")
    if not _is_kmajor(b) or not _is_kmajor(b_scale):
        raise ValueError("b and b_scale must be K-major (stride (1, n) / (1, ceil(n/128)))")
    if variant == 0 and split_k == 0:
        need = _plan_cache.get((m, n, k))
        if need is None:
            need = workspace_bytes(m, n, k) if (m > 0 and n > 0 and k > 0) else 0
            if len(_plan_cache) >= _PLANS_MAX:
                _plan_cache.clear()
            _plan_cache[(m, n, k)] = need
        if (m, n, k) not in _checked:
            if len(_checked) >= _CHECKED_MAX:
                _checked.clear()
            _checked[(m, n, k)] = need
    else:
        # a forced K split's planes; K blocks dealt to the workgroups (split_k < 0): a header and one fp32 tile per
        # workgroup, at most 64 MiB for every tile shape on 256 CUs
        need = split_k * m * n * 4 if split_k > 1 else ((64 << 20) + 16384 if split_k < 0 else 0)
        if split_k > 0 and split_k & _lib.SPLIT_SUM_IN_KERNEL:
            # summed in the kernel: a header and split_k fp32 tiles per tile (the largest tile is 256 x 256)
            need = 16384 + (split_k & ~_lib.SPLIT_SUM_IN_KERNEL) * (m + 255) * (n + 255) * 4
    dev = a.device
    ws_ptr, ws_len = None, 0
    if need:
        ws = _workspace(dev, need, _stream_ptr(dev))
        ws_ptr, ws_len = ws.data_ptr(), ws.numel()
    _call(gemm_ex, dev, a.data_ptr(), b.data_ptr(), a_scale.data_ptr(), b_scale.data_ptr(),
          c.data_ptr(), ws_ptr, ws_len, m, n, k, variant, split_k)
    return c


def grouped_kernel(data, variant: int = 0):
    """Grouped (MoE expert) variant: ``data = (a, b, a_scale, b_scale, row_offsets, c)``.
    ``variant`` forces a tile (FP8BS_VARIANT_*) for testing; 0 lets the library choose.

    Row-offset convention of 2-amd-moe/3-amd-fp8-moe-hip-myhgemm.py:142-148, :328-336 with the
    total appended: ``row_offsets`` is int32 [E+1], contiguous, on the GPU; expert e owns rows
    [row_offsets[e], row_offsets[e+1]) of the expert-contiguous ``a`` ([rows, k], K-major) and ``c``
    ([rows, n]).  ``b`` is [E, n, k] with each expert K-major (stride (n*k, 1, n)); ``b_scale`` is
    [E, ceil(n/128), k/128] with stride (nb*kb, 1, nb).  Fills and returns ``c``; no host sync.
    A call that splits K keeps a workspace of up to 64 MiB for this device and stream (the one `custom_kernel` uses).
    """
    if variant == 0 and _experts_native(data, False):
        return data[5]
    a, b, a_scale, b_scale, row_offsets, c = data
    rows, k = a.shape
    if b.dim() != 3:
        raise ValueError("b must be [E, n, k]")
    num_experts, n = b.shape[0], b.shape[1]
    _check_operands(a, b, a_scale, b_scale, c, rows, n, k)
    nb, kb = (n + 127) // 128, k // 128
    if b.shape != (num_experts, n, k) or b_scale.shape != (num_experts, nb, kb):
        raise ValueError("b / b_scale shapes do not match [E, n, k] / [E, ceil(n/128), k/128]")
    if not _experts_kmajor(b) or not _experts_kmajor(b_scale):
        raise ValueError("every expert of b and b_scale must be K-major")
    if row_offsets.dtype != torch.int32 or row_offsets.shape != (num_experts + 1,) or row_offsets.device != a.device \
            or not row_offsets.is_contiguous():
        raise ValueError("row_offsets must be a contiguous int32 tensor with num_experts+1 entries on the operands' GPU")
    dev = a.device
    ws_ptr, ws_len = _grouped_workspace(dev, _stream_ptr(dev), num_experts, rows, n, k) if variant == 0 else (None, 0)
    if variant == 0:
        _remember(False, num_experts, rows, n, k, _plan_cache.get(("grouped", num_experts, rows, n, k)))
    _call(_lib.calls().gemm_grouped_ws, dev, a.data_ptr(), b.data_ptr(), a_scale.data_ptr(), b_scale.data_ptr(), c.data_ptr(),
          row_offsets.data_ptr(), num_experts, rows, n, k, variant, 0, ws_ptr, ws_len)
    return c
