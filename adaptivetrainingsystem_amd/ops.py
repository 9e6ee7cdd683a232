"""Tensor-level wrappers of the libats_gfx950 entry points.

PyTorch is used for device memory and streams only: every function here
validates shapes on the host, allocates outputs with torch, and enqueues the
hand-written HIP kernels on torch's current stream.  Tensors must live on the
GPU; there is no CPU path.
"""
from __future__ import annotations

import ctypes
import functools
import threading
from array import array
from typing import Optional, Sequence, Tuple

import torch

from . import _lib
from ._lib import ATS_BF16, ATS_F32, IDX_I32, IDX_I64, ROUTE_SOFTMAX_TOPK, ROUTE_TOPK_SOFTMAX, AtsError, check

_DT = {torch.float32: ATS_F32, torch.bfloat16: ATS_BF16}


def _tag(t: torch.Tensor) -> int:
    try:
        return _DT[t.dtype]
    except KeyError:
        raise AtsError(f"unsupported dtype {t.dtype}: the gfx950 kernels take float32 or bfloat16") from None


def _need_gpu(*tensors: Optional[torch.Tensor]) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise AtsError("tensor is not on the GPU: the gfx950 path has no CPU fallback")


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_raw_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream() -> int:
    """Handle of torch's current stream on the current device.  The raw accessors skip the Stream object
    and the device bookkeeping of torch.cuda.current_stream (8 us a call, a tenth of a decode step)."""
    if _raw_stream is not None and _raw_device is not None:
        return _raw_stream(_raw_device())
    return torch.cuda.current_stream().cuda_stream


def _ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


# --------------------------------------------------------------------------- RMSNorm
def rmsnorm(x: torch.Tensor, weight: Optional[torch.Tensor], eps: float = 1e-6) -> torch.Tensor:
    _need_gpu(x, weight)
    H = x.shape[-1]
    xc = x.contiguous()
    if weight is not None:
        if weight.numel() != H:
            raise AtsError(f"rmsnorm: weight has {weight.numel()} elements, hidden size is {H}")
        weight = weight.contiguous()
    y = torch.empty_like(xc)
    rows = xc.numel() // H if H else 0
    check(_lib.load().ats_rmsnorm_fwd(xc.data_ptr(), _ptr(weight), y.data_ptr(), rows, H, float(eps), _tag(xc),
                                      _tag(weight) if weight is not None else ATS_F32, _stream()), "ats_rmsnorm_fwd")
    return y.view(x.shape)


# --------------------------------------------------------------------------- RoPE
def rope_table(seq_len: int, dim: int, theta: float = 10000.0, scaling_factor: Optional[float] = None,
               half: bool = False, device=None) -> Tuple[torch.Tensor, torch.Tensor]:
    device = torch.device("cuda") if device is None else torch.device(device)
    if device.type != "cuda":
        raise AtsError("rope_table: the table is built by a GPU kernel; pass a cuda device")
    cols = dim // 2 if half else dim
    cos = torch.empty(seq_len, cols, dtype=torch.float32, device=device)
    sin = torch.empty(seq_len, cols, dtype=torch.float32, device=device)
    with torch.cuda.device(device):
        check(_lib.load().ats_rope_table(cos.data_ptr(), sin.data_ptr(), seq_len, dim, cols, float(theta),
                                         1.0 if scaling_factor is None else float(scaling_factor), _stream()),
              "ats_rope_table")
    return cos, sin


def _bhl_strides(t: torch.Tensor):
    if t.stride(3) != 1:
        t = t.contiguous()
    return t, t.stride(0), t.stride(1), t.stride(2)


def rope(q: torch.Tensor, k: Optional[torch.Tensor], cos: torch.Tensor, sin: torch.Tensor,
         position_offset: int = 0, inverse: bool = False) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """q [B,Hq,L,D], k [B,Hkv,L,D] (any batch/head/position strides), cos/sin float32
    [>= offset+L, D or D/2].  Returns new contiguous tensors.  inverse=True applies the
    inverse rotation, i.e. the gradient of the forward rotation."""
    _need_gpu(q, k, cos, sin)
    if q.dim() != 4 or (k is not None and k.dim() != 4):
        raise AtsError("rope: q and k must be [batch, heads, seq, head_dim]")
    B, Hq, L, D = q.shape
    Hkv = 0
    if k is not None:
        if k.shape[0] != B or k.shape[2] != L or k.shape[3] != D or k.dtype != q.dtype:
            raise AtsError(f"rope: k {tuple(k.shape)}/{k.dtype} does not match q {tuple(q.shape)}/{q.dtype}")
        Hkv = k.shape[1]
    if cos.dtype != torch.float32 or sin.dtype != torch.float32 or cos.shape != sin.shape or cos.dim() != 2:
        raise AtsError("rope: cos/sin must be float32 2-D tables of equal shape")
    if cos.stride(1) != 1 or sin.stride(1) != 1 or cos.stride(0) != sin.stride(0):
        cos, sin = cos.contiguous(), sin.contiguous()
    q, qsb, qsh, qsl = _bhl_strides(q)
    q_out = torch.empty((B, Hq, L, D), dtype=q.dtype, device=q.device)
    k_out = None
    ksb = ksh = ksl = 0
    if k is not None:
        k, ksb, ksh, ksl = _bhl_strides(k)
        k_out = torch.empty((B, Hkv, L, D), dtype=k.dtype, device=k.device)
    name = "ats_rope_bwd" if inverse else "ats_rope_fwd"
    check(getattr(_lib.load(), name)(q.data_ptr(), _ptr(k), q_out.data_ptr(), _ptr(k_out), cos.data_ptr(),
                                     sin.data_ptr(), cos.stride(0), cos.shape[0], B, Hq, Hkv, L, D,
                                     int(position_offset), qsb, qsh, qsl, ksb, ksh, ksl, _tag(q), _stream()), name)
    return q_out, k_out


def rope_strided(ins: Sequence[Optional[torch.Tensor]], outs: Sequence[Optional[torch.Tensor]], cos: torch.Tensor,
                 sin: torch.Tensor, position_offset: int = 0, inverse: bool = False) -> None:
    """Rotates ins[0], ins[1] into outs[0], outs[1] and copies ins[2] into outs[2] (None: no such segment), one launch; all
    [B, heads, L, D] of one type with any strides but that of D."""
    _need_gpu(*ins, *outs, cos, sin)
    given = [t for t in ins if t is not None]
    B, _, L, D = given[0].shape
    src, dst, ss, ds, heads = [], [], [], [], []
    for i, o in zip(ins, outs):
        if i is None:
            src.append(None), dst.append(None), heads.append(0)
            ss += [0, 0, 0]
            ds += [0, 0, 0]
            continue
        if i.dim() != 4 or i.shape != o.shape or i.shape[0] != B or i.shape[2] != L or i.shape[3] != D \
                or i.dtype != given[0].dtype or o.dtype != i.dtype or o.stride(3) != 1:
            raise AtsError(f"rope_strided: segment {tuple(i.shape)}/{i.dtype} -> {tuple(o.shape)}/{o.dtype}")
        i, *strides = _bhl_strides(i)
        given.append(i)                              # (a copy stays alive until the launch is queued)
        src.append(i.data_ptr()), dst.append(o.data_ptr()), heads.append(i.shape[1])
        ss += strides
        ds += o.stride()[:3]
    if cos.dtype != torch.float32 or sin.dtype != torch.float32 or cos.shape != sin.shape or cos.dim() != 2:
        raise AtsError("rope_strided: cos/sin must be float32 2-D tables of equal shape")
    if cos.stride(1) != 1 or sin.stride(1) != 1 or cos.stride(0) != sin.stride(0):
        cos, sin = cos.contiguous(), sin.contiguous()
    check(_lib.load().ats_rope_strided((ctypes.c_void_p * 3)(*src), (ctypes.c_void_p * 3)(*dst), (ctypes.c_int64 * 9)(*ss),
                                       (ctypes.c_int64 * 9)(*ds), cos.data_ptr(), sin.data_ptr(), cos.stride(0), cos.shape[0],
                                       B, (ctypes.c_int * 3)(*heads), L, D, int(position_offset), int(inverse),
                                       _tag(given[0]), _stream()), "ats_rope_strided")


def rope_append(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                k_cache: torch.Tensor, v_cache: torch.Tensor, cache_pos: int,
                position_offset: int = 0) -> torch.Tensor:
    """rope(q, k) with the rotated keys, and the values beside them, written into the cache buffers
    k_cache / v_cache [B, Hkv, capacity, D] at positions cache_pos .. cache_pos + L - 1 (one launch instead of the
    rotation and two strided copies).  Returns the rotated q as a new contiguous tensor."""
    done = _lib.native().rope_append(q, k, v, cos, sin, k_cache, v_cache, cache_pos, position_offset)
    if done is not None:
        return done
    _need_gpu(q, k, v, cos, sin, k_cache, v_cache)
    if q.dim() != 4 or k.dim() != 4 or v.shape != k.shape or k_cache.dim() != 4 or v_cache.shape != k_cache.shape:
        raise AtsError("rope_append: q, k, v [batch, heads, seq, head_dim] and two caches of one shape")
    B, Hq, L, D = q.shape
    Hkv = k.shape[1]
    if (k.shape[0] != B or k.shape[2] != L or k.shape[3] != D or k.dtype != q.dtype or v.dtype != q.dtype
            or k_cache.dtype != q.dtype or v_cache.dtype != q.dtype or k_cache.shape[0] != B
            or k_cache.shape[1] != Hkv or k_cache.shape[3] != D or k_cache.stride() != v_cache.stride()
            or k_cache.stride(3) != 1):
        raise AtsError(f"rope_append: k/v {tuple(k.shape)}, caches {tuple(k_cache.shape)} do not match q {tuple(q.shape)}")
    if cos.dtype != torch.float32 or sin.dtype != torch.float32 or cos.shape != sin.shape or cos.dim() != 2:
        raise AtsError("rope_append: cos/sin must be float32 2-D tables of equal shape")
    if cos.stride(1) != 1 or sin.stride(1) != 1 or cos.stride(0) != sin.stride(0):
        cos, sin = cos.contiguous(), sin.contiguous()
    q, qsb, qsh, qsl = _bhl_strides(q)
    k, ksb, ksh, ksl = _bhl_strides(k)
    v, vsb, vsh, vsl = _bhl_strides(v)
    q_out = torch.empty((B, Hq, L, D), dtype=q.dtype, device=q.device)
    check(_lib.load().ats_rope_fwd_append(q.data_ptr(), k.data_ptr(), v.data_ptr(), q_out.data_ptr(),
                                          k_cache.data_ptr(), v_cache.data_ptr(), cos.data_ptr(), sin.data_ptr(),
                                          cos.stride(0), cos.shape[0], B, Hq, Hkv, L, D, int(position_offset),
                                          qsb, qsh, qsl, ksb, ksh, ksl, vsb, vsh, vsl, k_cache.stride(0),
                                          k_cache.stride(1), k_cache.stride(2), int(cache_pos), k_cache.shape[2],
                                          _tag(q), _stream()), "ats_rope_fwd_append")
    return q_out


# --------------------------------------------------------------------------- router
def router_logits(x: torch.Tensor, gate_weight: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x [T,H], gate_weight [E,H] (same dtype) -> float32 logits [T,E]."""
    _need_gpu(x, gate_weight, bias)
    if x.dim() != 2 or gate_weight.dim() != 2 or x.shape[1] != gate_weight.shape[1] or x.dtype != gate_weight.dtype:
        raise AtsError(f"router_logits: x {tuple(x.shape)}/{x.dtype} vs weight {tuple(gate_weight.shape)}/{gate_weight.dtype}")
    T, H = x.shape
    E = gate_weight.shape[0]
    x, gate_weight = x.contiguous(), gate_weight.contiguous()
    if bias is not None:
        if bias.numel() != E:
            raise AtsError("router_logits: bias must have one entry per expert")
        bias = bias.to(torch.float32).contiguous()
    logits = torch.empty(T, E, dtype=torch.float32, device=x.device)
    check(_lib.load().ats_router_logits(x.data_ptr(), gate_weight.data_ptr(), _ptr(bias), logits.data_ptr(), T, H, E,
                                        _tag(x), _stream()), "ats_router_logits")
    return logits


def route_topk(logits: torch.Tensor, k: int, temperature: float = 1.0, variant: int = ROUTE_SOFTMAX_TOPK,
               load_balancing_weight: float = 0.01, with_stats: bool = True):
    """float32 logits [T,E] -> dict(indices int32 [T,k], weights f32 [T,k], hist int32 [E],
    prob_colsum f32 [E], aux f32 [1])."""
    _need_gpu(logits)
    if logits.dim() != 2 or logits.dtype != torch.float32:
        raise AtsError("route_topk: logits must be a float32 [tokens, experts] tensor")
    logits = logits.contiguous()
    T, E = logits.shape
    dev = logits.device
    idx = torch.empty(T, k, dtype=torch.int32, device=dev)
    w = torch.empty(T, k, dtype=torch.float32, device=dev)
    hist = colsum = aux = ws = None
    ws_bytes = 0
    lib = _lib.load()
    if with_stats:
        # one buffer for the three outputs; the finalize kernel writes every element (nothing runs for T == 0)
        stats = (torch.empty if T > 0 else torch.zeros)(2 * E + 1, dtype=torch.int32, device=dev)
        hist = stats[:E]
        colsum = stats[E:2 * E].view(torch.float32)
        aux = stats[2 * E:].view(torch.float32)
        ws_bytes = lib.ats_route_topk_workspace(T, E)
        ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=dev)
    check(lib.ats_route_topk(logits.data_ptr(), T, E, int(k), float(temperature), int(variant), idx.data_ptr(),
                             w.data_ptr(), _ptr(hist), _ptr(colsum), _ptr(aux), float(load_balancing_weight),
                             _ptr(ws), ws_bytes, _stream()), "ats_route_topk")
    return {"indices": idx, "weights": w, "hist": hist, "prob_colsum": colsum, "aux": aux}


def routing_counts(hist: torch.Tensor, kept: torch.Tensor, assignments: int, counts: Optional[torch.Tensor] = None) -> torch.Tensor:
    """float32 [E] share of the assignments that each expert was chosen for; with counts (int64 [E + 1]) hist is added to its
    first E and the number of dropped assignments to its last element."""
    _need_gpu(hist, kept, counts)
    E = hist.numel()
    if hist.dtype != torch.int32 or kept.dtype != torch.int32 or kept.numel() != E:
        raise AtsError("routing_counts: hist and kept must be int32 of one size")
    if counts is not None and (counts.dtype != torch.int64 or counts.numel() != E + 1 or not counts.is_contiguous()):
        raise AtsError("routing_counts: counts must be contiguous int64 [experts + 1]")
    usage = torch.empty(E, dtype=torch.float32, device=hist.device)
    check(_lib.load().ats_routing_counts(hist.contiguous().data_ptr(), kept.contiguous().data_ptr(), E, int(assignments),
                                         usage.data_ptr(), _ptr(counts), _stream()), "ats_routing_counts")
    return usage


def routing_totals(hist: torch.Tensor, kept: torch.Tensor, tokens: int, counts: torch.Tensor) -> None:
    """Adds hist to the first E of counts (int64 [E + 2]), the number of dropped assignments to the next and tokens to the last."""
    _need_gpu(hist, kept, counts)
    E = hist.numel()
    if hist.dtype != torch.int32 or kept.dtype != torch.int32 or kept.numel() != E:
        raise AtsError("routing_totals: hist and kept must be int32 of one size")
    if counts.dtype != torch.int64 or counts.numel() != E + 2 or not counts.is_contiguous():
        raise AtsError("routing_totals: counts must be contiguous int64 [experts + 2]")
    check(_lib.load().ats_routing_totals(hist.contiguous().data_ptr(), kept.contiguous().data_ptr(), E, int(tokens), counts.data_ptr(),
                                         _stream()), "ats_routing_totals")


def aux_loss_clean_logits(clean_logits: torch.Tensor, hist: torch.Tensor, k: int, variant: int,
                          load_balancing_weight: float) -> torch.Tensor:
    """Load-balancing loss when routing ran on noisy logits: usage from the routed histogram, importance from
    the noise-free, un-tempered logits (MS/core/model.py:1190-1192, 1244-1263).  Returns a float32 scalar."""
    T, E = clean_logits.shape
    colsum = route_topk(clean_logits, k, 1.0, variant, load_balancing_weight)["prob_colsum"]
    usage = hist.float() / (T * k + 1e-9)
    return torch.clamp((usage * (colsum / T)).sum() * (E * load_balancing_weight), max=1.0)


# --------------------------------------------------------------------------- dispatch
def expert_capacity(total_tokens: int, top_k: int, num_experts: int, capacity_factor: float) -> int:
    """Host-side integer, in double arithmetic then truncated, exactly as the reference computes it."""
    return int((total_tokens * top_k / num_experts) * capacity_factor)


def dispatch_plan(indices: torch.Tensor, num_experts: int, capacity: int):
    """indices [T,k] int32/int64 -> dict of int32 tensors: slot [T*k], token_map [E,C], hist [E],
    kept [E], offsets [E+1], row_src [min(T*k,E*C)], row_of [T*k], status [1]."""
    _need_gpu(indices)
    if indices.dim() != 2 or indices.dtype not in (torch.int32, torch.int64):
        raise AtsError("dispatch_plan: indices must be an int32/int64 [tokens, k] tensor")
    indices = indices.contiguous()
    T, k = indices.shape
    E, C = int(num_experts), int(capacity)
    dev = indices.device
    i32 = dict(dtype=torch.int32, device=dev)
    n = T * k
    out = {
        "slot": torch.empty(n, **i32), "token_map": torch.empty(E, C, **i32), "hist": torch.empty(E, **i32),
        "kept": torch.empty(E, **i32), "offsets": torch.empty(E + 1, **i32),
        "row_src": torch.empty(max(1, min(n, E * C)), **i32), "row_of": torch.empty(n, **i32),
        "status": torch.empty(1, **i32),
    }
    lib = _lib.load()
    ws_bytes = max(lib.ats_dispatch_plan_workspace(max(T, 1), k, E), 4 * E)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    check(lib.ats_dispatch_plan(indices.data_ptr(), IDX_I64 if indices.dtype == torch.int64 else IDX_I32, T, k, E, C,
                                out["slot"].data_ptr(), out["token_map"].data_ptr(), out["hist"].data_ptr(),
                                out["kept"].data_ptr(), out["offsets"].data_ptr(), out["row_src"].data_ptr(),
                                out["row_of"].data_ptr(), out["status"].data_ptr(), ws.data_ptr(), ws_bytes,
                                _stream()), "ats_dispatch_plan")
    return out


def gather_rows(src: torch.Tensor, row_map: torch.Tensor, div: int = 1) -> torch.Tensor:
    """out[r] = src[row_map[r] // div] (zeros where row_map[r] < 0)."""
    _need_gpu(src, row_map)
    if src.dim() != 2 or row_map.dtype != torch.int32:
        raise AtsError("gather_rows: src must be 2-D and row_map int32")
    src, row_map = src.contiguous(), row_map.contiguous()
    n, H = row_map.numel(), src.shape[1]
    out = torch.empty(n, H, dtype=src.dtype, device=src.device)
    check(_lib.load().ats_gather_rows(src.data_ptr(), row_map.data_ptr(), int(div), out.data_ptr(), n, H, _tag(src),
                                      _stream()), "ats_gather_rows")
    return out


def invert_token_map(token_map: torch.Tensor, n_assign: int) -> torch.Tensor:
    _need_gpu(token_map)
    if token_map.dtype != torch.int32:
        raise AtsError("invert_token_map: token_map must be int32")
    token_map = token_map.contiguous()
    row_of = torch.empty(n_assign, dtype=torch.int32, device=token_map.device)
    check(_lib.load().ats_invert_token_map(token_map.data_ptr(), token_map.numel(), row_of.data_ptr(), n_assign,
                                           _stream()), "ats_invert_token_map")
    return row_of


# --------------------------------------------------------------------------- expert FFN
_pointer_table_cache: dict = {}


def weight_pointer_table(weights: Sequence[torch.Tensor]) -> torch.Tensor:
    """Device array of the experts' weight base addresses (int64)."""
    for w in weights:
        _need_gpu(w)
        if not w.is_contiguous():
            raise AtsError("expert weights must be contiguous")
    # the table holds nothing but the addresses it is keyed by, so an entry can never go stale
    key = (weights[0].device,) + tuple(w.data_ptr() for w in weights)
    table = _pointer_table_cache.get(key)
    if table is None:
        if len(_pointer_table_cache) > 256:
            _pointer_table_cache.clear()
        table = torch.tensor(key[1:], dtype=torch.int64, device=weights[0].device)
        _pointer_table_cache[key] = table
    return table


# kinds of fill_tables (see ats_fill_tables)
TABLE_INDEX, TABLE_KV_OF_HEAD, TABLE_SLOT_OF_HEAD, TABLE_HEAD_OF_SLOT, TABLE_FROM_ARRAY, TABLE_CONSTANT = range(6)


def fill_tables(device: torch.device, specs: Sequence[tuple], heads: Tuple[int, int, int] = (0, 0, 0)) -> list:
    """Device tables base + x(i) * stride from one launch; a spec is (kind, n, base, stride, wide[, index]) and gives an
    int64 (wide) or int32 tensor of n entries; heads = (batch, query heads, key/value heads)."""
    most = max(spec[1] for spec in specs)
    rows = torch.empty(len(specs), most, dtype=torch.int64, device=device)
    at, arr, outs = rows.data_ptr(), (_lib.Table * len(specs))(), []
    for i, (row, (kind, n, base, stride, wide, *index)) in enumerate(zip(rows.unbind(0), specs)):
        if index:
            _need_gpu(index[0])
            if index[0].dtype != torch.int32 or index[0].numel() < n or not index[0].is_contiguous():
                raise AtsError("fill_tables: the index array must be contiguous int32 with one entry per table entry")
        arr[i] = (at + i * most * 8, base, stride, index[0].data_ptr() if index else None, n, kind, wide)
        if not wide:
            row = row.view(torch.int32)
        outs.append(row if row.numel() == n else row[:n])
    check(_lib.load().ats_fill_tables(arr, len(specs), *heads, _stream()), "ats_fill_tables")
    return outs


def address_table(t: torch.Tensor) -> torch.Tensor:
    """The address of one matrix on the device, written by a launch: for a matrix that lives for one call.  (A cached table
    uploads every address that it has not seen, and that copy waits until the queue has drained.)"""
    return upload(array("q", [t.data_ptr()]), t.device)


def stack_weights(ws: Sequence[torch.Tensor]) -> Tuple[torch.Tensor, torch.Tensor]:
    """torch.cat(ws, dim=0) of weights of one type and width, and the address table of the result."""
    w0 = ws[0]
    if len(ws) > 8 or not all(w.is_cuda and w.is_contiguous() and w.dim() == 2 and w.dtype == w0.dtype and w.device == w0.device
                              and w.shape[1] == w0.shape[1] and w.numel() > 0 and w.numel() * w.element_size() % 16 == 0
                              and w.data_ptr() % 16 == 0 for w in ws):
        out = torch.cat(list(ws), dim=0)
        return out, address_table(out)
    n = len(ws)
    out = torch.empty(sum(w.shape[0] for w in ws), w0.shape[1], dtype=w0.dtype, device=w0.device)
    table = torch.empty(1, dtype=torch.int64, device=w0.device)
    check(_lib.load().ats_stack_rows((ctypes.c_void_p * n)(*[w.data_ptr() for w in ws]),
                                     (ctypes.c_int64 * n)(*[w.numel() * w.element_size() for w in ws]), n, out.data_ptr(),
                                     table.data_ptr(), _stream()), "ats_stack_rows")
    return out, table


def upload(words: array, device: torch.device) -> torch.Tensor:
    """An int64 array on the device, sent with launches instead of a copy that waits for the queue."""
    lib, (src, n) = _lib.load(), words.buffer_info()
    buf = torch.empty(n, dtype=torch.int64, device=device)
    step = lib.ats_upload_max_bytes()
    for off in range(0, n * 8, step):
        check(lib.ats_upload(buf.data_ptr() + off, src + off, min(step, n * 8 - off), _stream()), "ats_upload")
    return buf


def wgrad_slices(M: int, N: int, rows: int) -> int:
    """K slices of a weight gradient [M, N] over `rows` bfloat16 rows.  Its 256 x 256 tiles are few (16 of a [1024, 1024]
    gradient) and its K long: slices over workgroups, added in float32, fill the chip.  Least estimated time in microseconds:
    rounds of 256 CUs at 12 per tile and 1.36 per 64-row slab (one slice may also run on lower tiles, 1.08 for 192 and 0.78
    for 128 rows), the partial results written and read at 14 TB/s (they stay in the last-level cache) and 7 for the launch
    that adds them.  Measured, one slice | the rule's | others: 16384 rows [1024, 2048] 205 | 71 (eight) | 111 (four),
    [2048, 2048] 207 | 114 (four) | 139 (three), [2048, 4096] 212 | 202 (two), [4096, 4096] 357 | (two 403);
    4096 rows [1024, 2048] 58 | 40 (eight) | 49 (four), [2048, 2048] 60 | 51 (four), [2048, 4096] 61 | (two 74);
    2048 rows [512, 2048] 30 | 32 (four), [1024, 2048] 34 | (three 38), [2048, 2048] 34 | (two 48, four 41);
    1024 rows [512, 2048] 21 | (two 28)."""
    slabs = -(-rows // 64)
    tiles = lambda height: -(-M // height) * -(-N // 256)
    best, slices = min(-(-tiles(h) // 256) * (slabs * per_slab + 12.0) for h, per_slab in ((256, 1.36), (192, 1.08), (128, 0.78))), 1
    for s in range(2, min(16, slabs // 8) + 1):
        t = -(-tiles(256) * s // 256) * (-(-slabs // s) * 1.36 + 12.0) + s * M * N * 8 / 14e6 + 7.0
        if t < best - max(2.5, 0.03 * best):      # (below that the estimates do not tell them apart)
            best, slices = t, s
    return slices


def wgrad_dense(lhsT: torch.Tensor, rhsT: torch.Tensor, rows: int, heights: Optional[Sequence[int]] = None):
    """lhsT @ rhsT^T over the first `rows` columns (zero padded to a multiple of 64) of two contiguous transposed operands
    [M, ld], [N, ld]: the weight gradient of a linear layer.  heights (which add up to M): the gradients of stacked layers,
    a list of tensors with memory of their own."""
    _need_gpu(lhsT, rhsT)
    (M, ld), N, es, dtype = lhsT.shape, rhsT.shape[0], lhsT.element_size(), lhsT.dtype
    slices = wgrad_slices(M, N, rows) if dtype == torch.bfloat16 and (M * N) % 8 == 0 else 1
    slabs = max(1, -(-rows // 64))
    per = -(-slabs // slices)
    slices = -(-slabs // per)
    tab = array("q", [lhsT.data_ptr() + i * per * 64 * es for i in range(slices)] +
                [rhsT.data_ptr() + i * per * 64 * es for i in range(slices)])
    rc = [i * M for i in range(slices)] + [M] * slices + [min(per, slabs - i * per) * 64 for i in range(slices)]
    tab.frombytes(array("i", rc + [0] * (len(rc) % 2)).tobytes())
    buf = upload(tab, lhsT.device)
    r32 = buf[2 * slices:].view(torch.int32)
    parts = grouped_gemm_nt(buf[slices:2 * slices], ld, N, r32[:slices], r32[slices:2 * slices], slices * M, slices * M, N, ld,
                            a_ptrs=buf[:slices], lda=ld, k_count=r32[2 * slices:3 * slices], dtype=dtype,
                            out_dtype=dtype if slices == 1 else torch.float32)
    return _wgrad_result(parts, slices, M, N, dtype, heights)


def _wgrad_result(parts: torch.Tensor, slices: int, M: int, N: int, dtype: torch.dtype, heights: Optional[Sequence[int]]):
    if heights is None:
        return parts if slices == 1 else sum_partials(parts.view(slices, M * N), dtype).view(M, N)
    if slices == 1:
        return [part.clone() for part in parts.split(list(heights))]
    return [sum_partials(part, dtype) for part in parts.view(slices, M, N).split(list(heights), dim=1)]


def wgrad_linear_supported(dy: torch.Tensor, x: torch.Tensor) -> bool:
    """Whether wgrad_linear takes these operands: bfloat16, 16-byte aligned rows within 4 GiB."""
    return dy.dtype == torch.bfloat16 and x.dtype == dy.dtype and all(
        t.dim() == 2 and t.shape[0] > 0 and t.shape[1] > 0 and t.shape[1] % 8 == 0 and t.stride(1) == 1
        and t.stride(0) >= t.shape[1] and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0
        and (t.shape[0] + 63) * t.stride(0) * 2 < 1 << 32 for t in (dy, x))


def wgrad_linear(dy: torch.Tensor, x: torch.Tensor, heights: Optional[Sequence[int]] = None):
    """dy^T @ x for dy [T, M] and x [T, N] with rows of any stride, as they lie: the weight gradient of a linear layer; the
    bits of wgrad_dense on transposed copies, and its heights."""
    _need_gpu(dy, x)
    if not wgrad_linear_supported(dy, x) or dy.shape[0] != x.shape[0]:
        raise AtsError("wgrad_linear: bfloat16 [T, M], [T, N] of 16-byte aligned rows within 4 GiB")
    (T, M), N, dtype = dy.shape, x.shape[1], dy.dtype
    slabs = -(-T // 64)
    slices = -(-slabs // -(-slabs // wgrad_slices(M, N, T)))
    start, count = _single_group(M, x.device)
    parts = torch.empty(slices * M, N, dtype=dtype if slices == 1 else torch.float32, device=x.device)
    check(_lib.load().ats_wgrad_tn(dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), parts.data_ptr(), T, M, N, slices,
                                   start.data_ptr(), count.data_ptr(), _DT[dtype], _DT[parts.dtype], _stream()), "ats_wgrad_tn")
    return _wgrad_result(parts, slices, M, N, dtype, heights)


def wgrad_tables(k_start: torch.Tensor, M: int, lhsT: torch.Tensor, rhsT: torch.Tensor) -> list:
    """(a_ptrs, b_ptrs, row_start, row_count) of the weight-gradient product of [*, padded] transposed operands: group e
    contracts over the columns from k_start[e] and writes rows e * M .. + M."""
    E, es = k_start.numel(), lhsT.element_size()
    return fill_tables(k_start.device, [(TABLE_FROM_ARRAY, E, lhsT.data_ptr(), es, True, k_start),
                                        (TABLE_FROM_ARRAY, E, rhsT.data_ptr(), es, True, k_start),
                                        (TABLE_INDEX, E, 0, M, False), (TABLE_CONSTANT, E, M, 0, False)])


def grouped_gateup_swiglu(a: torch.Tensor, w_gu_ptrs: torch.Tensor, row_start: torch.Tensor, row_count: torch.Tensor,
                          n_rows_out: int, max_rows: int, H: int, I: int, a_rows: Optional[torch.Tensor] = None,
                          a_row_div: int = 1) -> torch.Tensor:
    _need_gpu(a, w_gu_ptrs, row_start, row_count, a_rows)
    if a.dim() != 2 or a.shape[1] != H or not a.is_contiguous():
        raise AtsError("grouped_gateup_swiglu: activations must be a contiguous [rows, H] tensor")
    E = w_gu_ptrs.numel()
    if row_start.numel() < E or row_count.numel() < E or row_start.dtype != torch.int32 or row_count.dtype != torch.int32:
        raise AtsError("grouped_gateup_swiglu: row_start/row_count must be int32 with one entry per expert")
    h = torch.empty(n_rows_out, I, dtype=a.dtype, device=a.device)
    check(_lib.load().ats_grouped_gateup_swiglu(a.data_ptr(), int(a.shape[0]), _ptr(a_rows), int(a_row_div), w_gu_ptrs.data_ptr(),
                                                h.data_ptr(), row_start.data_ptr(), row_count.data_ptr(), E,
                                                int(max_rows), H, I, _tag(a), _stream()), "ats_grouped_gateup_swiglu")
    return h


def grouped_gateup_swiglu_save(a: torch.Tensor, w_gu_ptrs: torch.Tensor, row_start: torch.Tensor,
                               row_count: torch.Tensor, n_rows_out: int, max_rows: int, H: int, I: int,
                               a_rows: Optional[torch.Tensor] = None, a_row_div: int = 1,
                               t_col0: Optional[torch.Tensor] = None
                               ) -> Optional[Tuple[torch.Tensor, torch.Tensor, Optional[torch.Tensor]]]:
    """Training forward of the gate/up projection: (gu [rows, 2I], h [rows, I], hT) from one kernel, or None when
    the sizes are not prefill-sized (the caller then runs the plain product and silu_mul).  hT is None unless
    t_col0 (the k_start of wgrad_plan) is given and the dtype is bfloat16: then it is h transposed into the
    weight-gradient layout [I, wgrad_padded_rows] (see transpose_grouped_rows), written by the same kernel."""
    _need_gpu(a, w_gu_ptrs, row_start, row_count, a_rows)
    if a.dim() != 2 or a.shape[1] != H or not a.is_contiguous():
        raise AtsError("grouped_gateup_swiglu_save: activations must be a contiguous [rows, H] tensor")
    E = w_gu_ptrs.numel()
    if row_start.numel() < E or row_count.numel() < E or row_start.dtype != torch.int32 or row_count.dtype != torch.int32:
        raise AtsError("grouped_gateup_swiglu_save: row_start/row_count must be int32 with one entry per expert")
    lib = _lib.load()
    if not lib.ats_grouped_gateup_swiglu_save_supported(int(a.shape[0]), E, int(max_rows), H, I, _tag(a)):
        return None
    h = torch.empty(n_rows_out, I, dtype=a.dtype, device=a.device)
    gu = torch.empty(n_rows_out, 2 * I, dtype=a.dtype, device=a.device)
    hT, ld = _transposed_copy_buffer(I, row_count, t_col0, max_rows, E, a.dtype, a.device)
    check(lib.ats_grouped_gateup_swiglu_save(a.data_ptr(), int(a.shape[0]), _ptr(a_rows), int(a_row_div),
                                             w_gu_ptrs.data_ptr(), h.data_ptr(), gu.data_ptr(), row_start.data_ptr(),
                                             row_count.data_ptr(), E, int(max_rows), H, I, _tag(a), _ptr(hT), ld,
                                             _ptr(t_col0) if hT is not None else None, _stream()),
          "ats_grouped_gateup_swiglu_save")
    return gu, h, hT


def _transposed_copy_buffer(C: int, row_count: torch.Tensor, t_col0: Optional[torch.Tensor], max_rows: int, E: int,
                            dtype: torch.dtype, device) -> Tuple[Optional[torch.Tensor], int]:
    """The [C, padded rows] buffer that a training launch fills with the transposed copy of its result (bfloat16
    launches with the experts' first columns given), the columns of experts without rows already cleared."""
    if t_col0 is None or dtype != torch.bfloat16:
        return None, 0
    _need_gpu(t_col0)
    if t_col0.dtype != torch.int32 or t_col0.numel() < E:
        raise AtsError("transposed copy: t_col0 must be int32 with one entry per expert")
    ld = wgrad_padded_rows(max_rows, E)
    out = torch.empty(C, ld, dtype=dtype, device=device)
    check(_lib.load().ats_transposed_zero_empty_groups(out.data_ptr(), ld, C, row_count.data_ptr(), t_col0.data_ptr(), E,
                                                       _tag(out), _stream()), "ats_transposed_zero_empty_groups")
    return out, ld


def grouped_down_dgrad_dsilu_supported(E: int, max_rows: int, H: int, I: int, dtype: torch.dtype,
                                       transposed_weights: bool = True) -> bool:
    """Whether grouped_down_dgrad_dsilu has a kernel for these sizes (with the transposed, or the forward's own, weights)."""
    lib = _lib.load()
    fn = lib.ats_grouped_down_dgrad_dsilu_supported if transposed_weights else lib.ats_grouped_down_dgrad_dsilu_nn_supported
    return bool(fn(int(E), int(max_rows), int(H), int(I), _DT[dtype]))


def grouped_down_dgrad_dsilu(dy: torch.Tensor, w_dT_ptrs: torch.Tensor, gu: torch.Tensor, row_start: torch.Tensor,
                             row_count: torch.Tensor, max_rows: int, H: int, I: int,
                             t_col0: Optional[torch.Tensor] = None, transposed_weights: bool = True
                             ) -> Optional[Tuple[torch.Tensor, Optional[torch.Tensor]]]:
    """Training backward of the down projection and of silu(g) * u in one kernel: (dgu [rows, 2I], dguT) from
    dy [rows, H], the transposed down weights ([I, H] per expert) and the saved gu; None when the groups are not
    prefill-sized (the caller then runs the plain product and silu_mul_bwd).  dguT is None unless t_col0 (the
    k_start of wgrad_plan) is given and the dtype is bfloat16: then it is dgu transposed into the weight-gradient
    layout [2I, wgrad_padded_rows], written by the same kernel.  transposed_weights=False: the pointer table holds
    the forward's own down weights ([H, I] per expert; bfloat16, ats_grouped_down_dgrad_dsilu_nn)."""
    _need_gpu(dy, w_dT_ptrs, gu, row_start, row_count)
    if dy.dim() != 2 or dy.shape[1] != H or not dy.is_contiguous():
        raise AtsError("grouped_down_dgrad_dsilu: dy must be a contiguous [rows, H] tensor")
    if gu.dim() != 2 or gu.shape[1] != 2 * I or not gu.is_contiguous() or gu.dtype != dy.dtype or gu.shape[0] < dy.shape[0]:
        raise AtsError("grouped_down_dgrad_dsilu: gu must be a contiguous [rows, 2I] tensor of dy's dtype")
    E = w_dT_ptrs.numel()
    if row_start.numel() < E or row_count.numel() < E or row_start.dtype != torch.int32 or row_count.dtype != torch.int32:
        raise AtsError("grouped_down_dgrad_dsilu: row_start/row_count must be int32 with one entry per expert")
    lib = _lib.load()
    if not grouped_down_dgrad_dsilu_supported(E, max_rows, H, I, dy.dtype, transposed_weights):
        return None
    dgu = torch.empty_like(gu)
    dguT, ld = _transposed_copy_buffer(2 * I, row_count, t_col0, max_rows, E, dy.dtype, dy.device)
    fn = lib.ats_grouped_down_dgrad_dsilu if transposed_weights else lib.ats_grouped_down_dgrad_dsilu_nn
    check(fn(dy.data_ptr(), w_dT_ptrs.data_ptr(), gu.data_ptr(), dgu.data_ptr(), row_start.data_ptr(),
             row_count.data_ptr(), E, int(max_rows), H, I, _tag(dy), _ptr(dguT), ld,
             _ptr(t_col0) if dguT is not None else None, _stream()),
          "ats_grouped_down_dgrad_dsilu" if transposed_weights else "ats_grouped_down_dgrad_dsilu_nn")
    return dgu, dguT


def grouped_down(h: torch.Tensor, w_d_ptrs: torch.Tensor, row_start: torch.Tensor, row_count: torch.Tensor,
                 max_rows: int, H: int, I: int, out: Optional[torch.Tensor] = None,
                 out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    _need_gpu(h, w_d_ptrs, row_start, row_count, out)
    if h.dim() != 2 or h.shape[1] != I or not h.is_contiguous():
        raise AtsError("grouped_down: h must be a contiguous [rows, I] tensor")
    E = w_d_ptrs.numel()
    if out is None:
        out = torch.empty(h.shape[0], H, dtype=out_dtype or h.dtype, device=h.device)
    check(_lib.load().ats_grouped_down(h.data_ptr(), w_d_ptrs.data_ptr(), out.data_ptr(), row_start.data_ptr(),
                                       row_count.data_ptr(), E, int(max_rows), H, I, _tag(h), _tag(out), _stream()),
          "ats_grouped_down")
    return out


def down_k_splits(E: int, max_rows: int, N: int, K: int, dtype: torch.dtype) -> int:
    """Slices of K for a projection with few rows per expert.  Such a product streams its weights, and
    it takes several hundred workgroups to keep the memory system busy; the plain tilings give
    E * ceil(N / 128) of them up to 32 rows per expert and E * ceil(rows / 128) * ceil(N / 256) above.
    When that is under 384, 32-row tiles (64-row tiles above 32 rows) with K cut into slices are used
    instead, if two or more slices are needed to fill the chip (measured on MI355X: 8 x [4096, 14336]
    weights x 16 rows 199 -> 160 us with 2 slices; one [4096, 4096] weight x 64 rows 50 -> 10 us with 8,
    x 256 rows 51 -> 23 us with 2; [4096, 14336] x 64 rows 156 -> 22 us with 8).
    Powers of two up to 16, slices of at least 512 columns, at most 256 rows per expert.

    bfloat16 experts of more than 20 rows against 32 MB of weights or more: those slices or the plain launch, slices on the band tiles
    (up to 72 rows on average, 100 with many experts) or on the direct-to-LDS tile (up to 256 rows x 256 columns, one per CU), whichever
    is estimated to take the least time (ats_down_k_slices).  Measured with the combine behind it, weights from HBM, rows per expert
    24 | 32 | 48 | 64 | 72 | 96 | 128 | 192 | 224, plain -> in the slices that are chosen, microseconds:
      8 x [4096, 14336]  160 -> 159 | 161 -> 164 | 164 | 173 -> 170 | 179 -> 172 | 267 -> 169 | 262 -> 169 | 264 -> 191 | 331 -> 222
      4 x [4096, 14336]  97 -> 90 | 104 -> 90 | 97 -> 85 | 126 -> 90 | 184 -> 92 | 227 -> 94 | 191 -> 102 | 239 -> 141 | 279 -> 178
      2 x [4096, 14336]  60 -> 47 | 67 -> 48 | 72 -> 50 | 99 -> 53 | 106 -> 53 | 116 -> 64
      16 x [2048, 8192]  102 -> 105 | 101 -> 102 | 107 -> 106 | 109 -> 111 | 110 -> 112 | 168 -> 142 | 162 -> 133 | 162 -> 141 | 198 -> 156
      16 x [2048, 5632]  66 -> 68 | 69 -> 71 | 73 -> 76 | 75 -> 78 | 77 -> 83 | 121 -> 81 | 147 -> 83 | 117 -> 110 | 143 -> 115
      8 x [2048, 5632]   43 -> 39 | 49 -> 39 | 46 -> 40 | 64 -> 43 | 64 -> 44 | 64 -> 52 | 88 -> 53 | 100 -> 72 | 132 -> 76
      4 x [1024, 8192]   32 -> 23 | 37 -> 24 | 35 -> 26 | 37 -> 27 | 38 -> 27 | 38 -> 36 | 44 -> 38 | 61 -> 47 | 135 -> 44
      8 x [1024, 4096]   24 -> 21 | 25 -> 21 | 25 -> 23 | 31 -> 23 | 31 -> 25 | 31 | 40 | 43 | 85 -> 50
      64 x [2048, 1408]  plain everywhere
    (all with equal chances for every expert; slices that gain nothing with these gain a fifth where sizes fall as rank^-1.5).  385
    points, 2-64 experts of 21-100 rows: 1.4 % slower than the fastest of all routes on average.
    Below 32 MB of weights everything comes from the last-level cache and the first rule stands."""
    slab = 64 if dtype == torch.bfloat16 else 32
    if E <= 0 or max_rows <= 0:
        return 1
    rows = -(-max_rows // E)
    if rows > 256:
        return 1
    if E > 1 and max_rows // E <= 20:
        return 1        # the plain launch streams the weights itself (8 x [4096, 14336], 16 rows each: 157 against 159 us)
    n128 = (N + 127) // 128
    plain = E * n128 if max_rows // E <= 32 else E * ((rows + 127) // 128) * ((N + 255) // 256)
    s = 1
    if plain < 384:
        # 32-row tiles (three workgroups per CU) up to 32 rows, 64-row tiles (two per CU) above
        groups = E * (1 if rows <= 32 else (rows + 63) // 64) * n128
        enough = 384 if rows <= 32 else 256
        while s < 16 and groups * s < enough and K % (2 * s * slab) == 0 and K // (2 * s) >= 512:
            s *= 2
    if E > 1 and dtype == torch.bfloat16 and E * N * K >= 1 << 24:
        return int(_lib.load().ats_down_k_slices(int(E), int(max_rows), int(N), int(K), s))
    return s


def grouped_down_splitk(h: torch.Tensor, w_d_ptrs: torch.Tensor, row_start: torch.Tensor, row_count: torch.Tensor,
                        max_rows: int, H: int, I: int, k_splits: int) -> torch.Tensor:
    """Float32 partial results [k_splits, rows, H] of grouped_down with K cut into k_splits slices
    (decode sizes only); sum_partials or combine_partials add them up."""
    _need_gpu(h, w_d_ptrs, row_start, row_count)
    if h.dim() != 2 or h.shape[1] != I or not h.is_contiguous():
        raise AtsError("grouped_down_splitk: h must be a contiguous [rows, I] tensor")
    E = w_d_ptrs.numel()
    parts = torch.empty(k_splits, h.shape[0], H, dtype=torch.float32, device=h.device)
    check(_lib.load().ats_grouped_down_splitk(h.data_ptr(), w_d_ptrs.data_ptr(), parts.data_ptr(), row_start.data_ptr(),
                                              row_count.data_ptr(), E, int(max_rows), h.shape[0], H, I, int(k_splits),
                                              _tag(h), _stream()), "ats_grouped_down_splitk")
    return parts


def sum_partials(parts: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """parts float32 [S, ...] (contiguous slices, any distance apart) -> their sum over S in slice order, rounded once to
    out_dtype."""
    _need_gpu(parts)
    if parts.dtype != torch.float32 or parts.dim() < 2 or parts.shape[0] < 1 or not parts[0].is_contiguous():
        raise AtsError("sum_partials: parts must be float32 [slices, ...] of contiguous slices")
    out = torch.empty(parts.shape[1:], dtype=out_dtype, device=parts.device)
    step = parts.stride(0) if parts.shape[0] > 1 else out.numel()
    check(_lib.load().ats_sum_partials(parts.data_ptr(), parts.shape[0], step, out.data_ptr(), out.numel(), _tag(out), _stream()),
          "ats_sum_partials")
    return out


# --------------------------------------------------------------------------- combine
def gather_sum(y: torch.Tensor, row_of: torch.Tensor, num_tokens: int, k: int, out_dtype: torch.dtype) -> torch.Tensor:
    """combine with every weight 1: y [rows, H], or float32 partial results [slices, rows, H] as in combine_partials
    (k <= 8, H % 8 == 0)."""
    _need_gpu(y, row_of)
    if row_of.dtype != torch.int32 or row_of.numel() != num_tokens * k or y.dim() not in (2, 3):
        raise AtsError("gather_sum: y [rows, H] or [slices, rows, H], row_of int32 with tokens*k entries")
    if y.dim() == 3 and (y.dtype != torch.float32 or not y.is_contiguous()):
        raise AtsError("gather_sum: partial results must be a contiguous float32 [slices, rows, H] tensor")
    H = y.shape[-1]
    out = torch.empty(num_tokens, H, dtype=out_dtype, device=y.device)
    row_of = row_of.contiguous()
    if y.dim() == 3:
        check(_lib.load().ats_gather_sum_partials(y.data_ptr(), y.shape[0], y.shape[1] * H, row_of.data_ptr(), out.data_ptr(), num_tokens,
                                                  int(k), H, _tag(out), _stream()), "ats_gather_sum_partials")
    else:
        y = y.contiguous()
        check(_lib.load().ats_gather_sum(y.data_ptr(), row_of.data_ptr(), out.data_ptr(), num_tokens, int(k), H, _tag(y), _tag(out),
                                         _stream()), "ats_gather_sum")
    return out


def combine(y: torch.Tensor, row_of: torch.Tensor, weights: torch.Tensor, num_tokens: int, k: int,
            out_dtype: Optional[torch.dtype] = None, residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """y [rows, H] (any leading shape); row_of int32 [T*k]; weights f32 [T,k] -> out [T,H]."""
    _need_gpu(y, row_of, weights, residual)
    if row_of.dtype != torch.int32 or weights.dtype != torch.float32:
        raise AtsError("combine: row_of must be int32 and weights float32")
    if row_of.numel() != num_tokens * k or weights.numel() != num_tokens * k:
        raise AtsError("combine: row_of/weights must have tokens*k entries")
    y2 = y.reshape(-1, y.shape[-1]).contiguous()
    H = y2.shape[1]
    out = torch.empty(num_tokens, H, dtype=out_dtype or y.dtype, device=y.device)
    if residual is not None:
        residual = residual.reshape(num_tokens, H).contiguous()
        if residual.dtype != out.dtype:
            raise AtsError("combine: residual must have the output dtype")
    check(_lib.load().ats_combine(y2.data_ptr(), row_of.contiguous().data_ptr(), weights.contiguous().data_ptr(),
                                  _ptr(residual), out.data_ptr(), num_tokens, int(k), H, _tag(y2), _tag(out),
                                  _stream()), "ats_combine")
    return out


def combine_scatter_add(y: torch.Tensor, row_of: torch.Tensor, weights: torch.Tensor, num_tokens: int, k: int,
                        out: torch.Tensor, out_rows: torch.Tensor) -> bool:
    """combine whose result is added onto rows out_rows[t] (int32, distinct, negative = skip) of `out` [N, H] in
    place, with the bits of combine followed by scatter_add_rows.  Returns False (nothing done) when the sizes
    are outside the vector kernel (k > 8, H not a multiple of 8, unaligned views)."""
    _need_gpu(y, row_of, weights, out, out_rows)
    if row_of.dtype != torch.int32 or weights.dtype != torch.float32 or out_rows.dtype != torch.int32:
        raise AtsError("combine_scatter_add: row_of / out_rows must be int32 and weights float32")
    if row_of.numel() != num_tokens * k or weights.numel() != num_tokens * k or out_rows.numel() != num_tokens:
        raise AtsError("combine_scatter_add: row_of/weights must have tokens*k entries, out_rows one per token")
    y2 = y.reshape(-1, y.shape[-1]).contiguous()
    H = y2.shape[1]
    if out.dim() != 2 or out.shape[1] != H or not out.is_contiguous():
        raise AtsError("combine_scatter_add: out must be a contiguous [rows, H] tensor")
    if k > 8 or H % 8 or y2.data_ptr() % 16 or out.data_ptr() % 16:
        return False
    check(_lib.load().ats_combine_scatter_add(y2.data_ptr(), row_of.contiguous().data_ptr(),
                                              weights.contiguous().data_ptr(), out_rows.contiguous().data_ptr(),
                                              out.data_ptr(), num_tokens, int(k), H, _tag(y2), _tag(out), _stream()),
          "ats_combine_scatter_add")
    return True


def combine_partials(parts: torch.Tensor, row_of: torch.Tensor, weights: torch.Tensor, num_tokens: int, k: int,
                     out_dtype: torch.dtype, residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """combine over the float32 partial results [S, rows, H] of grouped_down_splitk: an expert row is their
    sum in slice order, rounded to out_dtype like the unsplit projection's result, before the weighting."""
    _need_gpu(parts, row_of, weights, residual)
    if row_of.dtype != torch.int32 or weights.dtype != torch.float32:
        raise AtsError("combine_partials: row_of must be int32 and weights float32")
    if row_of.numel() != num_tokens * k or weights.numel() != num_tokens * k:
        raise AtsError("combine_partials: row_of/weights must have tokens*k entries")
    if parts.dim() != 3 or parts.dtype != torch.float32 or not parts.is_contiguous():
        raise AtsError("combine_partials: partial results must be a contiguous float32 [slices, rows, H] tensor")
    S, rows, H = parts.shape
    out = torch.empty(num_tokens, H, dtype=out_dtype, device=parts.device)
    if residual is not None:
        residual = residual.reshape(num_tokens, H).contiguous()
        if residual.dtype != out.dtype:
            raise AtsError("combine_partials: residual must have the output dtype")
    check(_lib.load().ats_combine_partials(parts.data_ptr(), S, rows * H, row_of.contiguous().data_ptr(),
                                           weights.contiguous().data_ptr(), _ptr(residual), out.data_ptr(),
                                           num_tokens, int(k), H, _tag(out), _stream()), "ats_combine_partials")
    return out


# --------------------------------------------------------------------------- the MoE layer as one call
_MOE_FIELDS = ("logits", "indices", "weights", "routed", "prob_colsum", "slot", "token_map", "hist", "kept", "offsets",
               "row_src", "row_of", "status")
_moe_layouts: dict = {}        # sizes -> byte offsets (numbers only), as the native call takes them and as a tuple


def _moe_layout(T: int, H: int, I: int, E: int, k: int, C: int, k_splits: int, tag: int):
    key = (T, H, I, E, k, C, k_splits, tag)
    layout = _moe_layouts.get(key)
    if layout is None:
        layout = (ctypes.c_int64 * 19)()
        check(_lib.load().ats_moe_forward_layout(*key, layout), "ats_moe_forward_layout")
        if len(_moe_layouts) >= 256:
            _moe_layouts.clear()
        layout = _moe_layouts[key] = (layout, tuple(layout))
    return layout


def moe_forward(x: torch.Tensor, gate: torch.Tensor, gate_bias: Optional[torch.Tensor], w_gu_ptrs: torch.Tensor,
                w_d_ptrs: torch.Tensor, I: int, k: int, C: int, temperature: float, variant: int,
                load_balancing_weight: float, target: Optional[torch.Tensor] = None,
                target_rows: Optional[torch.Tensor] = None):
    """The layer's inference stages (router .. combine) queued by one native call: x [T, H], gate [E, H] of x's dtype,
    pointer tables over the expert weights.  Returns (out [T, H], aux float32 scalar, plan); with target / target_rows the
    result is added onto those rows of target, which is returned as out.  moe_plan_views(plan) names the routing tensors."""
    _need_gpu(x, gate, gate_bias, w_gu_ptrs, w_d_ptrs, target, target_rows)
    T, H = x.shape
    E = gate.shape[0]
    dev, dtype, tag = x.device, x.dtype, _tag(x)
    if gate.shape[1] != H or gate.dtype != dtype or w_gu_ptrs.numel() != E or w_d_ptrs.numel() != E:
        raise AtsError(f"moe_forward: x {tuple(x.shape)}/{dtype}, gate {tuple(gate.shape)}/{gate.dtype}, {w_gu_ptrs.numel()} experts")
    if not (x.is_contiguous() and gate.is_contiguous()):
        raise AtsError("moe_forward: x and the gate weight must be contiguous")
    if gate_bias is not None:
        if gate_bias.numel() != E:
            raise AtsError("moe_forward: bias must have one entry per expert")
        gate_bias = gate_bias.to(torch.float32).contiguous()
    splits = 1
    if target is None:
        if k <= 8 and H % 8 == 0:
            splits = down_k_splits(E, min(T * k, E * C), H, I, dtype)
        out = torch.empty(T, H, dtype=dtype, device=dev)
    else:
        out = target
    native, layout = _moe_layout(T, H, I, E, k, C, splits, tag)
    plan = torch.empty(layout[15], dtype=torch.uint8, device=dev)
    scratch = torch.empty(layout[17], dtype=torch.uint8, device=dev)
    aux = torch.empty((), dtype=torch.float32, device=dev)
    check(_lib.load().ats_moe_forward(x.data_ptr(), gate.data_ptr(), _ptr(gate_bias), w_gu_ptrs.data_ptr(),
                                      w_d_ptrs.data_ptr(), out.data_ptr(), _ptr(target_rows), aux.data_ptr(),
                                      plan.data_ptr(), scratch.data_ptr(), native, T, H, I, E, k, C, splits,
                                      float(temperature), variant, float(load_balancing_weight), tag, _stream()),
          "ats_moe_forward")
    return out, aux, (plan, layout, T, E, k, C)        # (tensors and integers: a layer that keeps it can be pickled)


def moe_plan_views(handle) -> dict:
    """The routing tensors of a moe_forward call, as route_topk and dispatch_plan return them."""
    plan, layout, T, E, k, C = handle
    n = T * k
    shapes = {"logits": (T, E), "indices": (T, k), "weights": (T, k), "routed": (E,), "prob_colsum": (E,), "slot": (n,),
              "token_map": (E, C), "hist": (E,), "kept": (E,), "offsets": (E + 1,), "row_src": (min(n, E * C),),
              "row_of": (n,), "status": (1,)}
    out = {}
    for i, name in enumerate(_MOE_FIELDS):
        count = 1
        for d in shapes[name]:
            count *= d
        dt = torch.float32 if name in ("logits", "weights", "prob_colsum") else torch.int32
        out[name] = plan[layout[i]:layout[i] + 4 * count].view(dt).view(shapes[name])
    del out["routed"]          # the same counts as hist
    return out


# --------------------------------------------------------------------------- MoD helpers
def row_dot(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None, temperature: float = 1.0,
            want_prob: bool = False, want_copy: bool = False):
    """score[t] = x[t,:] . w (+ bias); optionally sigmoid(score / temperature).  want_copy: the same pass also
    writes a copy of the rows ([T, H], returned last), the start of a residual output."""
    _need_gpu(x, w, bias)
    x2 = x.reshape(-1, x.shape[-1]).contiguous()
    T, H = x2.shape
    w = w.reshape(-1).contiguous()
    if w.numel() != H or w.dtype != x2.dtype:
        raise AtsError("row_dot: weight must have H elements of x's dtype")
    if bias is not None:
        bias = bias.reshape(-1).to(torch.float32).contiguous()
    score = torch.empty(T, dtype=torch.float32, device=x.device)
    prob = torch.empty(T, dtype=torch.float32, device=x.device) if want_prob else None
    copy = torch.empty_like(x2) if want_copy else None
    check(_lib.load().ats_row_dot_copy(x2.data_ptr(), w.data_ptr(), _ptr(bias), score.data_ptr(), _ptr(prob),
                                       float(temperature), _ptr(copy), T, H, _tag(x2), _stream()), "ats_row_dot_copy")
    res = (score, prob) if want_prob else (score,)
    if want_copy:
        res = res + (copy,)
    return res if len(res) > 1 else res[0]


def select_topk_per_sequence(scores: torch.Tensor, keep: int) -> torch.Tensor:
    """scores f32 [B,L] -> flat token ids (b*L+pos) of the `keep` best per sequence, ascending, int32 [B*keep]."""
    _need_gpu(scores)
    if scores.dim() != 2 or scores.dtype != torch.float32:
        raise AtsError("select_topk_per_sequence: scores must be float32 [batch, seq]")
    scores = scores.contiguous()
    B, L = scores.shape
    sel = torch.empty(B * keep, dtype=torch.int32, device=scores.device)
    check(_lib.load().ats_select_topk_per_sequence(scores.data_ptr(), B, L, int(keep), sel.data_ptr(), _stream()),
          "ats_select_topk_per_sequence")
    return sel


def scatter_add_rows(base: torch.Tensor, rows: torch.Tensor, delta: torch.Tensor) -> torch.Tensor:
    """base[rows[i]] += delta[i] in place (rows distinct); returns base."""
    _need_gpu(base, rows, delta)
    if not base.is_contiguous() or base.dim() != 2 or rows.dtype != torch.int32 or delta.dtype != base.dtype:
        raise AtsError("scatter_add_rows: base must be contiguous 2-D, rows int32, delta of base's dtype")
    delta = delta.reshape(-1, base.shape[1]).contiguous()
    check(_lib.load().ats_scatter_add_rows(base.data_ptr(), rows.contiguous().data_ptr(), delta.data_ptr(),
                                           rows.numel(), base.shape[1], _tag(base), _stream()),
          "ats_scatter_add_rows")
    return base


def kth_value_mask(values: torch.Tensor, kth: int, return_count: bool = False):
    """float32 mask of values >= the kth smallest value (1-based), same shape as `values`; with
    `return_count` also the number of ones as a one-element int64 device tensor (written by the kernel)."""
    _need_gpu(values)
    if values.dtype != torch.float32:
        raise AtsError("kth_value_mask: values must be float32")
    v = values.contiguous()
    mask = torch.empty_like(v)
    lib = _lib.load()
    ws_bytes = int(lib.ats_kth_value_workspace(v.numel()))       # 16 bytes, or with room for the digit histograms
    ws = torch.zeros(ws_bytes // 8, dtype=torch.int64, device=v.device) if v.numel() == 0 else \
        torch.empty(ws_bytes // 8, dtype=torch.int64, device=v.device)
    check(lib.ats_kth_value_mask(v.data_ptr(), v.numel(), int(kth), mask.data_ptr(), ws.data_ptr(), ws_bytes,
                                 _stream()), "ats_kth_value_mask")
    return (mask, ws[1:2]) if return_count else mask


def topk_mask_ste(values: torch.Tensor, k: int, want_ste: bool = True):
    """float32 mask with exactly min(k, n) ones at the k largest of `values` (lower index first among equals)
    and, with `want_ste`, the straight-through weights (mask - values) + values; both of `values`' shape."""
    _need_gpu(values)
    if values.dtype != torch.float32:
        raise AtsError("topk_mask_ste: values must be float32")
    v = values.contiguous()
    mask = torch.empty_like(v)
    ste = torch.empty_like(v) if want_ste else None
    lib = _lib.load()
    ws_bytes = int(lib.ats_kth_value_workspace(v.numel()))
    ws = torch.empty(max(ws_bytes // 8, 2), dtype=torch.int64, device=v.device)
    check(lib.ats_topk_mask_ste(v.data_ptr(), v.numel(), int(k), mask.data_ptr(), _ptr(ste), ws.data_ptr(), ws_bytes,
                                _stream()), "ats_topk_mask_ste")
    return (mask, ste) if want_ste else mask


def mod_route_bwd(prob: torch.Tensor, grad_weights: Optional[torch.Tensor], grad_probs: Optional[torch.Tensor],
                  temperature: float = 1.0, need_bias: bool = True):
    """Gradient of the MoD router's logits, float32 [n], and of its bias, float32 [1] (or None)."""
    _need_gpu(prob, grad_weights, grad_probs)
    p = prob.reshape(-1).contiguous()
    n = p.numel()
    for g in (grad_weights, grad_probs):
        if g is not None and (g.dtype != torch.float32 or g.numel() != n):
            raise AtsError("mod_route_bwd: gradients must be float32 with one value per token")
    if p.dtype != torch.float32:
        raise AtsError("mod_route_bwd: probabilities must be float32")
    gw = None if grad_weights is None else grad_weights.reshape(-1).contiguous()
    gp = None if grad_probs is None else grad_probs.reshape(-1).contiguous()
    gl = torch.empty(n, dtype=torch.float32, device=p.device)
    db = torch.empty(1, dtype=torch.float32, device=p.device) if need_bias else None
    check(_lib.load().ats_mod_route_bwd(_ptr(gw), _ptr(gp), p.data_ptr(), float(temperature), gl.data_ptr(), _ptr(db), n,
                                        _stream()), "ats_mod_route_bwd")
    return gl, db


def swiglu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """gate * silu(up) (dense-FFN convention of the fused wrapper)."""
    _need_gpu(gate, up)
    if gate.shape != up.shape or gate.dtype != up.dtype:
        raise AtsError("swiglu_mul: gate and up must match")
    g, u = gate.contiguous(), up.contiguous()
    out = torch.empty_like(g)
    check(_lib.load().ats_swiglu_mul(g.data_ptr(), u.data_ptr(), out.data_ptr(), g.numel(), _tag(g), _stream()),
          "ats_swiglu_mul")
    return out


# --------------------------------------------------------------------------- backward pass
def rmsnorm_bwd(x: torch.Tensor, weight: Optional[torch.Tensor], dy: torch.Tensor, eps: float = 1e-6,
                need_dw: bool = True) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """Gradients of rmsnorm: dx (x's shape and dtype) and dw (float32 [H]) or None."""
    _need_gpu(x, weight, dy)
    H = x.shape[-1]
    if dy.shape != x.shape or dy.dtype != x.dtype:
        raise AtsError(f"rmsnorm_bwd: dy {tuple(dy.shape)}/{dy.dtype} does not match x {tuple(x.shape)}/{x.dtype}")
    xc, dyc = x.contiguous(), dy.contiguous()
    if weight is not None:
        weight = weight.contiguous()
    rows = xc.numel() // H if H else 0
    dx = torch.empty_like(xc)
    lib = _lib.load()
    dw = ws = None
    ws_bytes = 0
    if need_dw and weight is not None:
        dw = torch.empty(H, dtype=torch.float32, device=x.device)
        ws_bytes = lib.ats_rmsnorm_bwd_workspace(rows, H)
        ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=x.device)
    check(lib.ats_rmsnorm_bwd(xc.data_ptr(), _ptr(weight), dyc.data_ptr(), dx.data_ptr(), _ptr(dw), rows, H,
                              float(eps), _tag(xc), _tag(weight) if weight is not None else ATS_F32, _ptr(ws),
                              ws_bytes, _stream()), "ats_rmsnorm_bwd")
    return dx.view(x.shape), dw


def _rows_2d(t: torch.Tensor, name: str) -> torch.Tensor:
    if t.dim() != 2 or t.stride(1) != 1:
        raise AtsError(f"{name}: operands must be 2-D with contiguous rows")
    return t


def silu_mul(a: torch.Tensor, b: torch.Tensor, rows_dev: Optional[torch.Tensor] = None) -> torch.Tensor:
    """silu(a) * b for 2-D operands that may be column slices of a wider matrix.  rows_dev: optional
    int32 device scalar; rows at or beyond it are left untouched."""
    _need_gpu(a, b, rows_dev)
    a, b = _rows_2d(a, "silu_mul"), _rows_2d(b, "silu_mul")
    if a.shape != b.shape or a.dtype != b.dtype:
        raise AtsError("silu_mul: operand shapes / dtypes differ")
    out = torch.empty(a.shape, dtype=a.dtype, device=a.device)
    check(_lib.load().ats_silu_mul_fwd(a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), out.data_ptr(),
                                       out.stride(0) if out.numel() else a.shape[1], a.shape[0], _ptr(rows_dev),
                                       a.shape[1], _tag(a), _stream()), "ats_silu_mul_fwd")
    return out


def silu_mul_bwd(a: torch.Tensor, b: torch.Tensor, dout: torch.Tensor, da: Optional[torch.Tensor] = None,
                 db: Optional[torch.Tensor] = None,
                 rows_dev: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Gradients of silu(a) * b; da/db may be preallocated (e.g. the two halves of one matrix)."""
    _need_gpu(a, b, dout, da, db)
    a, b, dout = _rows_2d(a, "silu_mul_bwd"), _rows_2d(b, "silu_mul_bwd"), _rows_2d(dout, "silu_mul_bwd")
    if a.shape != b.shape or a.shape != dout.shape or a.dtype != b.dtype or a.dtype != dout.dtype:
        raise AtsError("silu_mul_bwd: operand shapes / dtypes differ")
    if da is None:
        da = torch.empty(a.shape, dtype=a.dtype, device=a.device)
    if db is None:
        db = torch.empty(a.shape, dtype=a.dtype, device=a.device)
    da, db = _rows_2d(da, "silu_mul_bwd"), _rows_2d(db, "silu_mul_bwd")
    cols = a.shape[1]
    st = lambda t: t.stride(0) if t.shape[0] > 1 else max(t.stride(0), cols)
    check(_lib.load().ats_silu_mul_bwd(a.data_ptr(), st(a), b.data_ptr(), st(b), dout.data_ptr(), st(dout),
                                       da.data_ptr(), st(da), db.data_ptr(), st(db), a.shape[0], _ptr(rows_dev), cols,
                                       _tag(a), _stream()), "ats_silu_mul_bwd")
    return da, db


def combine_bwd(dout: torch.Tensor, y: torch.Tensor, token_map: torch.Tensor, w: torch.Tensor,
                k: int) -> Tuple[torch.Tensor, torch.Tensor]:
    """Gradients of combine: dy (y's shape/dtype) and dw float32 [T, k]."""
    _need_gpu(dout, y, token_map, w)
    if dout.dim() != 2 or y.dim() != 2 or dout.shape[1] != y.shape[1] or token_map.dtype != torch.int32:
        raise AtsError("combine_bwd: dout [T,H], y [rows,H], token_map int32 [rows]")
    T, H = dout.shape
    n_rows = y.shape[0]
    if token_map.numel() < n_rows or w.numel() != T * k or w.dtype != torch.float32:
        raise AtsError("combine_bwd: token_map / weights do not match the row and token counts")
    dout, y, w = dout.contiguous(), y.contiguous(), w.contiguous()
    dy = torch.empty_like(y)
    dw = torch.empty(T, k, dtype=torch.float32, device=y.device)
    check(_lib.load().ats_combine_bwd(dout.data_ptr(), y.data_ptr(), token_map.data_ptr(), w.data_ptr(), dy.data_ptr(),
                                      dw.data_ptr(), n_rows, T, int(k), H, _tag(y), _tag(dout), _stream()),
          "ats_combine_bwd")
    return dy, dw


def route_bwd(logits_route: torch.Tensor, idx: torch.Tensor, w: torch.Tensor, dw: torch.Tensor,
              temperature: float = 1.0, mode: int = ROUTE_SOFTMAX_TOPK, logits_aux: Optional[torch.Tensor] = None,
              usage: Optional[torch.Tensor] = None, aux_scale: float = 0.0,
              aux_scale_dev: Optional[torch.Tensor] = None, aux_value: Optional[torch.Tensor] = None) -> torch.Tensor:
    """dlogits [T,E] float32 of the routing rule (and of the load-balancing loss when usage is given;
    its factor is aux_scale times the optional float32 device scalar aux_scale_dev, which counts as 0 unless the optional
    float32 device scalar aux_value is below 1)."""
    _need_gpu(logits_route, idx, w, dw, logits_aux, usage, aux_scale_dev, aux_value)
    if aux_value is not None and (aux_value.dtype != torch.float32 or aux_value.numel() != 1):
        raise AtsError("route_bwd: aux_value must be a float32 scalar tensor")
    if aux_scale_dev is not None and (aux_scale_dev.dtype != torch.float32 or aux_scale_dev.numel() != 1):
        raise AtsError("route_bwd: aux_scale_dev must be a float32 scalar tensor")
    T, E = logits_route.shape
    k = idx.shape[1]
    if (logits_route.dtype != torch.float32 or idx.dtype != torch.int32 or w.dtype != torch.float32
            or dw.dtype != torch.float32 or w.shape != idx.shape or dw.shape != idx.shape):
        raise AtsError("route_bwd: logits float32 [T,E], idx int32 [T,k], w/dw float32 [T,k]")
    logits_route, idx, w, dw = logits_route.contiguous(), idx.contiguous(), w.contiguous(), dw.contiguous()
    if usage is not None:
        usage = usage.contiguous().float()
        logits_aux = (logits_route if logits_aux is None else logits_aux).contiguous()
    out = torch.empty(T, E, dtype=torch.float32, device=logits_route.device)
    check(_lib.load().ats_route_bwd_clamped(logits_route.data_ptr(), _ptr(logits_aux), idx.data_ptr(), w.data_ptr(),
                                            dw.data_ptr(), _ptr(usage), float(aux_scale), _ptr(aux_scale_dev), _ptr(aux_value),
                                            float(temperature), int(mode), out.data_ptr(), T, E, k, _stream()),
          "ats_route_bwd_clamped")
    return out


def router_bwd(dlogits: torch.Tensor, x: torch.Tensor, gate_weight: torch.Tensor,
               base: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None,
               need_dx: bool = True, need_dw: bool = True) -> Tuple[Optional[torch.Tensor], Optional[torch.Tensor]]:
    """Gradients of router_logits: dx = base + dlogits @ Wg (x's dtype) and dWg float32 [E,H]."""
    _need_gpu(dlogits, x, gate_weight, base, out)
    T, H = x.shape
    E = gate_weight.shape[0]
    if dlogits.shape != (T, E) or dlogits.dtype != torch.float32 or gate_weight.dtype != x.dtype:
        raise AtsError("router_bwd: dlogits float32 [T,E]; x and the gate weight share a dtype")
    dlogits, xc, wg = dlogits.contiguous(), x.contiguous(), gate_weight.contiguous()
    lib = _lib.load()
    dx = dwg = None
    if need_dx:
        if base is not None:
            base = base.contiguous()
        dx = out if out is not None else torch.empty_like(xc)
        check(lib.ats_router_bwd_dx(dlogits.data_ptr(), wg.data_ptr(), _ptr(base), dx.data_ptr(), T, E, H, _tag(xc),
                                    _stream()), "ats_router_bwd_dx")
    if need_dw:
        dwg = torch.empty(E, H, dtype=torch.float32, device=x.device)
        ws_bytes = lib.ats_router_bwd_dw_workspace(T, E, H)
        ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=x.device)
        check(lib.ats_router_bwd_dw(dlogits.data_ptr(), xc.data_ptr(), dwg.data_ptr(), T, E, H, _tag(xc),
                                    ws.data_ptr(), ws_bytes, _stream()), "ats_router_bwd_dw")
    return dx, dwg


def transpose_batched(mats: Sequence[torch.Tensor], in_tab: Optional[torch.Tensor] = None) -> Tuple[list, torch.Tensor]:
    """Transposes E equally shaped contiguous matrices [R,C]; returns the list of [C,R] views of one
    buffer and the device pointer table over them."""
    _need_gpu(*mats)
    R, C = mats[0].shape
    for m in mats:
        if m.shape != (R, C) or m.dtype != mats[0].dtype or not m.is_contiguous():
            raise AtsError("transpose_batched: matrices must be contiguous and share shape and dtype")
    E = len(mats)
    buf = torch.empty(E, C, R, dtype=mats[0].dtype, device=mats[0].device)
    outs = [buf[e] for e in range(E)]
    if in_tab is None:
        in_tab = weight_pointer_table(list(mats))
    # (written on the device: an upload of addresses that change from call to call would wait for the queue to drain)
    step = C * R * buf.element_size()
    out_tab, = fill_tables(buf.device, [(TABLE_INDEX, E, buf.data_ptr(), step, True)])
    aligned = step % 16 == 0 and all(m.data_ptr() % 16 == 0 for m in mats)
    check(_lib.load().ats_transpose_batched(in_tab.data_ptr(), out_tab.data_ptr(), E, R, C, _tag(mats[0]), int(aligned),
                                            _stream()), "ats_transpose_batched")
    return outs, out_tab


def wgrad_plan(row_count: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Per expert: first column and padded width of its slice in the transposed activations."""
    _need_gpu(row_count)
    E = row_count.numel()
    k_start = torch.empty(E, dtype=torch.int32, device=row_count.device)
    k_count = torch.empty(E, dtype=torch.int32, device=row_count.device)
    check(_lib.load().ats_wgrad_plan(row_count.data_ptr(), E, k_start.data_ptr(), k_count.data_ptr(), _stream()),
          "ats_wgrad_plan")
    return k_start, k_count


def wgrad_padded_rows(max_rows: int, E: int) -> int:
    return int(_lib.load().ats_wgrad_padded_rows(int(max_rows), int(E)))


def transpose_grouped_rows(src: torch.Tensor, row_start: torch.Tensor, row_count: torch.Tensor, max_rows: int,
                           gather: Optional[torch.Tensor] = None, gather_div: int = 1) -> torch.Tensor:
    """[rows, C] -> [C, padded] with expert e in columns k_start[e] .. (see wgrad_plan), zero padded."""
    _need_gpu(src, row_start, row_count, gather)
    src = _rows_2d(src, "transpose_grouped_rows")
    E = row_count.numel()
    C = src.shape[1]
    ld = wgrad_padded_rows(max_rows, E)
    out = torch.empty(C, ld, dtype=src.dtype, device=src.device)
    check(_lib.load().ats_transpose_grouped_rows(src.data_ptr(), src.stride(0), C, _ptr(gather), int(gather_div),
                                                 row_start.data_ptr(), row_count.data_ptr(), E, int(max_rows),
                                                 out.data_ptr(), ld, _tag(src), _stream()),
          "ats_transpose_grouped_rows")
    return out


def grouped_gemm_nt(b_ptrs: torch.Tensor, ldb: int, b_rows: int, row_start: torch.Tensor, row_count: torch.Tensor,
                    n_rows_out: int, max_rows: int, N: int, K: int, a: Optional[torch.Tensor] = None,
                    a_ptrs: Optional[torch.Tensor] = None, lda: Optional[int] = None,
                    a_rows: Optional[torch.Tensor] = None, a_row_div: int = 1, k_count: Optional[torch.Tensor] = None,
                    dtype: Optional[torch.dtype] = None, out_dtype: Optional[torch.dtype] = None,
                    out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out[row_start[e]+m, :N] = A_e[m, :K_e] @ B_e[:N, :K_e]^T (see ats_grouped_gemm_nt)."""
    _need_gpu(a, a_ptrs, b_ptrs, row_start, row_count, a_rows, k_count)
    if (a is None) == (a_ptrs is None):
        raise AtsError("grouped_gemm_nt: give either a or a_ptrs")
    if a is not None:
        a = _rows_2d(a, "grouped_gemm_nt")
        dtype = a.dtype
        lda = a.stride(0)
    elif dtype is None or lda is None:
        raise AtsError("grouped_gemm_nt: a_ptrs needs dtype and lda")
    out_dtype = dtype if out_dtype is None else out_dtype
    E = b_ptrs.numel()
    if out is None:
        out = torch.empty(n_rows_out, N, dtype=out_dtype, device=b_ptrs.device)
    elif out.shape != (n_rows_out, N) or out.dtype != out_dtype or not out.is_contiguous():
        raise AtsError("grouped_gemm_nt: out must be a contiguous [n_rows_out, N] tensor of out_dtype")
    check(_lib.load().ats_grouped_gemm_nt(_ptr(a), _ptr(a_ptrs), int(lda), int(a.shape[0]) if a is not None else 0,
                                          _ptr(a_rows), int(a_row_div), b_ptrs.data_ptr(), int(ldb), int(b_rows),
                                          out.data_ptr(), N, row_start.data_ptr(), row_count.data_ptr(), _ptr(k_count),
                                          E, int(max_rows), int(N), int(K), _DT[dtype], _DT[out_dtype], _stream()),
          "ats_grouped_gemm_nt")
    return out


def grouped_gemm_nn_supported(E: int, max_rows: int, N: int, K: int, ldb: int, dtype: torch.dtype) -> bool:
    """Whether grouped_gemm_nn has a kernel for these sizes (bfloat16, prefill-sized groups)."""
    if dtype not in _DT:
        return False
    return bool(_lib.load().ats_grouped_gemm_nn_supported(int(E), int(max_rows), int(N), int(K), int(ldb), _DT[dtype]))


def grouped_gemm_nn(b_ptrs: torch.Tensor, ldb: int, row_start: torch.Tensor, row_count: torch.Tensor, n_rows_out: int,
                    max_rows: int, N: int, K: int, a: torch.Tensor, a_rows: Optional[torch.Tensor] = None,
                    a_row_div: int = 1, out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """out[row_start[e]+m, :N] = A_e[m, :K] @ B_e[:K, :N] with B_e = b_ptrs[e] stored [K, ldb] (see
    ats_grouped_gemm_nn): the data gradient of a linear layer against the weights as the forward holds them."""
    _need_gpu(a, b_ptrs, row_start, row_count, a_rows)
    a = _rows_2d(a, "grouped_gemm_nn")
    out_dtype = a.dtype if out_dtype is None else out_dtype
    E = b_ptrs.numel()
    out = torch.empty(n_rows_out, N, dtype=out_dtype, device=b_ptrs.device)
    check(_lib.load().ats_grouped_gemm_nn(a.data_ptr(), int(a.stride(0)), int(a.shape[0]), _ptr(a_rows), int(a_row_div),
                                          b_ptrs.data_ptr(), int(ldb), out.data_ptr(), N, row_start.data_ptr(),
                                          row_count.data_ptr(), E, int(max_rows), int(N), int(K), _DT[a.dtype],
                                          _DT[out_dtype], _stream()),
          "ats_grouped_gemm_nn")
    return out


def grouped_gemm_nn_slices(E: int, max_rows: int, N: int, K: int, ldb: int, dtype: torch.dtype) -> int:
    """Slices of K for a product against weights stored [K, ldb]; 0: multiply by a transposed copy."""
    if dtype != torch.bfloat16:
        return 0
    return int(_lib.load().ats_grouped_gemm_nn_slices(int(E), int(max_rows), int(N), int(K), int(ldb), _DT[dtype]))


def grouped_gemm_nn_sliced(b_ptrs: torch.Tensor, ldb: int, row_start: torch.Tensor, row_count: torch.Tensor, n_rows_out: int,
                           max_rows: int, N: int, K: int, a: torch.Tensor, k_splits: int) -> torch.Tensor:
    """grouped_gemm_nn for groups of up to 256 rows on average: the product [n_rows_out, N], or with more than one slice of
    K the float32 partial results [k_splits, n_rows_out, N]."""
    a = _rows_2d(a, "grouped_gemm_nn_sliced")
    if a.shape[0] < max_rows or n_rows_out < max_rows or a.shape[1] < K:
        raise AtsError("grouped_gemm_nn_sliced: fewer rows than max_rows, or than K columns")
    _need_gpu(a, b_ptrs, row_start, row_count)
    E = b_ptrs.numel()
    shape, dtype = ((n_rows_out, N), a.dtype) if k_splits == 1 else ((k_splits, n_rows_out, N), torch.float32)
    out = torch.empty(shape, dtype=dtype, device=b_ptrs.device)
    check(_lib.load().ats_grouped_gemm_nn_sliced(a.data_ptr(), int(a.stride(0)), b_ptrs.data_ptr(), int(ldb), out.data_ptr(),
                                                 int(n_rows_out), row_start.data_ptr(), row_count.data_ptr(), E,
                                                 int(max_rows), int(N), int(K), int(k_splits), _DT[a.dtype], _DT[dtype],
                                                 _stream()),
          "ats_grouped_gemm_nn_sliced")
    return out


def grouped_gemm_nn_f32_supported(E: int, max_rows: int, N: int, K: int) -> bool:
    """Whether a float32 product against [K, N] weights is faster read as they lie than through a transposed copy."""
    return bool(_lib.load().ats_grouped_gemm_nn_f32_supported(int(E), int(max_rows), int(N), int(K)))


def grouped_gemm_nn_f32(b_ptrs: torch.Tensor, ldb: int, row_start: torch.Tensor, row_count: torch.Tensor, max_rows: int, N: int,
                        K: int, a: torch.Tensor) -> torch.Tensor:
    """grouped_gemm_nn in float32 on the small tiles: [max_rows, N]."""
    _need_gpu(a, b_ptrs, row_start, row_count)
    a = _rows_2d(a, "grouped_gemm_nn_f32")
    if a.dtype != torch.float32 or a.shape[0] < max_rows or a.shape[1] < K:
        raise AtsError("grouped_gemm_nn_f32: a must be float32 [rows, K]")
    out = torch.empty(max_rows, N, dtype=torch.float32, device=a.device)
    check(_lib.load().ats_grouped_gemm_nn_f32(a.data_ptr(), a.stride(0), b_ptrs.data_ptr(), int(ldb), out.data_ptr(), N,
                                              row_start.data_ptr(), row_count.data_ptr(), b_ptrs.numel(), int(max_rows), int(N),
                                              int(K), _stream()), "ats_grouped_gemm_nn_f32")
    return out


def wgrad_f32_supported(a: torch.Tensor, b: torch.Tensor, E: int = 1) -> bool:
    """Whether wgrad_f32 takes these rows (float32, 16-byte aligned) and is faster than the product of transposed copies."""
    return all(t.dtype == torch.float32 and t.dim() == 2 and t.shape[0] > 0 and t.shape[1] % 4 == 0 and t.stride(1) == 1
               and t.stride(0) >= t.shape[1] and t.stride(0) % 4 == 0 and t.data_ptr() % 16 == 0 for t in (a, b)) \
        and bool(_lib.load().ats_grouped_wgrad_f32_supported(int(E), a.shape[0], a.shape[1], b.shape[1]))


def wgrad_f32(a: torch.Tensor, b: torch.Tensor, k_start: Optional[torch.Tensor] = None, k_count: Optional[torch.Tensor] = None,
              b_rows: Optional[torch.Tensor] = None, b_row_div: int = 1) -> torch.Tensor:
    """a^T @ b for rows as they lie, a [R, M], b [R, N]; per group [E, M, N] over the k_count[e] rows from k_start[e] where
    these are given, with b's row r taken from b_rows[r] // b_row_div if a gather table is given."""
    if not wgrad_f32_supported(a, b, 1 if k_count is None else k_count.numel()):
        raise AtsError("wgrad_f32: float32 rows of 16-byte multiples, of sizes that the small tiles serve")
    if (a.shape[0] != b.shape[0] if b_rows is None else b_rows.dtype != torch.int32 or b_rows.numel() < a.shape[0] or b_row_div < 1):
        raise AtsError("wgrad_f32: a and b must have the same number of rows, or an int32 row of b for every row of a")
    _need_gpu(a, b, k_start, k_count, b_rows)
    (R, M), N = a.shape, b.shape[1]
    E = 1 if k_count is None else k_count.numel()
    out = torch.empty((M, N) if k_count is None else (E, M, N), dtype=torch.float32, device=a.device)
    check(_lib.load().ats_grouped_wgrad_f32(a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), _ptr(b_rows), int(b_row_div),
                                            out.data_ptr(), _ptr(k_start), _ptr(k_count), E, R, M, N, _stream()),
          "ats_grouped_wgrad_f32")
    return out


# --------------------------------------------------------------------------- attention
def _key_bias(key_bias, B: int, Lk: int, q: torch.Tensor, who: str):
    if key_bias is None:
        return None
    if key_bias.shape != (B, Lk) or key_bias.dtype != torch.float32 or key_bias.device != q.device:
        raise AtsError(f"{who}: key_bias must be float32 [batch, keys] = [{B}, {Lk}] on the inputs' device")
    return key_bias.contiguous()


def _pair_bias(pair_bias, B: int, Hq: int, L: int, Lk: int, q: torch.Tensor, who: str):
    """Checks a pair bias, float32 [batch or 1, queries, keys] or [batch or 1, heads or 1, queries, keys], and
    returns it as a contiguous 4-D tensor with its batch and head strides in floats (0 where it is shared)."""
    if pair_bias.dim() == 3:
        pair_bias = pair_bias[:, None]
    if pair_bias.dim() != 4 or pair_bias.shape[0] not in (1, B) or pair_bias.shape[1] not in (1, Hq) \
            or tuple(pair_bias.shape[2:]) != (L, Lk) or pair_bias.dtype != torch.float32 or pair_bias.device != q.device:
        raise AtsError(f"{who}: pair_bias must be float32 [batch or 1, (heads or 1,) queries, keys] = "
                       f"[{B}, {Hq}, {L}, {Lk}] on the inputs' device")
    pair_bias = pair_bias.contiguous()
    heads = pair_bias.shape[1]
    return pair_bias, (0 if pair_bias.shape[0] == 1 else heads * L * Lk), (0 if heads == 1 else L * Lk)


def _attention_extras(key_bias, pair_bias, dropout_p: float, B: int, Hq: int, L: int, Lk: int, q: torch.Tensor, who: str):
    """Arguments of the extended entry points.  Returns (key_bias, pair_bias, batch stride, head stride): with a
    pair bias or dropout a per-key bias is folded into the pair bias (the kernels take one or the other)."""
    key_bias = _key_bias(key_bias, B, Lk, q, who)
    if not 0.0 <= dropout_p < 1.0:
        raise AtsError(f"{who}: dropout_p {dropout_p} must be in [0, 1)")
    sb = sh = 0
    if pair_bias is not None:
        pair_bias, sb, sh = _pair_bias(pair_bias, B, Hq, L, Lk, q, who)
        if key_bias is not None:
            pair_bias, sb, sh = _pair_bias(pair_bias + key_bias[:, None, None, :], B, Hq, L, Lk, q, who)
            key_bias = None
    elif dropout_p > 0.0 and key_bias is not None:
        pair_bias, sb, sh = key_bias[:, None, None, :].expand(B, 1, L, Lk).contiguous(), L * Lk, 0
        key_bias = None
    return key_bias, pair_bias, sb, sh


def causal_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: Optional[float] = None,
                     return_lse: bool = False, key_bias: Optional[torch.Tensor] = None, split_keys: bool = True,
                     pair_bias: Optional[torch.Tensor] = None, dropout_p: float = 0.0, dropout_seed: int = 0):
    """Causal grouped-query attention.  q [B,Hq,L,D]; k [B,Hkv,Lk,D] with a head's rows one after the other
    and any batch/head strides (e.g. a view of a larger cache buffer); v [B,Hkv,Lk,D] in any batch/head/position
    strides (e.g. a view of a fused projection output); bf16, D 64 or 128, Lk >= L.
    With Lk > L the leading Lk - L keys are a cache: query i sits at position i + Lk - L.
    key_bias [B, Lk] float32 (optional) is added to the scaled scores of a key for every query and head;
    (1 - attention_mask) * -1e4 is the reference's padding mask (MS/core/model.py:819-824).
    pair_bias [B or 1, L, Lk] or [B or 1, Hq or 1, L, Lk] float32 (optional) is added to the scaled scores of
    a (query, key) pair, for every head or per head: (1 - mask) * -1e4 for the reference's 4-D masks (same lines).
    dropout_p > 0 drops attention weights (model.py:831-833) by a hash of (dropout_seed, batch, head, query,
    key); causal_attention_bwd given the same seed sees the same mask.
    split_keys=False keeps the single-pass kernel where few rows against many keys would otherwise be cut
    into key ranges.  Returns out [B, L, Hq*D] (and lse [B,Hq,L] float32 if asked)."""
    if not return_lse and key_bias is None and pair_bias is None and dropout_p == 0.0:
        done = _lib.native().attention(q, k, v, q.shape[-1] ** -0.5 if scale is None else scale, split_keys)
        if done is not None:
            return done
    _need_gpu(q, k, v)
    if q.dim() != 4 or k.dim() != 4 or v.dim() != 4 or q.dtype != torch.bfloat16 or k.dtype != q.dtype or v.dtype != q.dtype:
        raise AtsError("causal_attention: q, k, v must be 4-D bfloat16 tensors [batch, heads, seq, head_dim]")
    B, Hq, L, D = q.shape
    Hkv, Lk = k.shape[1], k.shape[2]
    if k.shape != (B, Hkv, Lk, D) or v.shape != (B, Hkv, Lk, D) or Hq % Hkv != 0 or Lk < L:
        raise AtsError(f"causal_attention: shapes q {tuple(q.shape)} k {tuple(k.shape)} v {tuple(v.shape)}")
    q = q.contiguous()
    if k.stride(3) != 1 or k.stride(2) != D or k.stride(0) % 8 or k.stride(1) % 8 or k.data_ptr() % 16:
        k = k.contiguous()        # rows of a head must follow one another; batch and head strides are free
    key_bias, pair_bias, pair_sb, pair_sh = _attention_extras(key_bias, pair_bias, dropout_p, B, Hq, L, Lk, q,
                                                              "causal_attention")
    if v.stride(3) != 1 or any(st % 8 for st in v.stride()[:3]) or v.stride(2) < D or v.data_ptr() % 16:
        v = v.contiguous()
    lib = _lib.load()
    out = torch.empty(B, L, Hq * D, dtype=q.dtype, device=q.device)
    lse = torch.empty(B, Hq, L, dtype=torch.float32, device=q.device) if return_lse else None
    # decoding a few sequences: scratch for the partial results of key ranges that run side by side
    ws_bytes = lib.ats_attention_fwd_workspace(B, Hq, Hkv, L, Lk, D) if split_keys else 0
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=q.device) if ws_bytes else None
    check(lib.ats_attention_fwd_ex(q.data_ptr(), k.data_ptr(), k.stride(0), k.stride(1), v.data_ptr(), v.stride(0),
                                   v.stride(2), v.stride(1), _ptr(key_bias), _ptr(pair_bias), pair_sb, pair_sh,
                                   float(dropout_p), int(dropout_seed) & 0xFFFFFFFFFFFFFFFF, out.data_ptr(), _ptr(lse),
                                   B, Hq, Hkv, L, Lk, D, float(D ** -0.5 if scale is None else scale), _ptr(ws),
                                   ws_bytes, _stream()),
          "ats_attention_fwd_ex")
    return (out, lse) if return_lse else out


def prompt_attention_supported(x: torch.Tensor, weight: torch.Tensor, B: int, L: int, Hq: int, Hkv: int, D: int) -> bool:
    """Whether the attention of a prompt x [B * L, K] projected by weight rotates its queries itself (prompt_attention): a product
    in slices of K has its rotation in the sum of the slices."""
    return (x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == x.dtype
            and bool(_lib.load().ats_attention_fwd_rope_supported(B, Hq, Hkv, L, L, D))
            and linear_k_splits(B * L, weight.shape[0], x.shape[1], x.dtype) == 1)


def prompt_attention(qkv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, B: int, Hkv: int, D: int, scale: float,
                     keep_values: bool):
    """rope and causal_attention of the stacked projections qkv [B * L, (Hq + 2 Hkv) * D]: (out [B, L, Hq * D], rotated k, v),
    v contiguous with keep_values and a view of qkv without; None for operands that the launches do not read as they are."""
    if qkv.dim() != 2 or B <= 0 or Hkv <= 0 or D <= 0 or qkv.shape[0] % B or qkv.shape[1] % D or qkv.shape[1] <= 2 * Hkv * D:
        raise AtsError(f"prompt_attention: qkv {tuple(qkv.shape)} is not [{B} * positions, (heads + 2 * {Hkv}) * {D}]")
    return _lib.native().prompt_attention(qkv, cos, sin, B, Hkv, D, scale, keep_values)


def causal_attention_bwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, out: torch.Tensor, lse: torch.Tensor,
                         dout: torch.Tensor, scale: Optional[float] = None, key_bias: Optional[torch.Tensor] = None,
                         pair_bias: Optional[torch.Tensor] = None, dropout_p: float = 0.0, dropout_seed: int = 0):
    """Gradients of causal_attention: q [B,Hq,L,D], k, v [B,Hkv,Lk,D], out, dout [B,L,Hq*D], lse [B,Hq,L],
    key_bias, pair_bias, dropout_p and dropout_seed as in the forward.  Returns (dq, dk, dv) shaped like q, k, v."""
    _need_gpu(q, k, v, out, lse, dout)
    B, Hq, L, D = q.shape
    Hkv, Lk = k.shape[1], k.shape[2]
    if (q.dtype != torch.bfloat16 or k.shape != (B, Hkv, Lk, D) or v.shape != k.shape or out.shape != (B, L, Hq * D)
            or dout.shape != out.shape or lse.shape != (B, Hq, L) or lse.dtype != torch.float32):
        raise AtsError("causal_attention_bwd: shapes or dtypes do not match the forward's")
    q, k, v, out = q.contiguous(), k.contiguous(), v.contiguous(), out.contiguous()
    dout = dout.to(q.dtype).contiguous()
    lse = lse.contiguous()
    key_bias, pair_bias, pair_sb, pair_sh = _attention_extras(key_bias, pair_bias, dropout_p, B, Hq, L, Lk, q,
                                                              "causal_attention_bwd")
    lib = _lib.load()
    # delta = rowsum(dO * O) is formed inside the dQ kernel and handed to the dK/dV kernel through this buffer
    delta = torch.empty(B, Hq, L, dtype=torch.float32, device=q.device)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    # few key tiles: float32 sums of ranges of queries that run side by side; without memory for them in one range
    ws_bytes = lib.ats_attention_bwd_workspace(B, Hq, Hkv, L, Lk, D)
    try:
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=q.device) if ws_bytes else None
    except torch.OutOfMemoryError:
        ws = None
    check(lib.ats_attention_bwd_out_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), dout.data_ptr(),
                                       lse.data_ptr(), delta.data_ptr(), _ptr(key_bias), _ptr(pair_bias), pair_sb, pair_sh,
                                       float(dropout_p), int(dropout_seed) & 0xFFFFFFFFFFFFFFFF, dq.data_ptr(), dk.data_ptr(),
                                       dv.data_ptr(), B, Hq, Hkv, L, Lk, D, float(D ** -0.5 if scale is None else scale),
                                       _ptr(ws), ws_bytes, _stream()),
          "ats_attention_bwd_out_ws")
    return dq, dk, dv


# --------------------------------------------------------------------------- float32 attention
def _transpose_tables(src: torch.Tensor, in_tab: torch.Tensor, out_tab: torch.Tensor, R: int, C: int):
    """Matrix n at in_tab[n] ([R, C] contiguous) -> [C, R] at out_tab[n]; src gives the type."""
    check(_lib.load().ats_transpose_batched(in_tab.data_ptr(), out_tab.data_ptr(), in_tab.numel(), R, C, _tag(src), 1, _stream()),
          "ats_transpose_batched")


def _pad_rows(t: torch.Tensor, rows: int) -> torch.Tensor:
    """[..., r, D] -> [..., rows, D] contiguous, zero rows appended."""
    if t.shape[-2] == rows:
        return t.contiguous()
    out = t.new_zeros(*t.shape[:-2], rows, t.shape[-1])
    out[..., :t.shape[-2], :] = t
    return out


def _attention_f32_dims(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> Tuple[int, int, int, int, int, int]:
    """(B, Hq, Hkv, L, Lk, D) of a float32 attention, on either of its routes; raises for tensors that do not fit together."""
    if q.dim() != 4 or k.dim() != 4 or v.dim() != 4 or q.dtype != torch.float32 or k.dtype != q.dtype or v.dtype != q.dtype:
        raise AtsError("attention_f32: q, k, v must be 4-D float32 tensors [batch, heads, seq, head_dim]")
    B, Hq, L, D = q.shape
    Hkv, Lk = k.shape[1], k.shape[2]
    if k.shape != (B, Hkv, Lk, D) or v.shape != (B, Hkv, Lk, D) or Hq % Hkv != 0 or Lk < L or D % 4 or B * Hq > 4096:
        raise AtsError(f"attention_f32: shapes q {tuple(q.shape)} k {tuple(k.shape)} v {tuple(v.shape)} "
                       "(head_dim a multiple of 4, at most 4096 (batch, head) pairs)")
    return B, Hq, Hkv, L, Lk, D


def attention_f32(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: Optional[float] = None,
                  key_bias: Optional[torch.Tensor] = None, pair_bias: Optional[torch.Tensor] = None,
                  dropout_p: float = 0.0, dropout_seed: int = 0, return_weights: bool = False):
    """Causal grouped-query attention on float32 tensors with the values of the reference's _standard_attention
    (MS/core/model.py:807-839).  Where attention_f32_fused_supported takes the call it is one launch; otherwise the scores of
    every (batch, head) are materialised by a grouped product (float32 MFMA kernels), softmaxed in place
    (ats_attention_softmax_f32: scale, causal fill, masks, dropout) and multiplied with V by a second grouped product.  q [B,Hq,L,D], k, v [B,Hkv,Lk,D], D a multiple of 4;
    key_bias / pair_bias / dropout as in causal_attention.  Returns out [B, L, Hq*D]; with return_weights also
    the state the backward needs (padded weights before and after dropout)."""
    B, Hq, Hkv, L, Lk, D = _attention_f32_dims(q, k, v)
    _need_gpu(q, k, v)
    key_bias = _key_bias(key_bias, B, Lk, q, "attention_f32")
    if not 0.0 <= dropout_p < 1.0:
        raise AtsError(f"attention_f32: dropout_p {dropout_p} must be in [0, 1)")
    pair_sb = pair_sh = 0
    if pair_bias is not None:
        pair_bias, pair_sb, pair_sh = _pair_bias(pair_bias, B, Hq, L, Lk, q, "attention_f32")
    scale = float(D ** -0.5 if scale is None else scale)
    if not return_weights and attention_f32_fused_supported(q, k, v, pair_bias, dropout_p):
        return attention_f32_fused(q, k, v, scale, key_bias, want_stats=False)[0]
    dev = q.device
    lib = _lib.load()
    Lp, Lkp = (L + 3) // 4 * 4, (Lk + 3) // 4 * 4
    E = B * Hq
    qp, kp, vp = _pad_rows(q, Lp), _pad_rows(k, Lkp), _pad_rows(v, Lkp)
    vT = torch.empty(B * Hkv, D, Lkp, dtype=q.dtype, device=dev)
    kv_bytes = Lkp * D * 4
    row_start, row_count, k_tab, v_in, v_out, vT_tab = fill_tables(dev, [
        (TABLE_INDEX, E, 0, Lp, False), (TABLE_CONSTANT, E, Lp, 0, False),
        (TABLE_KV_OF_HEAD, E, kp.data_ptr(), kv_bytes, True), (TABLE_INDEX, B * Hkv, vp.data_ptr(), kv_bytes, True),
        (TABLE_INDEX, B * Hkv, vT.data_ptr(), kv_bytes, True), (TABLE_KV_OF_HEAD, E, vT.data_ptr(), kv_bytes, True)],
        (B, Hq, Hkv))
    # scores[e] = q[e] . k[kv_of[e]]^T
    w = grouped_gemm_nt(k_tab, D, Lkp, row_start, row_count, E * Lp, E * Lp, Lkp, D,
                        a=qp.view(E * Lp, D))
    w_drop = torch.empty_like(w) if dropout_p > 0 else None
    check(lib.ats_attention_softmax_f32(w.data_ptr(), _ptr(w_drop), B, Hq, L, Lp, Lk, Lkp, scale, _ptr(key_bias),
                                        _ptr(pair_bias), pair_sb, pair_sh, float(dropout_p),
                                        int(dropout_seed) & 0xFFFFFFFFFFFFFFFF, _stream()), "ats_attention_softmax_f32")
    # out[e] = weights[e] . v[kv_of[e]]  (NT product against v^T)
    _transpose_tables(vp, v_in, v_out, Lkp, D)
    used = w_drop if w_drop is not None else w
    o = grouped_gemm_nt(vT_tab, Lkp, D, row_start, row_count, E * Lp, E * Lp, D, Lkp, a=used)
    out = o.view(B, Hq, Lp, D)[:, :, :L].transpose(1, 2).reshape(B, L, Hq * D)
    if return_weights:
        return out, (w, w_drop, qp, kp, vp)
    return out


def attention_f32_fused_supported(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, pair_bias: Optional[torch.Tensor],
                                  dropout_p: float) -> bool:
    """Whether the kernels without materialised scores take this call (csrc/attention_f32_fused.hip)."""
    return (pair_bias is None and dropout_p == 0.0 and q.shape[-1] in (64, 128) and q.numel() > 0
            and all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (q, k, v)))


def attention_f32_fused(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: Optional[float],
                        key_bias: Optional[torch.Tensor], want_stats: bool = True) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """attention_f32 in one launch: out [B, L, Hq*D] and, for the backward pass, the maximum and the reciprocal sum of
    every row [B*Hq, L, 2]."""
    B, Hq, Hkv, L, Lk, D = _attention_f32_dims(q, k, v)
    _need_gpu(q, k, v)
    if not attention_f32_fused_supported(q, k, v, None, 0.0):
        raise AtsError("attention_f32_fused: contiguous, 16-byte aligned rows of head_dim 64 or 128")
    scale = float(D ** -0.5 if scale is None else scale)
    key_bias = _key_bias(key_bias, B, Lk, q, "attention_f32")
    out = torch.empty(B, L, Hq * D, dtype=torch.float32, device=q.device)
    stats = torch.empty(B * Hq, L, 2, dtype=torch.float32, device=q.device) if want_stats else None
    check(_lib.load().ats_attention_f32_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), _ptr(stats), B, Hq, Hkv,
                                            L, Lk, D, scale, _ptr(key_bias), _stream()), "ats_attention_f32_fwd")
    return out, stats


def attention_f32_fused_bwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, out: torch.Tensor, stats: torch.Tensor,
                            dout: torch.Tensor, scale: Optional[float], key_bias: Optional[torch.Tensor]):
    """Gradients of attention_f32_fused: (dq, dk, dv) in two launches."""
    B, Hq, Hkv, L, Lk, D = _attention_f32_dims(q, k, v)
    if any(t.shape != shape or t.dtype != torch.float32 for t, shape in ((out, (B, L, Hq * D)), (dout, (B, L, Hq * D)),
                                                                         (stats, (B * Hq, L, 2)))):
        raise AtsError("attention_f32_fused_bwd: out and dout must be float32 [batch, seq, heads * head_dim], stats as handed out")
    _need_gpu(q, k, v, out, stats, dout)
    q, k, v, out, stats, dout = (t if t.is_contiguous() and t.data_ptr() % 16 == 0 else t.clone(memory_format=torch.contiguous_format)
                                 for t in (q, k, v, out, stats, dout))
    scale = float(D ** -0.5 if scale is None else scale)
    key_bias = _key_bias(key_bias, B, Lk, q, "attention_f32")
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    delta = torch.empty(B * Hq * L, dtype=torch.float32, device=q.device)
    check(_lib.load().ats_attention_f32_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), stats.data_ptr(),
                                            dout.data_ptr(), delta.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B,
                                            Hq, Hkv, L, Lk, D, scale, _ptr(key_bias), _stream()),
          "ats_attention_f32_bwd")
    return dq, dk, dv


def attention_f32_bwd(state, dout: torch.Tensor, B: int, Hq: int, Hkv: int, L: int, Lk: int, D: int,
                      scale: Optional[float] = None, dropout_p: float = 0.0, dropout_seed: int = 0):
    """Gradients of attention_f32 from the state its forward returned: dV = P'^T.dO, dP' = dO.V^T, dS through
    ats_attention_softmax_bwd_f32, dQ = dS.K, dK = dS^T.Q, each a grouped float32 product (transposed operands
    are written by ats_transpose_batched; the query heads of a kv head are summed by ats_sum_partials).
    Returns (dq [B,Hq,L,D], dk, dv [B,Hkv,Lk,D])."""
    w, w_drop, qp, kp, vp = state
    _need_gpu(w, dout)
    dev = w.device
    lib = _lib.load()
    scale = float(D ** -0.5 if scale is None else scale)
    Lp, Lkp = qp.shape[2], kp.shape[2]
    E, rep = B * Hq, Hq // Hkv
    do = _pad_rows(dout.to(torch.float32).view(B, L, Hq, D).permute(0, 2, 1, 3), Lp)          # [B, Hq, Lp, D]
    kT = torch.empty(B * Hkv, D, Lkp, dtype=w.dtype, device=dev)
    doT, qT = (torch.empty(E, D, Lp, dtype=w.dtype, device=dev) for _ in range(2))
    matT = torch.empty(E, Lkp, Lp, dtype=w.dtype, device=dev)       # of the weights, then of dS
    ds = torch.empty(E * Lp, Lkp, dtype=w.dtype, device=dev)
    used = w_drop if w_drop is not None else w
    kv_bytes, q_bytes, s_bytes = Lkp * D * 4, Lp * D * 4, Lp * Lkp * 4
    # dV and dK: per query head a product over the queries, written so that the `rep` heads of a kv head are
    # `rep` slices of one buffer: group (b, hq) goes to slot (hq % rep) * (B * Hkv) + its kv matrix.  The b_ptrs and row
    # tables of those products are read in slot order.
    (row_start, row_count, v_tab, k_in, k_out, kT_tab, do_in, do_out, q_in, q_out, w_in, ds_in, mat_out, doT_tab, qT_tab,
     slot_start, slot_count) = fill_tables(dev, [
         (TABLE_INDEX, E, 0, Lp, False), (TABLE_CONSTANT, E, Lp, 0, False),
         (TABLE_KV_OF_HEAD, E, vp.data_ptr(), kv_bytes, True),
         (TABLE_INDEX, B * Hkv, kp.data_ptr(), kv_bytes, True), (TABLE_INDEX, B * Hkv, kT.data_ptr(), kv_bytes, True),
         (TABLE_KV_OF_HEAD, E, kT.data_ptr(), kv_bytes, True),
         (TABLE_INDEX, E, do.data_ptr(), q_bytes, True), (TABLE_INDEX, E, doT.data_ptr(), q_bytes, True),
         (TABLE_INDEX, E, qp.data_ptr(), q_bytes, True), (TABLE_INDEX, E, qT.data_ptr(), q_bytes, True),
         (TABLE_INDEX, E, used.data_ptr(), s_bytes, True), (TABLE_INDEX, E, ds.data_ptr(), s_bytes, True),
         (TABLE_SLOT_OF_HEAD, E, matT.data_ptr(), s_bytes, True),
         (TABLE_HEAD_OF_SLOT, E, doT.data_ptr(), q_bytes, True), (TABLE_HEAD_OF_SLOT, E, qT.data_ptr(), q_bytes, True),
         (TABLE_INDEX, E, 0, Lkp, False), (TABLE_CONSTANT, E, Lkp, 0, False)],
        (B, Hq, Hkv))
    # dP' = dO . V^T, then in place to dS (gradient of the raw scores)
    grouped_gemm_nt(v_tab, D, Lkp, row_start, row_count, E * Lp, E * Lp, Lkp, D, a=do.view(E * Lp, D), out=ds)
    check(lib.ats_attention_softmax_bwd_f32(w.data_ptr(), ds.data_ptr(), B, Hq, L, Lp, Lk, Lkp, scale, float(dropout_p),
                                            int(dropout_seed) & 0xFFFFFFFFFFFFFFFF, _stream()),
          "ats_attention_softmax_bwd_f32")
    # dQ = dS . K  (NT product against K^T)
    _transpose_tables(kp, k_in, k_out, Lkp, D)
    dq = grouped_gemm_nt(kT_tab, Lkp, D, row_start, row_count, E * Lp, E * Lp, D, Lkp, a=ds)
    dq = dq.view(B, Hq, Lp, D)[:, :, :L].contiguous()
    _transpose_tables(do, do_in, do_out, Lp, D)
    _transpose_tables(qp, q_in, q_out, Lp, D)

    def over_queries(in_tab, rhsT_tab) -> torch.Tensor:
        """sum over the heads of a kv group of mat[e]^T . rhs[e]: mat [E*Lp, Lkp], rhsT [E, D, Lp] -> [B,Hkv,Lkp,D]."""
        _transpose_tables(matT, in_tab, mat_out, Lp, Lkp)
        parts = grouped_gemm_nt(rhsT_tab, Lp, D, slot_start, slot_count, E * Lkp, E * Lkp, D, Lp, a=matT.view(E * Lkp, Lp))
        parts = parts.view(rep, B * Hkv * Lkp * D)
        total = sum_partials(parts, torch.float32) if rep > 1 else parts[0]
        return total.view(B, Hkv, Lkp, D)[:, :, :Lk].contiguous()

    dv = over_queries(w_in, doT_tab)
    dk = over_queries(ds_in, qT_tab)
    return dq, dk, dv


_COUNTS = 1 << 17
_count_tables: dict = {}       # device -> int32 0, 1, 2, .. (512 KB), written once
_count_views: dict = {}        # (T, device) -> places of it (making the two views takes 4 us, four times in a training pass)
_count_lock = threading.Lock()


def _single_group(T: int, device: torch.device):
    """row_start = [0], row_count = [T] of a one-group GEMM: two places of a constant table per device (two fill launches
    per call are a visible share of a small projection).  The table is complete before anybody gets it and lives as long as
    the process, so any stream, thread and captured graph may read it; counts beyond it, and a capture that comes before
    it, have two integers of their own."""
    pair = _count_views.get((T, device))
    if pair is not None:
        return pair
    table = _count_tables.get(device)
    if table is None or T >= _COUNTS:
        if T >= _COUNTS or torch.cuda.is_current_stream_capturing():
            return fill_tables(device, [(TABLE_CONSTANT, 1, 0, 0, False), (TABLE_CONSTANT, 1, T, 0, False)])
        with _count_lock:
            table = _count_tables.get(device)
            if table is None:          # (the copy from host memory returns when the data has arrived)
                table = _count_tables[device] = torch.arange(_COUNTS, dtype=torch.int32).to(device)
    if len(_count_views) >= 256:
        _count_views.clear()
    pair = _count_views[T, device] = table[:1], table[T:T + 1]
    return pair


@functools.lru_cache(maxsize=4096)
def linear_k_splits(T: int, N: int, K: int, dtype: torch.dtype) -> int:
    """Slices of K for a product with one weight [N, K].  33-256 rows only: bfloat16 by the estimated times of every route,
    float32 against a long K.  Up to 32 rows the plain launch streams the weights itself ([4096, 4096] x 16 rows: 10.3 us against
    14.2 with the slices and their sum)."""
    if not 32 < T <= 256 or K % 8 or N % 8:
        return 1
    if dtype == torch.bfloat16:
        return _lib.load().ats_linear_k_slices(T, N, K)
    return down_k_splits(1, T, N, K, dtype) if K * dtype.itemsize > 4096 else 1


def linear_rope_append(x: torch.Tensor, weight: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, k_cache: torch.Tensor,
                       v_cache: torch.Tensor, cache_pos: int, seq: int) -> Optional[torch.Tensor]:
    """linear_nt(x [batch * seq, K], weight [(Hq + 2 Hkv) * D, K]) and rope_append of its columns: where the product runs in
    slices of K one launch adds them up, rotates and appends (the same bits).  None where it does not."""
    if (x.dim() != 2 or weight.dim() != 2 or x.shape[1] != weight.shape[1] or k_cache.dim() != 4 or v_cache.shape != k_cache.shape
            or x.shape[0] != k_cache.shape[0] * seq or weight.shape[0] % k_cache.shape[3]
            or weight.shape[0] <= 2 * k_cache.shape[1] * k_cache.shape[3]):
        raise AtsError(f"linear_rope_append: x {tuple(x.shape)}, weight {tuple(weight.shape)}, {seq} positions, caches "
                       f"{tuple(k_cache.shape)} / {tuple(v_cache.shape)}")
    T, K = x.shape
    N, D = weight.shape[0], k_cache.shape[3]
    splits = linear_k_splits(T, N, K, x.dtype)
    if splits == 1 or not x.is_cuda or weight.dtype != x.dtype or not weight.is_contiguous():
        return None
    start, count = _single_group(T, x.device)
    return _lib.native().linear_rope_append(x, weight_pointer_table([weight]), start, count, splits, cos, sin, k_cache, v_cache,
                                            cache_pos, N // D - 2 * k_cache.shape[1], seq)


def linear_nt(x: torch.Tensor, weight: torch.Tensor, table: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x [T, K] @ weight[N, K]^T through the grouped GEMM kernels with a single group.  table: the (contiguous) weight's
    address on the device where the caller has it."""
    _need_gpu(x, weight)
    if x.dim() != 2 or weight.dim() != 2 or x.shape[1] != weight.shape[1] or x.dtype != weight.dtype:
        raise AtsError("linear_nt: x [T,K], weight [N,K], same dtype")
    T, K = x.shape
    N = weight.shape[0]
    x, weight = x.contiguous(), weight.contiguous()
    if table is None:
        table = weight_pointer_table([weight])
    start, count = _single_group(T, x.device)
    splits = linear_k_splits(T, N, K, x.dtype)
    done = _lib.native().linear(x, table, start, count, N, splits)
    if done is not None:
        return done
    if splits > 1:      # a few rows against a whole weight matrix: slices of K keep every CU streaming
        return sum_partials(grouped_down_splitk(x, table, start, count, T, N, K, splits), x.dtype)
    out = torch.empty(T, N, dtype=x.dtype, device=x.device)
    check(_lib.load().ats_linear_nt(x.data_ptr(), table.data_ptr(), out.data_ptr(), start.data_ptr(), count.data_ptr(), T, N, K,
                                    _tag(x), _stream()), "ats_linear_nt")
    return out
